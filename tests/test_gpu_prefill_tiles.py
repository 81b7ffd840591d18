"""GPU tests of the prefill products' row tiles past 512 tokens.

The row tile of q/k/v, of gate/up and, from 2177 tokens, of o_proj and down_proj is chosen by the
rounds of workgroups a prompt takes, and every tile sums each output in the same order. A row's
results depend neither on the tile nor on the rows after it, so the first S rows of a longer
prompt whose attention adds in the same order are the oracle of an S-token prompt, bit for bit.
The lengths are the first and the last of every range of lengths with one choice of tiles (the
rule and its tables restated from mq_prefill.hip) and those beside the lines between its kernels:
a first length leaves its last row tile one row, a last one fills it.

Before each prompt every buffer that is compared is cleared or filled with NaN, so a row that a
tile does not write shows.
"""

import os
import re

import pytest
import torch

from megaqwen_amd import build
from megaqwen_amd import megakernel_decode as MK
from megaqwen_amd import rope, weights

N_LAYERS, NUM_CUS = 2, 256
# attn_prefill serves prompts up to 768 tokens; attn_prefill_fa3 and, past 5888, attn_prefill_fa2
# add in the same order
LONG = {768: (513, 768), 8200: (769, 8192)}
# lines between kernels and tile families: gate/up 640, attention 768 and 5888, the partial sums'
# tiles 1023, 1536 and 2048, the residual in the epilogue 2176
LINES = (513, 640, 641, 768, 769, 1023, 1024, 1536, 1537, 2048, 2049, 2176, 2177, 5888, 5889, 8191, 8192)
# workgroups a row tile of q/k/v, gate/up, o_proj / down_proj, and the first length each serves
PRODUCTS = ((16, 513), (24, 641), (8, 2177))


def tables():
    """The (rows, us a round) tables of the three products, from the source."""
    text = open(os.path.join(build.CSRC, "mq_prefill.hip")).read()
    found = re.findall(r"constexpr RowTile TILES\[\] = \{(.*?)\};", text)
    assert len(found) == len(PRODUCTS)
    return [[(int(rows), float(us)) for rows, us in re.findall(r"\{(\d+), ([\d.]+)f\}", t)] for t in found]


def chosen(S, tabs):
    """The row tile of each product of an S-token prompt (None: below its range)."""
    return [min(tab, key=lambda t: t[1] * -(-nx * -(-S // t[0]) // NUM_CUS))[0] if S >= lo else None
            for tab, (nx, lo) in zip(tabs, PRODUCTS)]


def edges():
    tabs = tables()
    tiles = {S: chosen(S, tabs) for S in range(513, 8193)}
    ends = {S for S in range(513, 8192) if tiles[S] != tiles[S + 1]}
    return sorted(set(LINES) | ends | {S + 1 for S in ends}), tiles


def test_every_tile_is_reached():
    """Each tile of the tables is the choice for some of the lengths below."""
    lengths, tiles = edges()
    for p, tab in enumerate(tables()):
        assert {tiles[S][p] for S in lengths} - {None} == {rows for rows, _ in tab}


@pytest.fixture(scope="module")
def model(gpu_weights_gamma):
    w = gpu_weights_gamma
    n = max(LONG)
    cos, sin = (t.cuda() for t in rope.rope_tables(n))
    dec = MK.MegakernelPrefillDecoder(w["embed_weight"], w["layer_weights"][: 11 * N_LAYERS], w["final_norm_weight"],
                                      w["lm_head_weight"], cos, sin, N_LAYERS, n, n)
    return dec, weights.random_prompt(n, seed=5)


def _prefill(dec, ids):
    """The prompt's results, after every buffer they stand in was cleared or filled with NaN; rows
    past the prompt stay as they were."""
    S = len(ids)
    print(f"prefill S={S}", flush=True)
    dec.reset()
    rows = (dec.attn_out_, dec.hidden_float_)
    for t in (*rows, dec.q_proj_, dec.mlp_norm_, dec.mlp_intermediate_, dec.normalized_):
        t.fill_(float("nan"))
    dec.prefill_step(ids)
    for t in (dec.k_cache_, dec.v_cache_):
        assert not t[:, :, S:].any(), S
    for t in rows:
        assert t[S:].isnan().all(), S
    return [t.clone() for t in (dec.k_cache_[:, :, :S], dec.v_cache_[:, :, :S], *(t[:S] for t in rows))]


@pytest.mark.gpu
@pytest.mark.parametrize("long", sorted(LONG))
def test_rows_do_not_depend_on_the_tile(model, long):
    dec, ids = model
    want = _prefill(dec, ids[:long])
    lo, hi = LONG[long]
    for S in edges()[0]:
        if lo <= S <= hi:
            for name, got, ref in zip(("k", "v", "attention", "hidden"), _prefill(dec, ids[:S]), want):
                assert torch.equal(got, ref[:, :, :S] if name in "kv" else ref[:S]), (S, name)


@pytest.mark.gpu
def test_rows_are_the_same_bits_in_both_flash_forms(model):
    """attn_prefill_fa3 and attn_prefill_fa2 run the same operations on a score in the same order,
    so a row's bits do not turn at the length where the one takes over from the other."""
    dec, ids = model
    want = _prefill(dec, ids[:8200])
    for S in (769, 1117, 3000, 5888):
        for name, got, ref in zip(("k", "v", "attention", "hidden"), _prefill(dec, ids[:S]), want):
            assert torch.equal(got, ref[:, :, :S] if name in "kv" else ref[:S]), (S, name)
