"""GPU tests of the prefill products' row tiles past 512 tokens.

The row tile of q/k/v and gate/up, and past 2176 tokens of o_proj and down_proj, is chosen by the
rounds of workgroups a prompt takes, and every tile sums each output in the same order. A row's
results depend neither on the tile nor on the rows after it, so the first S rows of a longer
prompt that runs the same attention kernel are the oracle of an S-token prompt, bit for bit. The
lengths sit at the edges of the tiles' ranges and one past them, none a multiple of its tile but
the first (q/k/v: 64 rows up to 1024 tokens, 96 to 1536, 128 to 2048, 160 to 2560, 192 to 3072,
224 to 3584, 256 to 4096, 160 to 5120; gate/up: 96 to 960, 128 to 1280, 160 to 1600, 192 to 1920,
256 to 2560, 320 to 3200, 160 to 3360, 192 to 4032, 256; o_proj and down_proj: fp32 partials to
2176, then the residual added in the epilogue on 128 rows to 4096, 192 to 6144, 256).
"""

import pytest
import torch

from megaqwen_amd import megakernel_decode as MK
from megaqwen_amd import rope, weights

pytestmark = pytest.mark.gpu

N_LAYERS = 2
# attn_prefill serves prompts up to 768 tokens, attn_prefill_fa3 up to 5888, then attn_prefill_fa2
LONG = {767: [513, 641],
        6140: [769, 959, 961, 1023, 1025, 1281, 1537, 1601, 1921, 2047, 2049, 2175, 2177, 2561, 3073, 3201, 3361, 3585,
               4033, 4097, 5121],
        8200: [6145, 8191]}


@pytest.fixture(scope="module")
def model(gpu_weights_gamma):
    w = gpu_weights_gamma
    n = max(LONG)
    cos, sin = (t.cuda() for t in rope.rope_tables(n))
    dec = MK.MegakernelPrefillDecoder(w["embed_weight"], w["layer_weights"][: 11 * N_LAYERS], w["final_norm_weight"],
                                      w["lm_head_weight"], cos, sin, N_LAYERS, n, n)
    return dec, weights.random_prompt(n, seed=5)


def _results(dec, S):
    return [t.clone() for t in (dec.k_cache_[:, :, :S], dec.v_cache_[:, :, :S], dec.attn_out_[:S], dec.hidden_float_[:S])]


@pytest.mark.parametrize("long", sorted(LONG))
def test_rows_do_not_depend_on_the_tile(model, long):
    dec, ids = model
    print(f"prefill S={long}", flush=True)
    dec.prefill_step(ids[:long])
    want = _results(dec, long)
    for S in LONG[long]:
        print(f"prefill S={S}", flush=True)
        dec.prefill_step(ids[:S])
        for name, got, ref in zip(("k", "v", "attention", "hidden"), _results(dec, S), want):
            assert torch.equal(got, ref[:, :, :S] if name in "kv" else ref[:S]), (S, name)


def test_rows_are_the_same_bits_in_both_flash_forms(model):
    """attn_prefill_fa3 and attn_prefill_fa2 run the same operations on a score in the same order,
    so a row's bits do not turn at the length where the one takes over from the other."""
    dec, ids = model
    print("prefill S=8200", flush=True)
    dec.prefill_step(ids[:8200])
    want = _results(dec, 8200)
    for S in (769, 1117, 3000, 5888):
        print(f"prefill S={S}", flush=True)
        dec.reset()
        dec.prefill_step(ids[:S])
        for name, got, ref in zip(("k", "v", "attention", "hidden"), _results(dec, S), want):
            assert torch.equal(got, ref[:, :, :S] if name in "kv" else ref[:S]), (S, name)
