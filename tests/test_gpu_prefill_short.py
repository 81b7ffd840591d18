"""GPU tests of the single-launch prefill of short prompts (up to 256 tokens).

A row's results do not depend on the rows after it, and both prefill paths run the same
operations in the same order, so the first S rows of a 300-token prompt (launch by launch) are the
oracle of an S-token prompt, bit for bit: K and V of every layer, the attention rows and the
residual stream after the last layer. The ragged-length tests of test_gpu_prefill.py compare
both paths with the numpy oracle.
"""

from functools import partial

import pytest
import torch

from megaqwen_amd import _abi
from megaqwen_amd import megakernel_decode as MK
from megaqwen_amd import rope, weights

pytestmark = pytest.mark.gpu

N_LAYERS, LONG = 3, 300
ANY_XCD, GAVE_UP = 1, 2  # MQ_DEBUG_PREFILL_*


@pytest.fixture(scope="module")
def models(gpu_weights_gamma):
    """Two decoders over the first layers (distinct norm gains), and the long prompt's results."""
    w = gpu_weights_gamma
    cos, sin = (t.cuda() for t in rope.rope_tables(320))
    args = (w["embed_weight"], w["layer_weights"][: 11 * N_LAYERS], w["final_norm_weight"], w["lm_head_weight"], cos,
            sin, N_LAYERS, 320, 320)
    decs = [MK.MegakernelPrefillDecoder(*args) for _ in range(2)]
    ids = weights.random_prompt(LONG, seed=77)
    decs[0].prefill_step(ids)
    want = [t.clone() for t in (decs[0].k_cache_[:, :, :LONG], decs[0].v_cache_[:, :, :LONG],
                                decs[0].attn_out_[:LONG], decs[0].hidden_float_[:LONG])]
    return decs, ids, want


def _results(dec, S):
    return dec.k_cache_[:, :, :S], dec.v_cache_[:, :, :S], dec.attn_out_[:S], dec.hidden_float_[:S]


# row blocks of 16, groups of 4 blocks, relay waves of one or two blocks, the last launch-free length
@pytest.mark.parametrize("S", [1, 2, 15, 16, 17, 48, 63, 64, 65, 80, 127, 128, 129, 144, 192, 241, 255, 256, 257])
def test_short_prompt_equals_the_long_prompts_rows(models, S):
    (dec, _), ids, want = models
    print(f"prefill S={S}", flush=True)
    for rep in range(2):
        dec.reset()
        dec.prefill_step(ids[:S])
        for name, got, ref in zip(("k", "v", "attention", "hidden"), _results(dec, S), want):
            ref = ref[:, :, :S] if name in "kv" else ref[:S]
            assert torch.equal(got, ref), (name, rep)
        assert not dec.k_cache_[:, :, S:].any() and not dec.v_cache_[:, :, S:].any()


def test_short_prompts_on_two_streams(models):
    """Launches of two decoders that may overlap on two streams: each has its own sync words, and one
    that does not find workgroups of its own on every XCD runs from a single list."""
    decs, ids, want = models
    streams = [torch.cuda.Stream() for _ in decs]
    lengths = (128, 40)
    for dec in decs:
        dec.reset()
    torch.cuda.synchronize()
    for _ in range(4):
        for dec, st, S in zip(decs, streams, lengths):
            with torch.cuda.stream(st):
                dec.prefill_step_async(ids[:S])
    torch.cuda.synchronize()
    for dec, S in zip(decs, lengths):
        assert int(dec.output_token_.item()) >= 0
        assert torch.equal(dec.k_cache_[:, :, :S], want[0][:, :, :S])
        assert torch.equal(dec.hidden_float_[:S], want[3][:S])


@pytest.mark.parametrize("S", [1, 16, 17, 64, 65, 129, 256])
def test_single_list_gives_the_same_bits(models, S, monkeypatch):
    """The form for launches whose workgroups cannot be on every XCD at once (forced from the
    host): tasks from one list, every hand-over device-wide."""
    (dec, _), ids, want = models
    monkeypatch.setattr(_abi.lib(), "launch_prefill_float", partial(_abi.lib().mq_debug_prefill, ANY_XCD))
    print(f"prefill S={S}", flush=True)
    for rep in range(2):
        dec.reset()
        dec.prefill_step(ids[:S])
        for name, got, ref in zip(("k", "v", "attention", "hidden"), _results(dec, S), want):
            ref = ref[:, :, :S] if name in "kv" else ref[:S]
            assert torch.equal(got, ref), (name, rep)
        assert not dec.k_cache_[:, :, S:].any() and not dec.v_cache_[:, :, S:].any()


@pytest.mark.parametrize("failing", [0, 1])
def test_a_launch_that_gives_up_says_so_itself(models, failing, monkeypatch):
    """The give-up word belongs to the launch that set it (forced from the host): its own result is
    -3, a prefill beside it returns its token, whichever comes first."""
    decs, ids, _ = models
    lib, S = _abi.lib(), 40
    token = decs[0].prefill_step(ids[:S])
    normal, gave_up = lib.launch_prefill_float, partial(lib.mq_debug_prefill, GAVE_UP)
    print("prefill S=40, give-up word set", flush=True)
    for i, dec in enumerate(decs):
        monkeypatch.setattr(lib, "launch_prefill_float", gave_up if i == failing else normal)
        dec.prefill_step_async(ids[:S])
    got = [int(dec.output_token_.item()) for dec in decs]
    assert got[failing] == -3 and got[1 - failing] == token
    monkeypatch.setattr(lib, "launch_prefill_float", gave_up)
    with pytest.raises(_abi.MegakernelError, match="error flags 2"):
        decs[0].prefill_step(ids[:S])
    monkeypatch.setattr(lib, "launch_prefill_float", normal)
    assert decs[0].position() == 0 and decs[0].prefill_step(ids[:S]) == token
