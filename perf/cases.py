"""The calls that a user of this package makes, as cases that can be timed and compared.

Qwen3-0.6B at batch 1: one decoder block at a position (`decode_layer`), one decode step of
the whole model (`MegakernelDecoder.decode_step_with_logits`) at positions from the first
tokens of a chat to the end of a 16384-position cache, and the prefill of a prompt
(`MegakernelPrefillDecoder.prefill_step`, `MegakernelFusedPrefillDecoder.prefill_step`) from a
few tokens to 8192. Everything is bf16, the only type the package takes.

Weights are N(0, 0.02) as in the package's seeded models, norm gains 1 + 0.1 N(0, 1). The
context of a decode case is what a prefill leaves in the caches: K rows are RMS-normalised
and rotated, so their entries are N(0, 1); V rows are a projection of normalised rows of
1024 by weights of 0.02, so theirs are N(0, 0.64).
"""

import math

import torch

from megaqwen_amd import config as C
from megaqwen_amd import megakernel_decode as MK
from megaqwen_amd import rope

# Positions the decode kernel accepts, and the longest prompt of the package's configurations
MAX_POSITION, MAX_PROMPT, MAX_FUSED_PROMPT = 16384, 8192, 64
V_STD = 0.64  # 0.02 * sqrt(1024)


def listed():
    return [
        # one block of the model on its own, as a caller that checks or splits layers runs it
        {"name": "block_p200", "kind": "block", "n": 200},
        # the first tokens of a chat: the shortest context
        {"name": "decode_p12", "kind": "decode", "n": 12},
        # a chat of a few turns (the headline position)
        {"name": "decode_p200", "kind": "decode", "n": 200},
        # the end of a 2048-token generation
        {"name": "decode_p2047", "kind": "decode", "n": 2047},
        # generation behind an 8192-token prompt
        {"name": "decode_p8192", "kind": "decode", "n": 8192},
        # a nearly full 16384-position cache
        {"name": "decode_p15001", "kind": "decode", "n": 15001},
        # a one-line question, through the decoder made for prompts of up to 64 tokens
        {"name": "prefill_fused_s23", "kind": "fused", "n": 23},
        # an ordinary short prompt
        {"name": "prefill_s128", "kind": "prefill", "n": 128},
        # the default prompt limit (512 tokens)
        {"name": "prefill_s512", "kind": "prefill", "n": 512},
        # a prompt with a system message and some turns, of no round length
        {"name": "prefill_s1117", "kind": "prefill", "n": 1117},
        # a document of a few pages
        {"name": "prefill_s3000", "kind": "prefill", "n": 3000},
        # the longest prompt
        {"name": "prefill_s8192", "kind": "prefill", "n": 8192},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "decode", "decode", "decode", "fused", "prefill", "prefill", "prefill"])
    if kind == "fused":
        return {"kind": kind, "n": _log_uniform(rng, 1, MAX_FUSED_PROMPT)}
    if kind == "prefill":
        return {"kind": kind, "n": _log_uniform(rng, 2, MAX_PROMPT)}
    return {"kind": kind, "n": _log_uniform(rng, 2, MAX_POSITION - 1)}


def _layers(case):
    return 1 if case["kind"] == "block" else C.NUM_LAYERS


def _max_seq(case):
    """Cache length a user gives such a run: the 8448 of an 8192-token prompt with 256 new
    tokens, or the longest."""
    return 8448 if case["n"] <= 8192 else MAX_POSITION


_ROPE = {}


def _rope(max_seq):
    if max_seq not in _ROPE:
        _ROPE[max_seq] = tuple(t.cuda() for t in rope.rope_tables(max_seq))
    return _ROPE[max_seq]


def _normal(g, shape, std, mean=0.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=g).to(torch.bfloat16)


def _inputs(case, seed):
    """Weights, context and prompt, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, L = case["n"], _layers(case)
    x = {"flat": []}
    for _ in range(L):
        for name in C.LAYER_WEIGHT_NAMES:
            shape = C.LAYER_WEIGHT_SHAPES[name]
            x["flat"].append(_normal(g, shape, 0.1, 1.0) if len(shape) == 1 else _normal(g, shape, 0.02))
    if case["kind"] == "block":
        x["hidden"] = _normal(g, (C.HIDDEN_SIZE,), 1.0)
    else:
        x["embed"] = _normal(g, (C.VOCAB_SIZE, C.HIDDEN_SIZE), 0.02)
        x["norm"] = _normal(g, (C.HIDDEN_SIZE,), 0.1, 1.0)
    if case["kind"] in ("block", "decode"):
        # the context, per layer [8, n, 128]
        x["k"] = [_normal(g, (C.NUM_KV_HEADS, n, C.HEAD_DIM), 1.0) for _ in range(L)]
        x["v"] = [_normal(g, (C.NUM_KV_HEADS, n, C.HEAD_DIM), V_STD) for _ in range(L)]
    tokens = 1 if case["kind"] in ("block", "decode") else n
    x["ids"] = torch.randint(C.VOCAB_SIZE, (tokens,), generator=g, device="cuda", dtype=torch.int32).cpu()
    x["cos"], x["sin"] = _rope(_max_seq(case))
    return x


def _fill(cache, rows):
    for layer, r in enumerate(rows):
        cache[layer, :, : r.shape[1]] = r


def prepare(case, seed):
    x = _inputs(case, seed)
    n, kind, max_seq = case["n"], case["kind"], _max_seq(case)
    state = {"kind": kind, "n": n}
    if kind == "block":
        state.update(hidden=x["hidden"], flat=x["flat"], cos=x["cos"], sin=x["sin"])
        for name in ("k", "v"):
            state[name] = torch.zeros(1, C.NUM_KV_HEADS, max_seq, C.HEAD_DIM, dtype=torch.bfloat16, device="cuda")
            _fill(state[name], x[name])
        return state
    args = (x["embed"], x["flat"], x["norm"], x["embed"], x["cos"], x["sin"], C.NUM_LAYERS, max_seq)
    if kind == "decode":
        dec = MK.MegakernelDecoder(*args)
        _fill(dec.get_k_cache(), x["k"])
        _fill(dec.get_v_cache(), x["v"])
        state["token"] = int(x["ids"][0])
    elif kind == "fused":
        dec = MK.MegakernelFusedPrefillDecoder(*args, MAX_FUSED_PROMPT)
    else:
        dec = MK.MegakernelPrefillDecoder(*args, n)
    state.update(dec=dec, ids=x["ids"])
    return state


def run(state):
    n, kind = state["n"], state["kind"]
    if kind == "block":
        out = MK.decode_layer(state["hidden"], state["flat"], state["cos"], state["sin"], state["k"], state["v"], n)
        return {"hidden": out, "k": state["k"][:, :, n], "v": state["v"][:, :, n]}
    dec = state["dec"]
    if kind == "decode":
        dec.set_position(n)
        _, logits = dec.decode_step_with_logits(state["token"])
        return {"logits": logits, "normed": dec.normalized_state(), "hidden": dec.hidden_state(),
                "k": dec.get_k_cache()[:, :, n], "v": dec.get_v_cache()[:, :, n]}
    # The prefill has no logits: the final-norm row that its LM head multiplies stands for them
    # (the token itself may turn on a tie of two bf16 logits).
    dec.prefill_step(state["ids"])
    return {"normed": dec.final_normed_state(), "k": dec.get_k_cache()[:, :, :n], "v": dec.get_v_cache()[:, :, :n]}


def work(case):
    n, kind = case["n"], case["kind"]
    kv_row = 2 * C.NUM_KV_HEADS * C.HEAD_DIM * 2  # K and V bytes of one position and layer
    attention = 4 * C.NUM_Q_HEADS * C.HEAD_DIM  # flops of one query and key, both products
    matrices = C.LINEAR_PARAMS // C.NUM_LAYERS
    if kind == "block":
        return {"bytes": 2 * C.LAYER_PARAMS + kv_row * (n + 1) + 4 * C.HIDDEN_SIZE,
                "flops": 2 * matrices + attention * (n + 1)}
    if kind == "decode":
        return {"bytes": C.decode_bytes(n) + 4 * C.VOCAB_SIZE,
                "flops": 2 * C.LINEAR_PARAMS + C.NUM_LAYERS * attention * (n + 1) + 2 * C.VOCAB_SIZE * C.HIDDEN_SIZE}
    # weights once, an embedding row a token read, K and V written
    return {"bytes": C.WEIGHT_BYTES_PER_TOKEN + 2 * C.HIDDEN_SIZE * (n - 1) + C.KV_BYTES_PER_POSITION * n,
            "flops": C.prefill_flops(n)}


def tolerance(case):
    # Measured against exact(): a block's outputs are off by up to 0.0043 (the bf16 roundings of
    # its stages). Through 28 layers, each of which rounds to bf16 a dozen times, a prefill's are
    # off by 0.012 to 0.015 and a decode step's by 0.018 to 0.044; two implementations that sum in
    # another order differ by about as much. Stated: four times the block's, 0.03 for a whole model.
    return {"rel": 0.017} if case["kind"] == "block" else {"rel": 0.03}


# ---------------------------------------------------------------- in 64 bits

def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + C.RMS_EPS) * w


def _rotate(x, cos, sin):
    half = C.HEAD_DIM // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _block64(h, flat, cos, sin, k_ctx, v_ctx):
    """One decoder block on rows h [T, 1024] behind a context of k_ctx / v_ctx [8, n, 128] (or
    None): (h, new K rows [8, T, 128], new V rows)."""
    w = dict(zip(C.LAYER_WEIGHT_NAMES, (t.double() for t in flat)))
    T, D, group = h.shape[0], C.HEAD_DIM, C.NUM_Q_HEADS // C.NUM_KV_HEADS
    x = _rms(h, w["input_layernorm"])
    q = _rotate(_rms((x @ w["q_proj"].T).view(T, C.NUM_Q_HEADS, D), w["q_norm"]), cos[:, None], sin[:, None])
    k = _rotate(_rms((x @ w["k_proj"].T).view(T, C.NUM_KV_HEADS, D), w["k_norm"]), cos[:, None], sin[:, None])
    v = (x @ w["v_proj"].T).view(T, C.NUM_KV_HEADS, D)
    out = torch.empty(T, C.NUM_Q_HEADS, D, dtype=torch.float64, device=h.device)
    for g in range(C.NUM_KV_HEADS):
        kk = k[:, g] if k_ctx is None else torch.cat((k_ctx[g].double(), k[:, g]))
        vv = v[:, g] if v_ctx is None else torch.cat((v_ctx[g].double(), v[:, g]))
        for head in range(group * g, group * (g + 1)):
            for t0 in range(0, T, 2048):  # rows t0.. see keys up to their own
                t1 = min(T, t0 + 2048)
                keys = kk.shape[0] - T + t1
                s = (q[t0:t1, head] @ kk[:keys].T) / math.sqrt(D)
                if T > 1:
                    s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(keys - (t1 - t0) + 1), -math.inf)
                out[t0:t1, head] = torch.softmax(s, -1) @ vv[:keys]
    h = h + out.view(T, C.Q_SIZE) @ w["o_proj"].T
    x = _rms(h, w["post_attention_layernorm"])
    gate = x @ w["gate_proj"].T
    h = h + (gate * torch.sigmoid(gate) * (x @ w["up_proj"].T)) @ w["down_proj"].T
    return h, k.transpose(0, 1), v.transpose(0, 1)


def exact(case, seed):
    x = _inputs(case, seed)
    n, kind = case["n"], case["kind"]
    if kind == "block":
        at = slice(n, n + 1)
        h, k, v = _block64(x["hidden"].double()[None], x["flat"], x["cos"][at].double(), x["sin"][at].double(),
                           x["k"][0], x["v"][0])
        return {"hidden": h[0], "k": k[None, :, 0], "v": v[None, :, 0]}
    decode = kind == "decode"
    at = slice(n, n + 1) if decode else slice(0, n)
    cos, sin = x["cos"][at].double(), x["sin"][at].double()
    h = x["embed"][x["ids"].cuda().long()].double()
    ks, vs = [], []
    for layer in range(C.NUM_LAYERS):
        h, k, v = _block64(h, x["flat"][11 * layer : 11 * layer + 11], cos, sin, x["k"][layer] if decode else None,
                           x["v"][layer] if decode else None)
        ks.append(k)
        vs.append(v)
    k, v, last = torch.stack(ks), torch.stack(vs), h[-1]
    normed = _rms(last, x["norm"].double())
    if decode:
        return {"logits": x["embed"].double() @ normed, "normed": normed, "hidden": last, "k": k[:, :, 0],
                "v": v[:, :, 0]}
    return {"normed": normed, "k": k, "v": v}
