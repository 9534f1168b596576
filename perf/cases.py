"""The attention calls whose speed is tracked, as a program makes them.

Every case is one call of a public entry point of `rdnattention` on tensors
already in device memory.  The kinds:

  prefill   flash_attn: whole prompts, fp16, contiguous tensors
  extend    attention_forward_into: a block of new query rows against a longer
            key/value cache (a chunk of a long prompt, a prompt behind a shared
            prefix), K and V being views into one [B, S, 2, Hkv, D] cache
  decode    attention_forward_into: one or a few new rows per sequence
            against the cache, same views
  i8        flash_attn_int8qk: int8 Q/K/V with per-token Q and K scales
  i8q       flash_attn_int8qk_quantized: fp16 Q/K/V, quantised on the way

listed() holds the fixed cases; draw() gives others of the same kinds and
ranges.  A case is a dict of plain values: kind, b, hq, hkv, sq, sk, d,
causal, window (-1 = off), rope.
"""
import math

import torch

import rdnattention

KEYS = ("kind", "b", "hq", "hkv", "sq", "sk", "d", "causal", "window", "rope")

# a drawn case asks for at most this much work (below the largest listed ones)
MAX_FLOPS = 5.0e11
MAX_BYTES = 2.0e9


def _case(name, *values):
    case = dict(zip(KEYS, values))
    return dict(case, name=name) if name else case


def listed():
    return [
        # the quick-start call: a small encoder-sized batch, latency counts
        _case("f16_mha_s512_d64", "prefill", 1, 8, 8, 512, 512, 64, False, -1, False),
        # one request's prompt at an odd length
        _case("f16_prompt_s1237_d128", "prefill", 1, 32, 8, 1237, 1237, 128, True, -1, True),
        # a batch of prompts in an 8B-class grouped-query layer: the headline
        _case("f16_prefill_b4_s4096_d128", "prefill", 4, 32, 8, 4096, 4096, 128, True, -1, True),
        # long context, two-sided sliding window, large heads
        _case("f16_window_s16384_d256", "prefill", 1, 16, 16, 16384, 16384, 256, False, 4096, True),
        _case("f16_window_s4096_d512", "prefill", 1, 16, 16, 4096, 4096, 512, False, 4096, True),
        # a chunk of a long prompt against the part already cached
        _case("f16_extend_q256_k16640_d128", "extend", 1, 32, 8, 256, 16640, 128, True, -1, False),
        # one sequence, one new token, a short cache: the smallest call
        _case("f16_decode_b1_k2048_d128", "decode", 1, 32, 8, 1, 2048, 128, False, -1, False),
        # a served batch with long caches: memory bound
        _case("f16_decode_b16_k32768_d128", "decode", 16, 32, 8, 1, 32768, 128, False, -1, False),
        # large heads, a ragged cache
        _case("f16_decode_b8_k6001_d256", "decode", 8, 16, 8, 1, 6001, 256, False, -1, False),
        # INT8 prefill of long prompts
        _case("i8_prefill_b2_s8192_d128", "i8", 2, 32, 8, 8192, 8192, 128, True, -1, False),
        # INT8 decode: an int8 cache is kept because decode is memory bound
        _case("i8_decode_b8_k8192_d128", "i8", 8, 32, 8, 1, 8192, 128, False, -1, False),
        # INT8 from fp16 activations, quantisers included
        _case("i8q_b2_s2050_d64", "i8q", 2, 16, 4, 2050, 2050, 64, True, -1, False),
    ]


HEADS = ((8, 8), (16, 16), (32, 32), (32, 8), (32, 8), (16, 4), (16, 8), (24, 8), (40, 8), (32, 1))


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "extend", "decode", "decode", "i8", "i8", "i8q"))
    hq, hkv = rng.choice(HEADS)
    b = rng.choice((1, 1, 2, 4)) if kind != "decode" else rng.choice((1, 2, 4, 8, 16, 32))
    window, rope = -1, False
    if kind == "prefill":
        d = rng.choice((64, 128, 128, 32 * rng.randint(1, 16)))
        sq = sk = _log_int(rng, 128, 16384)
        causal = rng.random() < 0.75
        rope = rng.random() < 0.5
        if rng.random() < 0.25:
            window = _log_int(rng, 64, 4096)
    elif kind == "extend":
        d = rng.choice((64, 128, 128, 32 * rng.randint(1, 8)))
        sq, sk = _log_int(rng, 16, 1024), _log_int(rng, 1024, 32768)
        sk += sq
        causal = True
    elif kind == "decode":
        d = rng.choice((64, 128, 128, 32 * rng.randint(1, 8)))
        sq, sk = rng.choice((1, 1, 1, 2, 4)), _log_int(rng, 256, 32768)
        causal = sq > 1
    elif kind == "i8":
        d = rng.choice((64, 128))
        if rng.random() < 0.5:  # prefill
            sq = sk = _log_int(rng, 128, 8192)
            causal = True
        else:  # decode, or a chunk against a longer cache
            sq, sk = rng.choice((1, 1, 4, _log_int(rng, 16, 512))), _log_int(rng, 512, 32768)
            causal = sq > 1
    else:
        d = rng.choice((64, 128))
        sq = sk = _log_int(rng, 128, 8192)
        causal = rng.random() < 0.75
        rope = rng.random() < 0.5
    case = _case(None, kind, b, hq, hkv, sq, sk, d, causal, window, rope)
    while True:
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case
        if case["b"] > 1:
            case["b"] //= 2
        elif case["sk"] == case["sq"]:
            case["sq"] = case["sk"] = int(case["sk"] * 0.7)
        else:
            case["sk"] = case["sq"] + int((case["sk"] - case["sq"]) * 0.7)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _rope_tables(rows, d, device):
    """cos/sin of position / 10000^(2i/d), float32 [rows, d/2]."""
    inv = 10000.0 ** (-torch.arange(0, d, 2, device=device, dtype=torch.float64) / d)
    ang = torch.arange(rows, device=device, dtype=torch.float64)[:, None] * inv
    return ang.cos().float(), ang.sin().float()


def _rows_int8(x):
    """x -> (int8, float32 scale per row), the per-token scheme."""
    s = x.abs().amax(-1, keepdim=True) / 127.0
    return torch.clamp(torch.round(x / s), -127, 127).to(torch.int8), s.squeeze(-1).contiguous()


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    b, hq, hkv, sq, sk, d = (case[k] for k in ("b", "hq", "hkv", "sq", "sk", "d"))

    def randn(*shape, dtype=torch.float16):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype)

    kind = case["kind"]
    state = {"case": case}
    if kind in ("extend", "decode"):
        cache = randn(b, sk, 2, hkv, d)
        state["q"] = randn(b, hq, sq, d)
        state["k"] = cache[:, :, 0].transpose(1, 2)
        state["v"] = cache[:, :, 1].transpose(1, 2)
        state["out"] = torch.empty_like(state["q"])
    elif kind == "prefill":
        std = 0.5 if d >= 256 else 1.0
        state["q"], state["k"], state["v"] = (randn(b, h, s, d) * std for h, s in ((hq, sq), (hkv, sk), (hkv, sk)))
    else:
        # activations: V has channel offsets (what per-channel scales are for);
        # scores spread by 0.64, so that a row's largest probability does not
        # push most others below the scheme's step of 1/127
        q = randn(b, hq, sq, d, dtype=torch.float32) * 0.8
        k = randn(b, hkv, sk, d, dtype=torch.float32) * 0.8
        v = randn(b, hkv, sk, d, dtype=torch.float32) + randn(b, hkv, 1, d, dtype=torch.float32)
        if kind == "i8q":
            state["q"], state["k"], state["v"] = q.half(), k.half(), v.half()
        else:
            state["q"], state["q_scale"] = _rows_int8(q)
            state["k"], state["k_scale"] = _rows_int8(k)
            state["v_scale"] = 6.0 / 127.0
            state["v"] = torch.clamp(torch.round(v / state["v_scale"]), -127, 127).to(torch.int8)
    if case["rope"]:
        state["cos"], state["sin"] = _rope_tables(max(sq, sk), d, dev)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    q, k, v = state["q"], state["k"], state["v"]
    opts = {"is_causal": case["causal"], "window_size": case["window"]}
    if kind == "i8":
        return rdnattention.flash_attn_int8qk(q, k, v, state["q_scale"], state["k_scale"], state["v_scale"], **opts)
    if case["rope"]:
        opts["rot_cos"], opts["rot_sin"] = state["cos"], state["sin"]
    if kind == "i8q":
        return rdnattention.flash_attn_int8qk_quantized(q, k, v, **opts)
    if kind == "prefill":
        return rdnattention.flash_attn(q, k, v, **opts)
    rdnattention.attention_forward_into(q, k, v, state["out"], **opts)
    return state["out"]


# ---------------------------------------------------------------------------
# work and accuracy
# ---------------------------------------------------------------------------
def _bounds(case, rows):
    """First and last visible key of each query row (a tensor of row numbers):
    causal rows end at the last key, a causal window counts back from there,
    a two-sided one spans window / 2 keys each way."""
    sq, sk, w = case["sq"], case["sk"], case["window"]
    at = rows + (sk - sq)
    lo, hi = torch.zeros_like(at), torch.full_like(at, sk - 1)
    if case["causal"]:
        hi = torch.minimum(hi, at)
    if w > 0:
        lo = torch.maximum(lo, at - w + 1 if case["causal"] else at - w // 2)
        if not case["causal"]:
            hi = torch.minimum(hi, at + w // 2)
    return lo, hi


def work(case):
    b, hq, hkv, sq, sk, d = (case[k] for k in ("b", "hq", "hkv", "sq", "sk", "d"))
    lo, hi = _bounds(case, torch.arange(sq, dtype=torch.int64))
    pairs = int((hi - lo + 1).clamp(min=0).sum())
    keys = int(hi.max() - lo.min() + 1)  # keys that some row sees
    in_size = 1 if case["kind"] == "i8" else 2
    size = b * hq * sq * d * (in_size + 2) + 2 * b * hkv * keys * d * in_size
    if case["kind"] == "i8":
        size += 4 * b * (hq * sq + hkv * keys)
    if case["rope"]:
        size += 2 * max(sq, sk) * (d // 2) * 4
    return {"bytes": size, "flops": 4 * b * hq * pairs * d}


def tolerance(case):
    # Against float64, fp16 kernels are 2.5e-4 to 3.7e-4 off (fp16 inputs,
    # probabilities and output, fp32 sums) and INT8 ones 3e-4 to 9e-4
    # (probabilities are rounded to 1/127 of the largest one seen so far,
    # which another order of the keys changes): about four times that.
    if case["kind"] in ("i8", "i8q"):
        return {"rel": 5.0e-3, "max": 0.1}
    return {"rel": 1.5e-3, "max": 0.03}


def _rotate(x, cos, sin):
    """RoPE of interleaved channel pairs, position = row."""
    n = x.shape[-2]
    c, s = cos[:n].double(), sin[:n].double()
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)


def _quantised(x, dim):
    """x rounded to its int8 grid along `dim`, as float64."""
    s = x.float().abs().amax(dim, keepdim=True) * (1.0 / 127.0)
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(x.float() / s), -127, 127).double() * s.double()


def exact(case, seed):
    """softmax(Q K^T / sqrt(d)) V in float64 on the same numbers (for INT8: on
    the dequantised ones, with unrounded probabilities)."""
    st = prepare(case, seed)
    b, hq, hkv, sq, sk, d = (case[k] for k in ("b", "hq", "hkv", "sq", "sk", "d"))
    out = torch.empty(b, hq, sq, d, dtype=torch.float64, device=st["q"].device)
    block = max(1, min(sq, (1 << 28) // (8 * sk)))  # rows per step: 256 MB of scores
    for ib in range(b):
        for ih in range(hq):
            jh = ih // (hq // hkv)
            q, k, v = st["q"][ib, ih].double(), st["k"][ib, jh].double(), st["v"][ib, jh].double()
            if case["kind"] == "i8":
                q = q * st["q_scale"][ib, ih].double()[:, None]
                k = k * st["k_scale"][ib, jh].double()[:, None]
                v = v * st["v_scale"]
            if case["rope"]:
                q, k = _rotate(q, st["cos"], st["sin"]), _rotate(k, st["cos"], st["sin"])
            if case["kind"] == "i8q":
                if case["rope"]:  # the rotated rows are fp16 before they are quantised
                    q, k = q.half().double(), k.half().double()
                q, k, v = _quantised(q, -1), _quantised(k, -1), _quantised(v, -2)
            kt = k.t().contiguous()
            for r in range(0, sq, block):
                rows = torch.arange(r, min(r + block, sq), device=out.device)
                lo, hi = _bounds(case, rows)
                c0, c1 = int(lo.min()), int(hi.max()) + 1
                s = (q[r:r + block] @ kt[:, c0:c1]) * d ** -0.5
                keys = torch.arange(c0, c1, device=out.device)
                s.masked_fill_((keys < lo[:, None]) | (keys > hi[:, None]), -math.inf)
                out[ib, ih, r:r + block] = torch.softmax(s, -1) @ v[c0:c1]
    return out
