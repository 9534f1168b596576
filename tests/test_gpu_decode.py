"""Split-K decode path on the GPU against the CPU oracle.

The reference has no split-K kernel (docs/api.md:203-204); its decode shapes
run through the same FP16 entry point, so the bar is the FP16 one: max-abs
<= 2e-3, mean-abs <= 2e-4 and rel_rms < 5e-3 against the oracle on the same
inputs, for every mask mode, GQA ratio and stride layout the entry point
accepts.  The prefill kernel is run on the same inputs as a second path.
"""
import numpy as np
import pytest
import torch

import oracle
from tests.gpu_util import DECODE, assert_f16_parity, call_plan, forward_raw, log, reference_f16, seeded_inputs

pytestmark = pytest.mark.gpu

PATH_PREFILL, PATH_SPLITK = 1, 2

# b, hq, hkv, sq, sk, d, causal, window, rope
CASES = [
    (2, 8, 2, 1, 1000, 64, False, -1, False),
    (2, 8, 2, 4, 3000, 128, False, -1, False),
    (1, 32, 8, 1, 32768, 128, False, -1, False),
    (1, 32, 8, 4, 8192, 128, False, -1, False),
    (1, 32, 1, 1, 5000, 128, False, -1, False),   # MQA, 32 columns
    (1, 16, 2, 4, 2048, 64, False, -1, False),    # ratio 8 x Sq 4 = 32 columns
    (2, 4, 4, 3, 777, 32, False, -1, False),
    (2, 8, 2, 4, 3000, 128, True, -1, False),     # causal decode: last keys masked per row
    (1, 8, 2, 4, 3000, 128, True, 700, False),    # causal window
    (1, 8, 2, 2, 3000, 64, False, 900, False),    # two-sided window
    (1, 8, 2, 1, 2500, 128, False, -1, True),     # RoPE (Q row 0, K rows 0..Sk-1)
    (1, 4, 2, 5, 40, 64, True, -1, False),        # short: fewer keys than one wave round
]


@pytest.mark.parametrize("case", CASES, ids=[f"b{c[0]}h{c[1]}kv{c[2]}q{c[3]}k{c[4]}d{c[5]}c{int(c[6])}w{c[7]}r{int(c[8])}"
                                             for c in CASES])
def test_splitk_vs_oracle(gpu, oracle_lib, case):
    b, hq, hkv, sq, sk, d, causal, window, rope = case
    log(f"[splitk] {case}")
    q, k, v = seeded_inputs(21, b, hq, hkv, sq, sk, d)
    cos = sin = None
    if rope:
        cos, sin = oracle.rope_tables(max(sq, sk), d)
    ref = reference_f16(q, k, v, causal, window, cos, sin)
    cd = torch.from_numpy(cos).to(gpu) if rope else None
    sd = torch.from_numpy(sin).to(gpu) if rope else None
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    outs = {}
    for path in (PATH_SPLITK, PATH_PREFILL, 0):
        o = torch.full_like(qd, float("nan"))
        assert forward_raw(qd, kd, vd, o, causal, window, cd, sd, path=path) == 0
        outs[path] = o
    torch.cuda.synchronize()
    for path, o in outs.items():
        assert_f16_parity(o.float().cpu().numpy(), ref, f"path{path}")


def test_splitk_strided_cache_views(gpu, oracle_lib):
    """K/V sliced from one [B, S, 2, Hkv, D] cache (the decode benchmark's layout)."""
    g = torch.Generator().manual_seed(3)
    b, hq, hkv, sq, sk, d = 2, 16, 4, 4, 4096, 128
    buf = torch.randn(b, sk, 2, hkv, d, generator=g).half()
    q = torch.randn(b, hq, sq, d, generator=g).half()
    bd = buf.to(gpu)
    kv_k = bd[:, :, 0].transpose(1, 2)
    kv_v = bd[:, :, 1].transpose(1, 2)
    o1 = torch.empty(b, hq, sq, d, dtype=torch.float16, device=gpu)
    o2 = torch.empty_like(o1)
    qd = q.to(gpu)
    assert forward_raw(qd, kv_k, kv_v, o1, path=PATH_SPLITK) == 0
    assert forward_raw(qd, kv_k.contiguous(), kv_v.contiguous(), o2, path=PATH_SPLITK) == 0
    torch.cuda.synchronize()
    assert torch.equal(o1, o2)
    ref = reference_f16(q, buf[:, :, 0].transpose(1, 2), buf[:, :, 1].transpose(1, 2), False, -1)
    assert_f16_parity(o1.float().cpu().numpy(), ref, "strided_cache")


def test_splitk_rows_without_keys(gpu):
    """Causal with Sq > Sk through split-K: rows above the cache write 0."""
    q, k, v = seeded_inputs(5, 1, 4, 4, 8, 3, 64)
    out = torch.full_like(q, 7.0, device=gpu)
    assert forward_raw(q.to(gpu), k.to(gpu), v.to(gpu), out, causal=True, path=PATH_SPLITK) == 0
    torch.cuda.synchronize()
    o = out.float().cpu().numpy()
    assert np.all(o[:, :, :5] == 0)
    assert_f16_parity(o, reference_f16(q, k, v, True, -1), "no_keys")


def test_splitk_unsupported_shape_is_rejected(gpu):
    q = torch.zeros(1, 8, 9, 128, dtype=torch.float16, device=gpu)  # ratio 4 x 9 rows = 36 columns > 32
    k = torch.zeros(1, 2, 100, 128, dtype=torch.float16, device=gpu)
    out = torch.empty_like(q)
    import rdnattention

    assert forward_raw(q, k, k, out, path=PATH_SPLITK) == -3
    assert "split-K" in rdnattention.last_error()
    assert forward_raw(q, k, k, out, path=0) == 0  # auto falls back to the prefill kernel


# d, b, hq, hkv, sq, sk, causal, window: every head dim the automatic choice
# sends to split-K, at the edges of its tiles (32 keys), rounds (32 keys per
# wave) and columns (1 .. 32 rows per kv head), with one split and several, and
# both sides of the lines where the choice goes to the prefill kernel
AUTO_CASES = [(d, 1, 8, 2, 1, 513, False, -1) for d in range(32, 257, 32)] + [
    (256, 2, 4, 4, 1, 2049, False, -1),
    (256, 1, 32, 1, 1, 4100, False, -1),
    (224, 1, 8, 8, 5, 1023, True, -1),
    (192, 2, 8, 2, 8, 3000, True, -1),
    (160, 1, 6, 2, 3, 1500, True, 600),
    (96, 3, 5, 1, 4, 777, True, -1),
    (96, 1, 8, 2, 2, 4000, False, 900),
    (128, 1, 32, 1, 1, 30000, False, -1),
    (128, 33, 8, 8, 1, 520, False, -1),
    (128, 1, 8, 2, 1, 128, False, -1),  # below the decode kernel's shortest cache, and just above it
    (128, 1, 8, 2, 1, 129, False, -1),
    (64, 3, 4, 2, 4, 300, True, -1),
    (192, 1, 16, 2, 4, 511, True, 200),
    (32, 33, 8, 8, 1, 200, False, -1),  # 264 kv heads: prefill
    (256, 1, 16, 2, 2, 700, True, -1),  # D > 192: eight query heads per kv head
    (256, 1, 4, 2, 1, 700, False, -1),  # and two
    (224, 64, 8, 8, 1, 512, False, -1),
]


@pytest.mark.parametrize("case", AUTO_CASES, ids=["d{}b{}h{}kv{}q{}k{}c{:d}w{}".format(*c) for c in AUTO_CASES])
def test_auto_decode_vs_oracle(gpu, oracle_lib, case):
    """FP16 bar against the oracle; a second call, the no-allocation entry point
    and a captured graph's replays give the same bits."""
    from tests.gpu_util import lib

    d, b, hq, hkv, sq, sk, causal, window = case
    log(f"[auto decode] {case}")
    q, k, v = seeded_inputs(31, b, hq, hkv, sq, sk, d)
    ref = reference_f16(q, k, v, causal, window)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    outs = [torch.full_like(qd, float("nan")) for _ in range(4)]
    for o in outs[:2]:
        assert forward_raw(qd, kd, vd, o, causal, window) == 0
    o = outs[2]
    qs, ks, vs, os_ = qd.stride(), kd.stride(), vd.stride(), o.stride()
    assert lib().rdna_attention_forward_noalloc(
        qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), o.data_ptr(), None, None, *qs[:3], *ks[:3], *vs[:3], *os_[:3],
        b, hq, hkv, sq, sk, d, d ** -0.5, int(causal), 0, window, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert forward_raw(qd, kd, vd, outs[3], causal, window) == 0
    for _ in range(3):
        outs[3].fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[3], outs[0])
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])
    assert_f16_parity(outs[0].float().cpu().numpy(), ref, "auto decode")


# d, b, hq, hkv, sq, sk, causal, window, rope: prefill launches too small for
# the CUs, whose keys are split (every head dim; one and several row tiles, splits
# that end short or empty, a window) or, of two, whose groups alternate (a window,
# rows without keys; those under split keys: test_gpu_forms.py)
SPLIT_PREFILL_CASES = [(d, 1, 8, 2, 70, 1500, True, -1, False) for d in range(32, 257, 32)] + [
    (128, 1, 8, 2, 257, 5000, True, -1, True),
    (128, 1, 4, 4, 33, 2049, False, -1, False),
    (64, 2, 4, 2, 300, 1111, True, 500, False),
    (256, 1, 4, 2, 129, 2600, True, -1, True),
    (192, 1, 4, 1, 200, 1900, False, 1000, False),
    (96, 1, 5, 1, 1500, 900, True, -1, False),
]


@pytest.mark.parametrize("case", SPLIT_PREFILL_CASES,
                         ids=["d{}b{}h{}kv{}q{}k{}c{:d}w{}r{:d}".format(*c) for c in SPLIT_PREFILL_CASES])
def test_split_prefill_vs_oracle(gpu, oracle_lib, case):
    """FP16 bar against the oracle; a second call gives the same bits."""
    d, b, hq, hkv, sq, sk, causal, window, rope = case
    log(f"[split prefill] {case}")
    q, k, v = seeded_inputs(51, b, hq, hkv, sq, sk, d)
    cos = sin = cd = sd = None
    if rope:
        cos, sin = oracle.rope_tables(max(sq, sk), d)
        cd, sd = torch.from_numpy(cos).to(gpu), torch.from_numpy(sin).to(gpu)
    ref = reference_f16(q, k, v, causal, window, cos, sin)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    outs = [torch.full_like(qd, float("nan")) for _ in range(2)]
    for o in outs:
        assert forward_raw(qd, kd, vd, o, causal, window, cd, sd) == 0
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert_f16_parity(outs[0].float().cpu().numpy(), ref, "split prefill")


# d, b, hq, hkv, sq, sk: split prefill (both kernels), decode with several splits
# and with one, alternating groups
NONFINITE_CASES = [(64, 1, 8, 2, 70, 3000), (128, 1, 8, 2, 70, 3000), (256, 1, 8, 2, 70, 3000),
                   (128, 1, 8, 2, 4, 8192), (96, 1, 8, 2, 1, 4000), (256, 1, 32, 2, 1, 5000),
                   (128, 32, 8, 8, 1, 512), (64, 1, 8, 8, 512, 512), (128, 1, 8, 8, 512, 512)]
NONFINITE = ["q_nan", "k_nan", "k_inf", "k_neg_inf", "k_lowest", "v_inf"]


@pytest.mark.parametrize("what", NONFINITE)
@pytest.mark.parametrize("case", NONFINITE_CASES, ids=["d{}b{}h{}kv{}q{}k{}".format(*c) for c in NONFINITE_CASES])
def test_nonfinite_through_the_merges(gpu, case, what):
    """NaN, infinities and lowest scores as torch's float32 softmax treats them: a
    query row of NaN is NaN and leaves the other rows alone; a key whose score is
    NaN or +inf makes every row NaN that sees it, also where its split's partial
    is one of many; keys at -inf (here all of the first splits') or at the lowest
    scores (all of the last splits') weigh nothing; an infinite V reaches the
    output.  (The lowest scores come last: a running maximum that starts at
    -1e5 leaves the scores of the tile that ends it 2^-7 apart.)"""
    d, b, hq, hkv, sq, sk = case
    log(f"[non-finite] {case} {what}")
    g = torch.Generator(device=gpu).manual_seed(61)
    q = torch.randn(b, hq, sq, d, generator=g, device=gpu).abs().half() * 0.3  # positive: the sign of a score is K's
    k = torch.randn(b, hkv, sk, d, generator=g, device=gpu).half() * 0.3
    v = torch.randn(b, hkv, sk, d, generator=g, device=gpu).half()
    if what == "q_nan":
        q[:, :, sq // 2] = float("nan")
    elif what == "k_nan":
        k[:, :, 100] = float("nan")
    elif what == "k_inf":
        k[:, :, 100] = float("inf")
    elif what == "k_neg_inf":
        k[:, :, : sk // 2] = float("-inf")
    elif what == "k_lowest":
        k[:, :, sk // 2:] = -65504.0
    else:
        v[:, :, 100] = float("inf")
    out = torch.full_like(q, 7.0)
    assert forward_raw(q, k, v, out) == 0
    torch.cuda.synchronize()
    kr = k.float().repeat_interleave(hq // hkv, dim=1).transpose(2, 3).contiguous()
    vr = v.float().repeat_interleave(hq // hkv, dim=1)
    ref = torch.softmax(torch.matmul(q.float(), kr) * d ** -0.5, dim=-1)
    ref = torch.matmul(ref, vr)
    got = out.float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isposinf(got), torch.isposinf(ref))
    finite = torch.isfinite(ref)
    if finite.any():
        assert_f16_parity(got[finite].cpu().numpy(), ref[finite].cpu().numpy(), what)


@pytest.mark.parametrize("int8,d,sk", [(False, 96, 512), (False, 64, 600), (True, 64, 24), (True, 128, 70)])
def test_more_kv_heads_than_a_grid_dimension(gpu, int8, d, sk):
    """65536 (batch, kv head) pairs, one above what HIP allows in y, on one K and V
    (batch stride 0): every batch entry gives the bits of the first, which agrees
    with a call for it alone (decode kernels)."""
    import rdnattention as ra

    b, h = 8192, 8
    log(f"[kv heads] int8={int8} d{d} sk{sk}")
    g = torch.Generator(device=gpu).manual_seed(71)
    draw = (lambda *s: torch.randint(-127, 128, s, generator=g, device=gpu, dtype=torch.int8)) if int8 else (
        lambda *s: torch.randn(*s, generator=g, device=gpu).half())
    q, k, v = (draw(1, h, s, d) for s in (1, sk, sk))
    outs = []
    for n in (1, b):
        qn, kn, vn = (t.expand(n, -1, -1, -1) for t in (q, k, v))
        out = torch.full((n, h, 1, d), float("nan"), dtype=torch.float16, device=gpu)
        if int8:
            ra.attention_int8_forward_into(qn, kn, vn, out, 0.01, 0.01, 1 / 127)
        else:
            ra.attention_forward_into(qn, kn, vn, out)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[1], outs[1][:1].expand_as(outs[1]))
    diff = (outs[1][0].float() - outs[0][0].float()).abs().max().item()
    assert diff <= 2e-3, diff  # another order of the sums; the same INT8 P


@pytest.mark.parametrize("d,b,sk,lo,hi", [
    (128, 8, 8198, 4, 4), (128, 16, 2082, 1, 2), (128, 16, 32768, 2, 2), (128, 1, 512, 1, 1), (64, 20, 7166, 3, 3),
    (64, 12, 7447, 5, 5), (128, 3, 4000, 8, 10), (256, 8, 6001, 3, 4)])
def test_decode_splits(gpu, d, b, sk, lo, hi):
    """Eight kv heads per batch entry on 256 CUs: as many splits as fill whole rounds
    of workgroups, or every CU alike."""
    form, splits, scratch = call_plan(False, b, 64 if d > 192 else 8, 8, 1, sk, d)
    log(f"[decode splits] d{d} b{b} sk{sk}: {splits}")
    assert form == DECODE and lo <= splits <= hi
    assert scratch == (splits * b * (64 if d > 192 else 8) * (d + 2) * 4 if splits > 1 else 0)


# d, b, hq, hkv, sk: rows that end inside a 128-byte line, whose heads go to the XCDs
# in pairs where those fill whole rounds (the first two of each head dim) or not
@pytest.mark.parametrize("case", [(d, *c) for d in (32, 96, 160, 224)
                                  for c in ((2, 64, 8, 700), (4, 64, 4, 3000), (1, 64, 6, 900), (3, 20, 2, 2500))],
                         ids=lambda c: "d{}b{}h{}kv{}k{}".format(*c))
def test_decode_cache_views_every_head_dim(gpu, case):
    """K/V as views of one [B, S, 2, Hkv, D] cache: the bits of contiguous tensors."""
    d, b, hq, hkv, sk = case
    hq = hq // hkv * hkv
    assert call_plan(False, b, hq, hkv, 1, sk, d)[0] == DECODE
    g = torch.Generator(device=gpu).manual_seed(91)
    cache = torch.randn(b, sk, 2, hkv, d, generator=g, device=gpu).half()
    q = torch.randn(b, hq, 1, d, generator=g, device=gpu).half()
    k, v = cache[:, :, 0].transpose(1, 2), cache[:, :, 1].transpose(1, 2)
    outs = [torch.full_like(q, float("nan")) for _ in range(2)]
    assert forward_raw(q, k, v, outs[0]) == 0
    assert forward_raw(q, k.contiguous(), v.contiguous(), outs[1]) == 0
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    kr = k.float().repeat_interleave(hq // hkv, dim=1).transpose(2, 3).contiguous()
    vr = v.float().repeat_interleave(hq // hkv, dim=1)
    ref = torch.matmul(torch.softmax(torch.matmul(q.float(), kr) * d ** -0.5, dim=-1), vr)
    assert_f16_parity(outs[0].float().cpu().numpy(), ref.cpu().numpy(), "cache views")
