"""Split keys and decode where their edges are: windows, rows without keys, splits
that end empty, the shortest caches; each case asserts the kernels it takes
(rdna_attention_call_plan), so that a line moved elsewhere shows here."""
import numpy as np
import pytest
import torch

import oracle
from tests.gpu_util import (DECODE, I8_MAX_ABS, SPLIT, assert_f16_parity, call_plan, errors, forward_raw, log,
                            reference_f16, seeded_inputs)

pytestmark = pytest.mark.gpu


# d, hq, hkv, sq, sk, causal, window: windows that leave whole splits unseen by
# some rows, and rows above the cache, whose splits are all empty
F16_SPLIT = [(d, 4, 2, 100, 3000, True, 900) for d in (32, 64, 96, 128, 160, 256)] + [
    (64, 4, 2, 300, 5000, True, 1500), (128, 4, 2, 100, 3000, False, 1200), (256, 4, 2, 100, 3000, False, 1200),
    (64, 2, 2, 3000, 2900, True, -1), (128, 2, 2, 3000, 2900, True, -1), (192, 2, 2, 3000, 2900, True, -1),
    (128, 2, 2, 3000, 2900, False, 1500)]


@pytest.mark.parametrize("case", F16_SPLIT, ids=["d{}h{}kv{}q{}k{}c{:d}w{}".format(*c) for c in F16_SPLIT])
def test_f16_split_keys(gpu, oracle_lib, case):
    d, hq, hkv, sq, sk, causal, window = case
    form, splits, _ = call_plan(False, 1, hq, hkv, sq, sk, d, causal, window)
    log(f"[f16 split] {case} splits {splits}")
    assert form == SPLIT and splits > 1
    q, k, v = seeded_inputs(81, 1, hq, hkv, sq, sk, d)
    out = torch.full_like(q, 7.0, device=gpu)
    assert forward_raw(q.to(gpu), k.to(gpu), v.to(gpu), out, causal, window) == 0
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    assert_f16_parity(got, reference_f16(q, k, v, causal, window), "split")
    if causal and sq > sk:
        assert np.all(got[:, :, : sq - sk] == 0)


# b, hq, hkv, sq, sk, d, causal, window, V scales, form: the same of INT8, and
# decode on caches of one key to a few tiles (4 columns and 32 in the scratch)
INT8_FORMS = [(1, 4, 2, 300, 5000, d, True, 1500, sc, SPLIT) for d, sc in ((64, "one"), (128, "vtoken"))] + [
    (1, 2, 2, 3000, 2900, d, True, -1, sc, SPLIT) for d, sc in ((64, "vtoken"), (128, "channel"))] + [
    (128, 8, 8, 1, sk, d, False, -1, sc, DECODE) for d in (64, 128)
    for sk, sc in ((1, "one"), (63, "vtoken"), (64, "channel"), (65, "one"), (130, "vtoken"))] + [
    (40, 64, 8, 1, sk, d, False, -1, sc, DECODE) for d in (64, 128)
    for sk, sc in ((1, "channel"), (64, "one"), (129, "vtoken"))] + [
    (40, 64, 8, 4, 3, 64, True, -1, "one", DECODE),  # the first row sees no key
    (1, 4, 2, 3, 4000, 64, False, 1300, "channel", DECODE),
    (1, 8, 8, 32, 1111, 128, True, 700, "one", DECODE)]


@pytest.mark.parametrize("case", INT8_FORMS, ids=["b{}h{}kv{}q{}k{}d{}c{:d}w{}{}".format(*c) for c in INT8_FORMS])
def test_int8_forms(gpu, oracle_lib, case):
    """The kernel-exact emulation, to the INT8 bar and 2e-3 of the largest output (the
    same P in another order of the sums)."""
    import rdnattention as ra

    b, hq, hkv, sq, sk, d, causal, window, scales, form = case
    got_form, splits, _ = call_plan(True, b, hq, hkv, sq, sk, d, causal, window)
    log(f"[int8 forms] {case} splits {splits}")
    assert got_form == form and (form != SPLIT or splits > 1)
    rng = np.random.default_rng(82)
    qi, qs = oracle.quant_pertoken(rng.standard_normal((b, hq, sq, d)).astype(np.float32))
    ki, ks = oracle.quant_pertoken(rng.standard_normal((b, hkv, sk, d)).astype(np.float32))
    vi = rng.integers(-127, 128, (b, hkv, sk, d), dtype=np.int8)
    vs = 1.0 / 127.0
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    extra, vtok, vch = {}, None, None
    if scales == "vtoken":
        vtok = rng.uniform(0.2, 1.0, (b, hkv, sk)).astype(np.float32)
        extra["v_token"] = t(vtok)
    elif scales == "channel":
        vch = rng.uniform(0.2, 1.0, (b, hkv, d)).astype(np.float32)
        extra["v_channel"] = t(vch)
    outs = [torch.full((b, hq, sq, d), float("nan"), dtype=torch.float16, device=gpu) for _ in range(2)]
    for o in outs:
        ra.attention_int8_forward_into(t(qi), t(ki), t(vi), o, t(qs), t(ks), vs, is_causal=causal,
                                       window_size=window, **extra)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    got = outs[0].float().cpu().numpy()
    emu = oracle.attention_int8(qi, ki, vi, qs, ks, vs, causal=causal, window=window, v_token=vtok)
    if vch is not None:
        emu = emu * np.repeat(vch, hq // hkv, axis=1)[:, :, None, :]
    assert np.isfinite(got).all()
    mx, _, _ = errors(got, emu)
    assert mx <= min(I8_MAX_ABS, 2e-3 * np.abs(emu).max()), f"max_abs {mx:.3e} of {np.abs(emu).max():.3e}"


# int8, b, hq, hkv, sq, sk, d, form: every call with scratch for split keys
SCRATCH_CALLS = [(False, 1, 8, 2, 70, 3000, 64, SPLIT), (False, 1, 8, 2, 70, 3000, 256, SPLIT),
                 (False, 1, 8, 2, 2, 5000, 96, DECODE), (False, 2, 16, 2, 1, 3000, 256, DECODE),
                 (True, 1, 8, 2, 70, 3000, 64, SPLIT), (True, 1, 8, 2, 70, 3000, 128, SPLIT),
                 (True, 2, 8, 2, 1, 5000, 128, DECODE), (True, 2, 8, 2, 4, 5000, 64, DECODE)]


@pytest.mark.parametrize("case", SCRATCH_CALLS, ids=["i{:d}b{}h{}kv{}q{}k{}d{}f{}".format(*c) for c in SCRATCH_CALLS])
def test_split_key_calls_captured_and_on_streams(gpu, case):
    """The scratch of split keys in a captured graph, replayed three times with eager
    calls on other inputs between the replays, and in calls on three streams at
    once: the eager call's bits each time."""
    import rdnattention as ra

    int8, b, hq, hkv, sq, sk, d, form = case
    log(f"[split scratch] {case}")
    got_form, _, scratch = call_plan(int8, b, hq, hkv, sq, sk, d)
    assert got_form == form and scratch > 0
    g = torch.Generator(device=gpu).manual_seed(83)
    draw = (lambda *s: torch.randint(-127, 128, s, generator=g, device=gpu, dtype=torch.int8)) if int8 else (
        lambda *s: torch.randn(*s, generator=g, device=gpu).half())
    inputs = [(draw(b, hq, sq, d), draw(b, hkv, sk, d), draw(b, hkv, sk, d)) for _ in range(3)]

    def run(i, out):
        if int8:
            ra.attention_int8_forward_into(*inputs[i], out, 0.01, 0.01, 1 / 127)
        else:
            ra.attention_forward_into(*inputs[i], out)

    want = [torch.empty(b, hq, sq, d, dtype=torch.float16, device=gpu) for _ in inputs]
    for i, w in enumerate(want):
        run(i, w)
    torch.cuda.synchronize()
    assert not torch.equal(want[0], want[1])

    captured, other = torch.empty_like(want[0]), torch.empty_like(want[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(0, captured)
    for i in (1, 2, 1):
        captured.zero_()
        run(i, other)
        graph.replay()
        run(i, other)
        torch.cuda.synchronize()
        assert torch.equal(captured, want[0]) and torch.equal(other, want[i])

    streams = [torch.cuda.Stream() for _ in inputs]
    outs = [torch.empty_like(want[0]) for _ in inputs]
    torch.cuda.synchronize()
    for rep in range(5):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                run((i + rep) % 3, outs[i])
        torch.cuda.synchronize()
        for i, o in enumerate(outs):
            assert torch.equal(o, want[(i + rep) % 3])
