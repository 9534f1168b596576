"""Which kernels a call takes (rdna_attention_call_plan), without a GPU."""
import pytest

from tests.gpu_util import ALTERNATE, DECODE, SPLIT, WHOLE, call_plan


# int8, hkv per batch entry, sk, d
@pytest.mark.parametrize("int8,hkv,sk,d", [(True, 8, 64, 64), (True, 1, 8192, 128), (False, 8, 512, 96),
                                           (False, 8, 600, 128), (False, 1, 1024, 192)])
def test_decode_grid_limit(int8, hkv, sk, d):
    """The decode grids have the kv heads in y, of which HIP allows 65535: calls
    with more take the prefill kernels, whose grids have one dimension."""
    for b in (65536 // hkv, 100000 // hkv):
        form, splits, scratch = call_plan(int8, b, 4 * hkv, hkv, 1, sk, d)
        assert form != DECODE and splits == 1 and scratch == 0


# b, hkv, rows per kv head, sk, d, causal, window
INT8_SCRATCH = [(4096, 8, 8, 64, 64, False, -1), (8191, 8, 32, 120, 128, False, -1), (512, 8, 1, 1, 64, False, -1),
                (1024, 8, 4, 700, 128, True, -1), (64, 8, 16, 9001, 128, False, -1), (16, 8, 2, 4000, 64, True, 300),
                (128, 8, 32, 8192, 64, False, -1), (8, 8, 1, 300000, 128, False, -1)]


@pytest.mark.parametrize("case", INT8_SCRATCH, ids=["b{}kv{}m{}k{}d{}c{:d}w{}".format(*c) for c in INT8_SCRATCH])
def test_int8_decode_scratch(case):
    """Scores and block maxima are taken for the 64-key blocks that some row sees,
    whatever the splits, and never above 1 GiB."""
    b, hkv, m, sk, d, causal, window = case
    ratio = m // 2 if causal else m
    form, splits, scratch = call_plan(True, b, ratio * hkv, hkv, m // ratio, sk, d, causal, window)
    if form != DECODE:
        return
    lo = max(0, sk - m // ratio - window + 1) if window > 0 else 0
    blocks = (sk - 1) // 64 + 1 - lo // 64
    scores = b * hkv * blocks * 65 * (4 if m <= 4 else 32) * 4
    assert scores <= 1 << 30
    partials = splits * b * hkv * m * (d + 2) * 4 if splits > 1 else 0  # with a device
    assert scratch == scores + partials


# b, hkv, query heads per kv head, rows, sk, d: the calls that were slower on the
# decode kernels than on the prefill kernels, and their neighbours that are not
@pytest.mark.parametrize("b,hkv,ratio,sq,sk,d,decode", [
    (1, 8, 1, 1, 64, 64, False), (1, 8, 4, 1, 384, 128, False), (1, 8, 4, 1, 600, 64, True), (1, 8, 4, 1, 512, 128, True),
    (64, 8, 1, 1, 64, 128, False), (64, 8, 1, 1, 256, 128, True), (512, 8, 1, 1, 1, 64, True),
    (128, 8, 4, 2, 1, 128, False), (128, 8, 4, 4, 64, 64, False), (128, 8, 4, 4, 256, 64, True),
    (32, 8, 4, 8, 512, 128, False), (32, 8, 1, 32, 2048, 64, False), (16, 8, 4, 8, 2048, 128, True),
    (40, 8, 4, 2, 448, 64, True), (24, 8, 4, 4, 16384, 64, False), (16, 8, 4, 4, 16384, 64, True),
    (128, 8, 1, 32, 512, 128, False), (512, 8, 1, 32, 1024, 128, True), (24, 8, 8, 1, 1, 128, False),
    (80, 8, 8, 1, 1, 128, True)])
def test_int8_decode_line(b, hkv, ratio, sq, sk, d, decode):
    assert (call_plan(True, b, ratio * hkv, hkv, sq, sk, d)[0] == DECODE) == decode


def test_int8_decode_line_counts_visible_keys():
    """A window that leaves few keys of a long cache."""
    assert call_plan(True, 1, 32, 8, 1, 100000, 128, True, 200)[0] != DECODE
    assert call_plan(True, 1, 32, 8, 1, 100000, 128, True, 2000)[0] == DECODE


# int8, b, hq, hkv, sq, sk, d
@pytest.mark.parametrize("case,form", [
    ((False, 64, 8, 8, 64, 400, 32), WHOLE), ((False, 32, 8, 8, 64, 400, 32), ALTERNATE),
    ((False, 32, 8, 8, 64, 512, 128), WHOLE), ((False, 16, 8, 8, 64, 512, 128), ALTERNATE),
    ((False, 32, 32, 8, 9, 400, 128), WHOLE), ((False, 64, 8, 8, 64, 1024, 64), ALTERNATE),
    ((True, 64, 8, 8, 33, 130, 128), WHOLE), ((True, 64, 8, 8, 33, 400, 128), ALTERNATE)])
def test_alternate_line(case, form):
    """Rows that fill at most half a row tile, and D = 32, whose workgroups share a
    CU: where alternating groups were slower than whole row tiles, and not."""
    assert call_plan(*case)[0] == form
