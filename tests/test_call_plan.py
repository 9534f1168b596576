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
