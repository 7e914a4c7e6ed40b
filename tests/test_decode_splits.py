"""How the decode attention's contexts are split (host arithmetic; the kernels are tested on the GPU)."""
import pytest

from mini_inference_engine_amd.kernels.hip_backend import HipBackend


@pytest.mark.parametrize("heads", [(32, 4, 64), (32, 8, 128), (32, 32, 128), (34, 1, 64)])
@pytest.mark.parametrize("rows", [1, 3, 6, 10, 28, 64, 300])
@pytest.mark.parametrize("bound", [1, 31, 512, 2048, 8192])
def test_splits_cover_the_context_within_two_workgroups_a_unit(heads, rows, bound):
    Hq, Hkv, D = heads
    block = 32
    keys, splits = HipBackend.decode_splits(HipBackend, rows, Hq, Hkv, bound, None, block, D)
    base = rows * Hkv * -(-(Hq // Hkv) // 16)
    assert keys % block == 0 and keys * (splits - 1) < bound <= keys * splits
    assert splits == 1 or base * splits <= HipBackend.DECODE_TARGET_WORKGROUPS
