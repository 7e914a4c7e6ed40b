"""How the decode attention's contexts are split, and which pages prompt attention takes out of caches that it cannot load from where
they lie (host arithmetic; the kernels are tested on the GPU)."""
from types import SimpleNamespace

import pytest
import torch

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


# rows of the step, single tokens among them, the longest context said, pages of the cache; whether the pages are taken one by one
@pytest.mark.parametrize("case", [(3, 1, 40, 64, True), (3, 1, 0, 64, True), (2, 0, 96, 64, True), (2, 0, 96, 12, False), (9, 1, 96, 48, False),
                                  (9, 1, 96, 49, True)])
def test_pages_of_portions_are_never_more_than_the_caches(case):
    """The tables that come back lead to the same keys and values for every page of a row's own; what a table holds behind those is
    never looked up; and no more pages are copied than the caches have."""
    rows, single, context, pages, few = case
    page, width = 16, 6
    k = torch.arange(pages * 2 * page * 4, dtype=torch.float32).view(pages, 2, page, 4)
    bt = torch.randint(0, pages, (rows, width), generator=torch.Generator().manual_seed(rows), dtype=torch.int32)
    own = [1 + r % (-(-context // page) if context else width) for r in range(rows)]
    for r in range(rows):
        bt[r, own[r]:] = -1 if r % 2 else 1 << 30
    step = SimpleNamespace(num_rows=rows, num_decode_rows=single, max_context=context)
    keys, values, table = HipBackend._pages_of_portions(k, -k, bt, step, page)
    assert keys.data_ptr() != k.data_ptr() and keys.shape[0] <= pages and (table is not bt) == few
    for r in range(single, rows):
        there, here = bt[r, :own[r]].long(), table[r, :own[r]].long()
        assert torch.equal(keys[here], k[there]) and torch.equal(values[here], -k[there])
