"""Permutations through the stash in one pass (at most 2^24 keys) against the
oracle's layouts, around the tiles' and the path's edges, and the plans forced
at sizes that the direct path now serves; a captured call is refused."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
import tl_amd

pytestmark = pytest.mark.gpu

LAYOUTS = [("bst", 1), ("btree", 1), ("btree", 2), ("btree", 16), ("btree", 100),
           ("btree", 4096), ("mveb", 1), ("veb", 1)]


def check(layout, b, n, dtype, dev):
    ranks = ol.layout_ranks(layout, n, b).astype(np.int64)
    A = torch.arange(n, dtype=dtype, device=dev)
    tl_amd.permute(layout, A, b)
    assert np.array_equal(A.cpu().numpy(), ranks.astype(A.cpu().numpy().dtype)), (layout, b, n)
    tl_amd.unpermute(layout, A, b)
    assert torch.equal(A, torch.arange(n, dtype=dtype, device=dev)), (layout, b, n)


@pytest.mark.parametrize("plan", [False, True])
@pytest.mark.parametrize("layout,b", LAYOUTS)
def test_sizes(layout, b, plan, dev, monkeypatch):
    if plan:
        monkeypatch.setenv("TL_PERMUTE_PLAN", "1")
    for k, n in enumerate([2, 5, 255, 2047, 2049, 16384, 16385, 100003, 1000003]):
        check(layout, b, n, (torch.int32, torch.int64)[k % 2], dev)


@pytest.mark.parametrize("layout,b", [("bst", 1), ("btree", 16), ("mveb", 1)])
def test_path_edge(layout, b, dev):
    for n, dtype in [(1 << 24, torch.int64), ((1 << 24) + 1, torch.int32)]:
        check(layout, b, n, dtype, dev)


def test_capture_is_refused(dev):
    A = torch.arange(5000, dtype=torch.int64, device=dev)
    tl_amd.permute_btree(A, 16)   # the scratch is there
    tl_amd.unpermute("btree", A, 16)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with pytest.raises(tl_amd.TLError):
            tl_amd.permute_btree(A, 16, timed=False)
    torch.cuda.synchronize()
    assert torch.equal(A, torch.arange(5000, dtype=torch.int64, device=dev))
