"""Permutations that have nothing to do (a B-tree of one node, a key or none) are
accepted on a stream that is being captured, as any call that only enqueues."""
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,b,n", [("btree", 16, 16), ("btree", 4096, 2000), ("bst", 1, 1)])
def test_nothing_to_permute(layout, b, n, dev):
    A = torch.arange(n, dtype=torch.int64, device=dev)
    tl_amd.permute(layout, A, b)   # the library's context is there
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        A.add_(1)
        tl_amd.permute(layout, A, b, timed=False)
        tl_amd.unpermute(layout, A, b, timed=False)
    for k in (1, 2):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(A, torch.arange(k, n + k, dtype=torch.int64, device=dev))
