"""tl_release_scratch: what permutations, the sort and partitioned lookups keep for
the next call goes back to the device, and the calls work again after it."""
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu


def test_release_gives_memory_back(dev, monkeypatch):
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    n, nq = 50_000_017, 1 << 24
    keys = torch.arange(n, dtype=torch.int64, device=dev)
    A, S = keys.clone(), keys.clone()
    Q = torch.randint(0, n, (nq,), device=dev)
    ans = torch.empty_like(Q)
    torch.cuda.synchronize()
    left = []
    for _ in range(3):   # the first also loads the kernels, which stay
        A.copy_(keys)
        tl_amd.permute_btree(A, 16)
        S.copy_(keys)
        m, _ = tl_amd.sort_dedupe(S)
        assert m == n and torch.equal(S, keys)
        tl_amd.query_btree(A, 16, Q, ans)
        assert torch.equal(A[ans], Q)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        before = torch.cuda.mem_get_info(dev)[0]
        tl_amd.release_scratch()
        left.append(torch.cuda.mem_get_info(dev)[0])
        assert left[-1] - before > 500 << 20   # the sort's second buffer, a stash, a workspace
    assert left[2] == left[1] == left[0], left


def test_somewhat_larger_batch_needs_no_new_workspace(dev, monkeypatch):
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    n, nq = 5_000_011, 1 << 24
    A = torch.arange(n, dtype=torch.int64, device=dev)
    tl_amd.permute_btree(A, 16)
    Q = torch.randint(0, n, (nq + nq // 8,), device=dev)
    ans = torch.empty_like(Q)
    tl_amd.release_scratch()
    tl_amd.query_btree(A, 16, Q[:nq], ans)
    free = torch.cuda.mem_get_info(dev)[0]
    tl_amd.query_btree(A, 16, Q, ans)
    assert torch.cuda.mem_get_info(dev)[0] == free
    tl_amd.release_scratch()
