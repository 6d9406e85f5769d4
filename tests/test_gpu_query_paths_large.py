"""Large batches over large arrays: the plain descents, which small batches, captured
streams and short memory take, give the answers of the other paths and of the keys
themselves; and the variables that shape the plain descents keep them at every
size (no workspace is taken then)."""
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu

I, L = torch.int32, torch.int64


def lookup(layout, b, A, Q, ans, tables):
    if layout == "bst":
        tl_amd.query_bst(A, Q, ans)
    elif layout == "btree":
        tl_amd.query_btree(A, b, Q, ans)
    elif layout == "sorted":
        tl_amd.query_binary(A, Q, ans)
    else:
        query = tl_amd.query_mveb_nonperfect if layout == "mveb" else tl_amd.query_veb_nonperfect
        query(A, *tables, Q, ans)


@pytest.mark.parametrize("layout,b,n,dtype", [
    ("bst", 1, 1 << 30, L), ("btree", 16, 1 << 30, L), ("btree", 8, 300_000_007, I),
    ("btree", 33, 100_000_007, L), ("mveb", 1, 300_000_000, L), ("veb", 1, 300_000_000, I),
    ("sorted", 1, 1 << 30, L)])
def test_paths_agree(layout, b, n, dtype, dev, monkeypatch):
    print(f"[test] paths {layout} b={b} n={n}", flush=True)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    # even keys: every odd query is a miss
    A = torch.arange(n, dtype=dtype, device=dev).mul_(2)
    Q = torch.randint(0, 2 * n, (1 << 22,), generator=g, device=dev).to(dtype)
    if layout != "sorted":
        tl_amd.permute(layout, A, b)
    tables = None
    if layout in ("mveb", "veb"):
        t, idx, tidx, meta = tl_amd.veb_tableset_device(n, device=dev, classic=layout == "veb")
        tables = (t, idx, tidx, *meta.tolist()[:2])
    got = {}
    for path in ("plain", "tile", "part"):
        monkeypatch.setenv("TL_QUERY_PATH", path)
        got[path] = torch.full((Q.numel(),), -1, dtype=L, device=dev)
        lookup(layout, b, A, Q, got[path], tables)
    plain = got["plain"]
    assert torch.equal(plain, got["tile"]) and torch.equal(plain, got["part"])
    hit = Q % 2 == 0
    if layout == "sorted":
        assert torch.equal(plain, Q.to(L) // 2)
    else:
        assert bool((plain[~hit] == n).all())
        assert torch.equal(A[plain[hit]], Q[hit])


@pytest.mark.parametrize("name", ["TL_BTREE_WIDE", "TL_BTREE_QPG"])
def test_descent_variables_keep_the_descents(name, dev, monkeypatch):
    n = 5_000_011
    A = torch.arange(n, dtype=L, device=dev)
    tl_amd.permute_btree(A, 16)
    Q = torch.randint(0, n, (1 << 24,), device=dev)
    ans = torch.empty_like(Q)
    tl_amd.query_btree(A, 16, Q, ans)   # partitioned, kernels loaded
    monkeypatch.setenv(name, "2" if name == "TL_BTREE_QPG" else "0")
    tl_amd.query_btree(A, 16, Q, ans)
    tl_amd.release_scratch()
    free = torch.cuda.mem_get_info(dev)[0]
    tl_amd.query_btree(A, 16, Q, ans)
    assert torch.cuda.mem_get_info(dev)[0] == free
    assert bool((A[ans] == Q).all())
