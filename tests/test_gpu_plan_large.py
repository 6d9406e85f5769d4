"""The plans at size (TL_PERMUTE_PLAN), which serve short memory, stashes past 5 GiB
and arrays of 2^32 keys, against the one-pass slides' layouts slot for slot and
sampled slots of the oracle; and back by the inverse plans."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
import tl_amd

pytestmark = pytest.mark.gpu

I, L = torch.int32, torch.int64


@pytest.mark.parametrize("layout,b,n,dtype", [
    ("bst", 1, 1 << 30, L), ("bst", 1, (1 << 27) - 1, L), ("bst", 1, 500_000_003, I),
    ("btree", 16, 1 << 30, L), ("btree", 8, 200_000_001, I), ("btree", 2, 100_000_007, L),
    ("btree", 1, 60_000_011, I), ("btree", 100, 300_000_001, L)])
def test_plan(layout, b, n, dtype, dev, monkeypatch):
    ref = torch.arange(n, dtype=dtype, device=dev)
    tl_amd.permute(layout, ref, b)
    monkeypatch.setenv("TL_PERMUTE_PLAN", "1")
    A = torch.arange(n, dtype=dtype, device=dev)
    print(f"[test] plan {layout} b={b} n={n}", flush=True)
    tl_amd.permute(layout, A, b)
    assert torch.equal(A, ref)
    ranks = np.random.default_rng(n).integers(0, n, 20_000)
    o = ol.oracle()
    pos = np.array([o.or_btree_pos(int(x), n, b) for x in ranks], dtype=np.int64)
    assert np.array_equal(A[torch.from_numpy(pos).to(dev)].cpu().numpy(), ranks)
    tl_amd.unpermute(layout, A, b)
    assert torch.equal(A, torch.arange(n, dtype=dtype, device=dev))
    del A, ref
    torch.cuda.empty_cache()
