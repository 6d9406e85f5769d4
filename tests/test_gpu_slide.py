"""One-pass permutations of BSTs and B-trees past 128 MiB against the oracle's
layouts: perfect trees, one leaf, few leaves, many, nodes of one key to 4096;
arrays that start off a 16-byte line."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
import tl_amd

pytestmark = pytest.mark.gpu

I, L = torch.int32, torch.int64
CASES = [("bst", 1, (1 << 25) - 1, L), ("bst", 1, 1 << 25, L), ("bst", 1, (1 << 25) + 2, I),
         ("bst", 1, 20_000_003, L), ("btree", 1, 17_000_001, L), ("btree", 2, 3 ** 16 + 12345, I),
         ("btree", 16, 17 ** 6 + 100_000, L), ("btree", 16, 34_000_001, I),
         ("btree", 4096, 17_000_000, L)]


@pytest.mark.parametrize("layout,b,n,dtype", CASES)
def test_slide(layout, b, n, dtype, dev):
    ranks = torch.from_numpy(ol.layout_ranks(layout, n, b).astype(np.int64)).to(dev).to(dtype)
    buf = torch.full((n + 4,), -7, dtype=dtype, device=dev)
    for at in (0, 1):
        A = buf[at:at + n]
        A.copy_(torch.arange(n, dtype=dtype, device=dev))
        tl_amd.permute(layout, A, b)
        assert torch.equal(A, ranks), (layout, b, n, at)
        assert bool((buf[at + n:] == -7).all())
        tl_amd.unpermute(layout, A, b)
        assert torch.equal(A, torch.arange(n, dtype=dtype, device=dev)), (layout, b, n, at)
        buf.fill_(-7)
