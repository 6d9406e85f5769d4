"""Device memory that a batch holds for partitioned lookups: one workspace for the
one array that is worth partitioning, none where the query queues answer it."""
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("query_queue,limit", [(0, 20), (1, 1)])
def test_workspace_of_one_large_array(query_queue, limit, dev):
    n, nq = 5_000_011, 1 << 24
    A = torch.arange(n, dtype=torch.int64, device=dev)
    Q = torch.randint(0, n, (nq,), device=dev)
    arrays = [{"A": A, "kind": "u64", "b": 8, "layout": "btree", "Q": Q,
               "ans": torch.empty(nq, dtype=torch.int64, device=dev)}]
    for i in range(7):
        small = torch.arange(1000 + i, dtype=torch.int64, device=dev)
        arrays.append({"A": small, "kind": "u64", "b": 8, "layout": "btree", "Q": small[:100].clone(),
                       "ans": torch.empty(100, dtype=torch.int64, device=dev)})
    bare = [dict(a, Q=None) for a in arrays]
    torch.cuda.synchronize()
    held = []
    for items in (bare, arrays):   # without lookups: the permutations' share
        free = torch.cuda.mem_get_info(dev)[0]
        batch = tl_amd.Batch(items, query_queue=query_queue)
        held.append(free - torch.cuda.mem_get_info(dev)[0])
        if items is arrays:
            batch.run(graph=True)
            assert bool((A[arrays[0]["ans"]] == Q).all())
        del batch
    # 18 bytes a query and tables, once; allocations are whole pages of 2 MiB
    assert held[1] - held[0] <= limit * nq + (16 << 20), held
