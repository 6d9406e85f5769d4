"""A perfect vEB layout queried with its own tables through the other split's
entry point, on every path: the tables decide."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
import tl_amd
from test_gpu_query import make_keys, make_queries, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["plain", "tile", "part"])
@pytest.mark.parametrize("layout", ["mveb", "veb"])
@pytest.mark.parametrize("levels", [15, 23])
def test_tables_decide(path, layout, levels, dev, monkeypatch):
    monkeypatch.setenv("TL_QUERY_PATH", path)
    rng = np.random.default_rng(levels)
    n = (1 << levels) - 1
    keys = make_keys("u64", n, rng)
    A = ol.permute(layout, keys.copy(), 0)
    Q = make_queries("u64", keys, 100_001, rng)
    tables, idx, tidx, _ = tl_amd.veb_tableset_device(n, device=dev, classic=layout == "veb")
    exp = ol.search(layout, A, Q, "u64", 1)
    Ad, Qd = to_dev(A, "u64", dev), to_dev(Q, "u64", dev)
    ans = torch.zeros(Q.size, dtype=torch.int64, device=dev)
    for query in (tl_amd.query_mveb, tl_amd.query_veb):
        ans.zero_()
        query(Ad, tables, levels, Qd, ans, kind="u64")
        assert np.array_equal(ans.cpu().numpy().view(np.uint64), exp), query.__name__
