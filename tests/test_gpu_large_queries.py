"""The paths of large query batches (tile-sorted descents, partitioned lookups)
against the oracle, forced by TL_QUERY_PATH at the sizes where they can go
wrong: arrays at the smallest size and around a power of two (range and heap
edges), batches around a tile's edges, an array large enough for two passes,
keys that repeat, skewed batches, a batch that overlaps its answers, several
streams, and a captured call."""
import numpy as np
import pytest
import torch

import oracle_lib as ol
import tl_amd
from test_gpu_query import gpu_answers, make_keys, make_queries, to_dev

pytestmark = pytest.mark.gpu

CASES = [("bst", 1), ("btree", 16), ("btree", 7), ("btree", 1), ("btree", 200), ("mveb", 0),
         ("veb", 0)]


def expected(layout, A, Q, kind, b):
    return ol.search("binary" if layout == "sorted" else layout, A, Q, kind, max(b, 1))


def answers(layout, b, kind, A, Q, dev):
    if layout != "sorted":
        return gpu_answers(layout, b, kind, A, Q, dev)
    ans = torch.zeros(Q.size, dtype=torch.int64, device=dev)
    tl_amd.query_binary(to_dev(A, kind, dev), to_dev(Q, kind, dev), ans, kind=kind)
    return ans.cpu().numpy().view(np.uint64)


@pytest.mark.parametrize("path", ["tile", "part"])
@pytest.mark.parametrize("layout,b", CASES + [("sorted", 0)])
@pytest.mark.parametrize("kind", ["u32", "i64"])
def test_large_batch_matches_oracle(path, layout, b, kind, dev, monkeypatch):
    monkeypatch.setenv("TL_QUERY_PATH", path)
    rng = np.random.default_rng(7 + b)
    for n, nq in [(4096, 65536), (4097, 69633), (65535, 66001), (65537, 131071),
                  (1000003, 200001)]:
        keys = make_keys(kind, n, rng)
        A = keys if layout == "sorted" else ol.permute(layout, keys.copy(), b)
        Q = make_queries(kind, keys, nq, rng)
        if layout == "sorted":   # below the smallest key the reference's loop does not end
            exp = expected(layout, A, np.maximum(Q, keys[0]), kind, b)
            exp[Q < keys[0]] = n
        else:
            exp = expected(layout, A, Q, kind, b)
        assert np.array_equal(answers(layout, b, kind, A, Q, dev), exp), (n, nq)


@pytest.mark.parametrize("layout,b", CASES)
@pytest.mark.parametrize("kind", ["u64", "i32"])
def test_two_pass_partition_and_skew(layout, b, kind, dev, monkeypatch):
    """Past 2^22 keys the ranges take two passes; half of the batch is one key
    and its neighbours."""
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    rng = np.random.default_rng(11)
    n = 5_000_011
    keys = make_keys(kind, n, rng)
    A = ol.permute(layout, keys.copy(), b)
    Q = make_queries(kind, keys, 300_000, rng)
    Q[::2] = keys[n // 3 + rng.integers(0, 3, Q[::2].size)]
    got = answers(layout, b, kind, A, Q, dev)
    assert np.array_equal(got, expected(layout, A, Q, kind, b))


@pytest.mark.parametrize("n", [300_007, 5_000_011])
@pytest.mark.parametrize("layout,b", [("bst", 1), ("btree", 16), ("mveb", 0), ("sorted", 0)])
def test_crowded_range(n, layout, b, dev, monkeypatch):
    """One and two passes with nearly all queries in one range: more than its
    workgroup's share, and (two passes) more tiles of one bucket than a share has."""
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    rng = np.random.default_rng(13)
    keys = make_keys("u64", n, rng)
    A = keys if layout == "sorted" else ol.permute(layout, keys.copy(), b)
    Q = keys[n // 5 + rng.integers(0, 300, 400_001)]
    Q[::400] = keys[rng.integers(0, n, Q[::400].size)]
    assert np.array_equal(answers(layout, b, "u64", A, Q, dev), expected(layout, A, Q, "u64", b))


@pytest.mark.parametrize("path", ["tile", "part"])
@pytest.mark.parametrize("layout,b", [("bst", 1), ("btree", 16), ("btree", 8), ("mveb", 0)])
def test_repeated_keys(path, layout, b, dev, monkeypatch):
    """Runs of equal keys, also across range borders: the first on the descent."""
    monkeypatch.setenv("TL_QUERY_PATH", path)
    rng = np.random.default_rng(3)
    n = 300_007
    keys = np.sort(rng.integers(0, n // 3, n)).astype(np.uint64)
    keys[4000:9000] = keys[4000]
    keys.sort()
    A = ol.permute(layout, keys.copy(), b)
    Q = np.concatenate([keys[rng.integers(0, n, 60_000)], keys[3990:9010],
                        rng.integers(0, n, 10_000).astype(np.uint64)])
    got = answers(layout, b, "u64", A, Q, dev)
    assert np.array_equal(got, expected(layout, A, Q, "u64", b))


def test_batch_over_its_answers(dev, monkeypatch):
    """Queries in the answer buffer itself: the partition would overwrite them."""
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    rng = np.random.default_rng(5)
    keys = make_keys("u64", 200_003, rng)
    A = ol.permute("bst", keys.copy())
    Q = make_queries("u64", keys, 100_000, rng)
    buf = to_dev(Q, "u64", dev)
    tl_amd.query_bst(to_dev(A, "u64", dev), buf, buf, kind="u64")
    assert np.array_equal(buf.cpu().numpy().view(np.uint64), ol.search("bst", A, Q, "u64"))


def test_streams_and_capture(dev, monkeypatch):
    """Calls in flight on three streams (more than there are workspaces), then
    a captured call replayed with other queries in the same buffer."""
    monkeypatch.setenv("TL_QUERY_PATH", "part")
    rng = np.random.default_rng(9)
    keys = make_keys("u64", 500_009, rng)
    A_np = ol.permute("btree", keys.copy(), 16)
    A = to_dev(A_np, "u64", dev)
    Qs = [make_queries("u64", keys, 400_000, rng) for _ in range(3)]
    exp = [ol.search("btree", A_np, q, "u64", 16) for q in Qs]
    Qd = [to_dev(q, "u64", dev) for q in Qs]
    outs = [torch.zeros(q.size, dtype=torch.int64, device=dev) for q in Qs]
    streams = [torch.cuda.Stream() for _ in Qs]
    torch.cuda.synchronize()
    for _ in range(3):
        for q, o, s in zip(Qd, outs, streams):
            tl_amd.query_btree(A, 16, q, o, kind="u64", stream=s.cuda_stream, timed=False)
    torch.cuda.synchronize()
    for o, e in zip(outs, exp):
        assert np.array_equal(o.cpu().numpy().view(np.uint64), e)
    g = torch.cuda.CUDAGraph()
    Q, ans = Qd[0].clone(), torch.zeros_like(outs[0])
    with torch.cuda.graph(g):
        tl_amd.query_btree(A, 16, Q, ans, kind="u64", timed=False)
    for k in (1, 2, 0):
        Q.copy_(Qd[k])
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(ans.cpu().numpy().view(np.uint64), exp[k])
