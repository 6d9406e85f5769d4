"""The HBM traffic that bench.py reports for a permute is that of the path the
call takes: the one-pass slide by default, the plan where TL_PERMUTE_PLAN asks
for it.  Each has a committed rocprofv3 summary of its own."""
import bench

KEYS = 17.18e9   # read and written once: 2 * 2^30 * 8 bytes


def test_traffic_of_the_default_permutes(monkeypatch):
    monkeypatch.delenv("TL_PERMUTE_PLAN", raising=False)
    # every key moves once, and a second time through the stash: 0.38 n keys of
    # the B-tree, n / 2 of the BST
    assert 1.3 * KEYS < bench.permute_traffic("btree", 1 << 30, 16) < 1.45 * KEYS
    assert 1.45 * KEYS < bench.permute_traffic("bst", 1 << 30) < 1.6 * KEYS
    assert 0.95 * KEYS < bench.permute_traffic("mveb", 1 << 30) < 1.2 * KEYS
    assert bench.permute_traffic("btree", 1 << 30, 8) is None
    assert bench.permute_traffic("bst", 1 << 20) is None


def test_traffic_of_the_plans(monkeypatch):
    monkeypatch.setenv("TL_PERMUTE_PLAN", "1")
    assert 2.0 * KEYS < bench.permute_traffic("btree", 1 << 30, 16) < 2.5 * KEYS
    assert 1.8 * KEYS < bench.permute_traffic("bst", 1 << 30) < 2.4 * KEYS
