"""The bytes that bench.py holds a partitioned batch against are bytes that move: no
more than the traffic measured for it (descents of single queries read more)."""
import bench


def test_lookup_bytes_are_moved():
    n, nq = 1 << 30, 1 << 27
    t = bench.measured_traffic_entry("btree_b16_n2p30_u64_query_traffic.txt")
    moved = (t["plain_read_GB"] + t["plain_write_GB"]) * 1e9
    need = bench.lookup_bytes(n, nq, 8)
    assert need == nq * 16 + n * 8
    assert need < moved < nq * bench.btree_query_bytes(n, 16, 8)[1]
    assert bench.lookup_bytes(n, 1000, 4) == 1000 * (12 + 64)
