"""The splitter sort's buckets far past their average: inputs whose sampled places
(one of each equal share of the input, see sample_at) miss a crowd of keys, so
that one bucket of the first pass, or 8 of the second, hold them all: a bucket
more than fits the usual workgroup, as many as fit the largest, and more (which
ends in the radix sort)."""
import numpy as np
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu


def sampled(n, samples):
    i = np.arange(samples, dtype=np.uint64)
    lo = i * np.uint64(n) // np.uint64(samples)
    hi = (i + np.uint64(1)) * np.uint64(n) // np.uint64(samples)
    return (lo + (i * np.uint64(2654435761) % np.uint64(1 << 32)) % (hi - lo)).astype(np.int64)


# (keys, samples of the first pass, keys of the crowd)
@pytest.mark.parametrize("n,samples,crowd", [
    (200_000, 8192, 4_000), (200_000, 8192, 15_000), (200_000, 8192, 16_384),
    (200_000, 8192, 20_000), (3_200_000, 8192, 60_000), (3_200_000, 8192, 300_000)])
@pytest.mark.parametrize("kind", ["u64", "i64"])
def test_crowd_between_samples(kind, n, samples, crowd, dev):
    rng = np.random.default_rng(crowd)
    keys = rng.integers(1 << 40, 1 << 60, n)
    keys = np.where(rng.random(n) < 0.5, keys, -keys) if kind == "i64" else keys
    free = np.setdiff1d(np.arange(n), sampled(n, samples))
    # a dense run of keys, some of them twice, just past one that is sampled
    first = np.sort(keys[sampled(n, samples)])[samples // 3] + 1
    keys[rng.choice(free, crowd, replace=False)] = first + rng.integers(0, 8 * crowd, crowd)
    raw = torch.from_numpy(keys).to(dev)
    expect = torch.unique(raw)
    m, _ = tl_amd.sort_dedupe(raw, kind)
    assert m == expect.numel()
    assert torch.equal(raw[:m], expect)
