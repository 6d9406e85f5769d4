"""The splitter sort against torch.unique around its paths' edges (one bucket,
one pass, two passes), over inputs that crowd, repeat and are in order already;
and the radix sort it can fall back to."""
import numpy as np
import pytest
import torch

import tl_amd

pytestmark = pytest.mark.gpu

STORE = {"u32": torch.int32, "u64": torch.int64, "i32": torch.int32, "i64": torch.int64}


def inputs(kind, n, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    top = 1 << (31 if "32" in kind else 62)
    low = -top if kind[0] == "i" else 0
    rnd = lambda a, b: torch.randint(a, b, (n,), generator=g, device=dev)   # noqa: E731
    yield "wide", rnd(low, top)
    yield "narrow", rnd(0, max(2, n // 2))
    yield "heavy", torch.where(rnd(0, 10) > 0, torch.full((n,), 5, device=dev), rnd(0, top))
    yield "equal", torch.full((n,), top - 1, device=dev)
    yield "reverse", torch.arange(n, 0, -1, device=dev)
    yield "crowds", rnd(0, 8) * (top // 8) + rnd(0, 3000)


@pytest.mark.parametrize("kind", ["u32", "u64", "i32", "i64"])
@pytest.mark.parametrize("n", [2, 4096, 4097, 70001, 1572863, 1572865, 5000011])
def test_split_sort(kind, n, dev, monkeypatch):
    for name, raw in inputs(kind, n, dev):
        A = raw.to(STORE[kind])
        expect = torch.unique(raw)   # non-negative, or a signed kind
        for radix in ("0", "1") if n < 100000 else ("0",):
            monkeypatch.setenv("TL_SORT_RADIX", radix)
            B = A.clone()
            m, _ = tl_amd.sort_dedupe(B, kind)
            assert m == expect.numel(), (name, radix)
            assert torch.equal(B[:m].to(torch.int64), expect), (name, radix)
