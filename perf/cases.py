"""The work a program has this library do, as cases that can be timed.

A case names one call (or, for a batch, one replay) through the Python surface
of the library, with its sizes, key type, layout and data:

  build    a sorted array laid out in place                 (permute)
  unbuild  a layout put back into sorted order, in place    (unpermute)
  query    a batch of lookups over a built layout, or by binary search of the
           sorted keys
  learned  B-tree lookups from a fitted start-node model
  sort     raw keys, with repeats, to sorted distinct keys
  batch    many independent arrays laid out and queried by one graph replay

Every output is whole numbers (keys, slots, counts), so `exact` has nothing to
say: two programs agree bit for bit or one of them is wrong.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "tree-layouts_amd", "python"))
import tl_amd as tl  # noqa: E402

KINDS = ("u32", "u64", "i32", "i64")
LAYOUTS = ("bst", "btree", "mveb", "veb")
NODE_WIDTHS = (2, 3, 4, 7, 8, 12, 15, 16, 17, 31, 32, 33, 64)
CHUNK = 1 << 26   # keys generated at a time


def listed():
    return [
        # one request of a service that keeps a small index: launch and call overhead
        _query("lookup_bst_u32_1k", "bst", "u32", 1000, 64, hits=0.5),
        # an index of a few pages rebuilt on each update: the smallest build past one workgroup
        _build("build_btree_u64_100k", "btree", "u64", 100_003, b=16),
        # the perfect million-key BST with as many lookups, half of them misses
        _query("query_bst_u32_1m", "bst", "u32", (1 << 20) - 1, 1 << 20, hits=0.5),
        # a ragged BST of 4-byte keys, several times the caches' size
        _build("build_bst_u32_500m", "bst", "u32", 500_000_003),
        # the headline build
        _build("build_btree_u64_1g", "btree", "u64", 1 << 30, b=16, keys="lognormal"),
        # a layout taken back to sorted order to merge new keys: signed keys, narrower nodes
        _build("unbuild_btree_i32_200m", "btree", "i32", 200_000_001, b=8, op="unbuild"),
        # the non-perfect mvEB build
        _build("build_mveb_u64_300m", "mveb", "u64", 300_000_000, keys="geometric"),
        # the headline lookups: plain root descent
        _query("query_btree_u64_1g", "btree", "u64", 1 << 30, 1 << 27, b=16, keys="lognormal"),
        # the same lookups from the learned start node
        _query("learned_btree_u64_1g", "btree", "u64", 1 << 30, 1 << 27, b=16, keys="lognormal",
               op="learned", leaves=1 << 16),
        # skewed lookups over the non-perfect mvEB
        _query("query_mveb_u64_300m", "mveb", "u64", 300_000_000, 1 << 26, keys="geometric",
               zipf=True),
        # raw 40-bit identifiers in any order, one in ten repeated, made ready for a layout
        {"name": "sort_u64_100m", "op": "sort", "kind": "u64", "n": 100_000_000, "bits": 40},
        # many tenants' indexes of very different sizes, built and queried together
        {"name": "batch_512", "op": "batch", "count": 512, "lo": 8, "hi": 22, "b": 8},
    ]


def draw(rng):
    op = rng.choices(("query", "build", "unbuild", "learned", "sort", "batch"),
                     (6, 4, 2, 1, 2, 1))[0]
    if op == "batch":
        return {"op": op, "count": _size(rng, 8, 512), "lo": rng.randint(6, 9),
                "hi": rng.randint(14, 22), "b": rng.choice(NODE_WIDTHS)}
    kind = rng.choice(KINDS)
    if op == "sort":
        n = _size(rng, 1 << 10, 150_000_000)
        bits = rng.randint(max(20, n.bit_length() + 1), min(62, 8 * tl.WIDTH[kind]))
        return {"op": op, "kind": kind, "n": n, "bits": bits}
    keys = rng.choice(("uniform", "geometric", "lognormal")) if tl.WIDTH[kind] == 8 else "uniform"
    if op in ("build", "unbuild"):
        n = _size(rng, 1 << 8, 1 << (29 if tl.WIDTH[kind] == 4 else 30))
        c = _build(None, rng.choice(LAYOUTS), kind, n, rng.choice(NODE_WIDTHS), keys, op)
    else:
        n = _size(rng, 1 << 8, 1 << 28)
        nq = _size(rng, 1 << 6, 1 << 26)
        hits = rng.choice((0.5, 0.9, 1.0))
        layout = "btree" if op == "learned" else rng.choice(LAYOUTS + ("btree", "sorted"))
        leaves = rng.choice((1 << 10, 1 << 16)) if op == "learned" else 0
        c = _query(None, layout, kind, n, nq, rng.choice(NODE_WIDTHS), keys, hits,
                   rng.random() < 0.25, op, leaves)
    del c["name"]
    return c


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    op = case["op"]
    if op == "batch":
        return _prepare_batch(case, g)
    kind, n = case["kind"], case["n"]
    if op == "sort":
        # nine keys in ten are distinct, the tenth repeats one of them
        fresh = n - n // 10
        top = max(1, int(1.9 * 2 ** case["bits"] / fresh) - 1)
        keys = _sorted_keys({"n": fresh, "kind": kind, "keys": "uniform", "top": top}, g)
        raw = torch.cat([keys, keys[torch.randint(0, fresh, (n - fresh,), generator=g,
                                                  device="cuda")]])
        raw = raw[torch.randperm(n, generator=g, device="cuda")]
        return {"op": op, "kind": kind, "raw": raw, "A": torch.empty_like(raw)}
    A = _sorted_keys(case, g)
    s = {"op": op, "kind": kind, "layout": case["layout"], "b": case["b"], "A": A}
    if op == "build":
        return s
    if op == "unbuild":
        tl.permute(s["layout"], A, s["b"], kind)
        return s
    s["Q"] = _queries(case, A, g)
    s["ans"] = torch.empty(case["nq"], dtype=torch.int64, device="cuda")
    if op == "learned":
        s["model"], _ = tl.learned_fit(A, case["leaves"], kind)
    if s["layout"] in ("mveb", "veb"):
        tables, idx, tidx, meta = tl.veb_tableset_device(n, classic=s["layout"] == "veb")
        d, num, _ = meta.tolist()[:3]
        s["tables"] = (tables, idx, tidx, d, num)
    if s["layout"] != "sorted":
        tl.permute(s["layout"], A, s["b"], kind)
    return s


def run(state):
    op = state["op"]
    if op == "batch":
        # the arrays arrive sorted, in buffers of their own
        for work, keys in state["buffers"]:
            work.copy_(keys)
        state["batch"].run(graph=True, timed=False)
        return [work for work, _ in state["buffers"]] + [state["ans"]]
    A, kind = state["A"], state["kind"]
    if op == "sort":
        # the raw keys stay the program's own: the sort works on a copy
        A.copy_(state["raw"])
        m, _ = tl.sort_dedupe(A, kind)
        return m, A[:m]
    layout, b = state["layout"], state["b"]
    if op == "build":
        tl.permute(layout, A, b, kind, timed=False)
        return A
    if op == "unbuild":
        tl.unpermute(layout, A, b, kind, timed=False)
        return A
    Q, ans = state["Q"], state["ans"]
    if op == "learned":
        tl.query_btree_learned(A, b, state["model"], Q, ans, None, kind, timed=False)
    elif layout == "bst":
        tl.query_bst(A, Q, ans, kind, timed=False)
    elif layout == "btree":
        tl.query_btree(A, b, Q, ans, kind, timed=False)
    elif layout == "sorted":
        tl.query_binary(A, Q, ans, kind, timed=False)
    else:
        query = tl.query_mveb_nonperfect if layout == "mveb" else tl.query_veb_nonperfect
        query(A, *state["tables"], Q, ans, kind, timed=False)
    return ans


def work(case):
    op = case["op"]
    if op == "batch":
        keys = query = 0
        for n, kind in _batch_shapes(case):
            w = tl.WIDTH[kind]
            keys += 2 * n * w
            query += 4 * n * (w + 8)
        return {"bytes": keys + query, "flops": 0}
    n, w = case["n"], tl.WIDTH[case["kind"]]
    if op in ("build", "unbuild", "sort"):
        return {"bytes": 2 * n * w, "flops": 0}
    # every lookup reads at least one line of the array, no line is needed twice
    nq = case["nq"]
    return {"bytes": nq * (w + 8) + min(n * w, nq * 64), "flops": 0}


def exact(case, seed):
    return None


# ---- cases ------------------------------------------------------------------

def _build(name, layout, kind, n, b=16, keys="uniform", op="build"):
    return {"name": name, "op": op, "layout": layout, "kind": kind, "n": n, "b": b, "keys": keys}


def _query(name, layout, kind, n, nq, b=16, keys="uniform", hits=1.0, zipf=False, op="query",
           leaves=0):
    return {"name": name, "op": op, "layout": layout, "kind": kind, "n": n, "nq": nq, "b": b,
            "keys": keys, "hits": hits, "zipf": zipf, "leaves": leaves}


def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# ---- data -------------------------------------------------------------------

def _store(kind):
    """Keys are stored in signed tensors; the key type's name says how they compare."""
    return torch.int32 if tl.WIDTH[kind] == 4 else torch.int64


def _first(kind):
    return -(1 << 31) + 1 if kind == "i32" else 1


def _gaps(case, m, g):
    if case["keys"] == "lognormal":
        x = torch.empty(m, dtype=torch.float32, device="cuda").normal_(0.0, 2.0, generator=g)
        return x.exp_().ceil_().to(torch.int64).clamp_(min=1)
    if case["keys"] == "geometric":   # p = 0.1
        u = torch.rand(m, generator=g, device="cuda").clamp_(min=1e-7)
        return u.log_().div_(math.log(0.9)).ceil_().to(torch.int64).clamp_(min=1)
    top = case.get("top", 64)
    if "top" not in case and tl.WIDTH[case["kind"]] == 4:   # the keys stay below 2^32 of them
        top = max(1, min(64, int(1.9 * 2 ** 32 / case["n"]) - 1))
    return torch.randint(1, top + 1, (m,), generator=g, device="cuda")


def _sorted_keys(case, g):
    """n ascending distinct keys: a running sum of random gaps."""
    n, kind = case["n"], case["kind"]
    A = torch.empty(n, dtype=_store(kind), device="cuda")
    last = torch.full((), _first(kind), dtype=torch.int64, device="cuda")
    for at in range(0, n, CHUNK):
        m = min(CHUNK, n - at)
        v = _gaps(case, m, g).cumsum(0).add_(last)
        last = v[-1].clone()
        A[at:at + m] = v
    return A


def _queries(case, A, g):
    """nq lookups: hits of uniform or Zipf(1.1) rank, the rest uniform between
    the smallest and the largest key."""
    n, nq, kind = case["n"], case["nq"], case["kind"]
    Q = torch.empty(nq, dtype=A.dtype, device="cuda")
    lo, hi = (int(v) for v in A[[0, n - 1]].tolist())
    if kind == "u32":
        lo, hi = lo & 0xFFFFFFFF, hi & 0xFFFFFFFF
    for at in range(0, nq, CHUNK):
        m = min(CHUNK, nq - at)
        if case["zipf"]:   # inverse of the continuous distribution, ranks spread over the keys
            u = torch.rand(m, generator=g, dtype=torch.float64, device="cuda")
            r = u.mul_((n + 1.0) ** -0.1 - 1.0).add_(1.0).pow_(-10.0).to(torch.int64)
            at_key = (r * 2654435761) % n
        else:
            at_key = torch.randint(0, n, (m,), generator=g, device="cuda")
        q = A[at_key]
        if case["hits"] < 1.0:
            miss = torch.rand(m, generator=g, device="cuda") >= case["hits"]
            other = torch.randint(lo, hi + 1, (m,), generator=g, device="cuda")
            q = torch.where(miss, other.to(A.dtype), q)
        Q[at:at + m] = q
    return Q


def _batch_shapes(case):
    """(keys, key type) of every array: sizes spread over the logarithm of
    [2^lo, 2^hi], key types in turn."""
    gen = torch.Generator()
    gen.manual_seed(5)
    u = torch.rand(case["count"], generator=gen, dtype=torch.float64)
    sizes = (2.0 ** (case["lo"] + u * (case["hi"] - case["lo"]))).long().tolist()
    return [(n, "i32" if i % 2 else "u64") for i, n in enumerate(sizes)]


def _prepare_batch(case, g):
    shapes = _batch_shapes(case)
    # arrays start on 256-byte boundaries of one buffer per key width
    starts, total = [], {4: 0, 8: 0}
    for n, kind in shapes:
        w = tl.WIDTH[kind]
        starts.append(total[w])
        total[w] += (n + 63) // 64 * 64
    keys = {}
    for w, kind in ((4, "i32"), (8, "u64")):
        keys[w] = _sorted_keys({"n": max(1, total[w]), "kind": kind, "keys": "uniform"}, g)
    work_of = {w: k.clone() for w, k in keys.items()}
    ans = torch.empty(4 * sum(n for n, _ in shapes), dtype=torch.int64, device="cuda")
    arrays, at = [], 0
    for i, ((n, kind), a) in enumerate(zip(shapes, starts)):
        w = tl.WIDTH[kind]
        pick = torch.randint(0, n, (4 * n,), generator=g, device="cuda")
        arrays.append({"A": work_of[w][a:a + n], "kind": kind, "b": case["b"],
                       "layout": LAYOUTS[(i // 2) % 3], "Q": keys[w][a:a + n][pick],
                       "ans": ans[at:at + 4 * n]})
        at += 4 * n
    return {"op": "batch", "batch": tl.Batch(arrays), "ans": ans,
            "buffers": [(work_of[w], keys[w]) for w in (4, 8)]}
