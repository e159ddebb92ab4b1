"""The closure work this framework is used for, as timed cases.

Each case is one call (or one short sequence of calls) a program makes on data
it already holds on the GPU: the dense closure of a pedigree in each numbering
(parents first, parents last, arbitrary), the AVOS product of closures, edge
insertion into a closed graph, the sparse DAG closure with and without a plan,
the squaring closure, a batch of components, and the canonical ordering of a
closed graph.  Graphs are the layered synthetic pedigrees of
redblackgraph_amd.synth; every output is a whole number, so results are exact.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from redblackgraph_amd import dense, synth
from redblackgraph_amd import sparse_dev as sd
from redblackgraph_amd._dtypes import elem_type
from redblackgraph_amd.batched import BatchedClosure
from redblackgraph_amd.gpu import CSRMatrixGPU, transitive_closure_dag_gpu, transitive_closure_gpu
from redblackgraph_amd.sparse.csgraph._ordering import canonical_order_device


def _closure(name, n, dtype, numbering, layers, p, lookback):
    c = {"kind": "closure", "n": n, "dtype": dtype, "numbering": numbering, "layers": layers, "p": p,
         "lookback": lookback}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the small dense closure of the parity workload: one family's pedigree, bound by latency and launches
        _closure("closure_512_i32_lower", 512, "int32", "lower", 10, 0.8, 3),
        # a mid-sized pedigree numbered parents last, the layout the reference's upper triangular option takes
        _closure("closure_1100_i32_upper", 1100, "int32", "upper", 11, 0.8, 4),
        # a pedigree as it comes from a file, in no particular numbering: entries on both sides of the diagonal
        _closure("closure_2304_i32_any", 2304, "int32", "any", 12, 0.8, 4),
        # the wide element type, for pedigrees deeper than 31 bits of ancestry
        _closure("closure_4096_i64_lower", 4096, "int64", "lower", 24, 0.75, 4),
        # the large dense closure, this repository's headline workload
        _closure("closure_8192_i32_lower", 8192, "int32", "lower", 24, 0.75, 4),
        # R @ R of a large closure, the dense AVOS product
        {"name": "product_8192_i32", "kind": "product", "m": 8192, "k": 8192, "n": 8192, "dtype": "int32",
         "layers": 24, "p": 0.75, "lookback": 4},
        # new parent edges into a graph a server holds closed (the largest request of its stream)
        {"name": "insert_4095_i32", "kind": "insert", "n": 4095, "edges": 64, "dtype": "int32"},
        # a county-sized sparse pedigree closed once, without a plan (the largest size of the reference's table)
        {"name": "dag_21162_i64", "kind": "dag", "n": 21162, "dtype": "int64", "layers": 12, "p": 0.7,
         "lookback": 1, "plan": False},
        # the 1M-vertex sparse closure, repeated with the plan such a program keeps
        {"name": "dag_1000005_i64", "kind": "dag", "n": 1_000_005, "dtype": "int64", "layers": 15, "p": 0.7,
         "lookback": 1, "plan": True},
        # repeated squaring, the closure that needs no vertex order
        {"name": "squaring_11012_i32", "kind": "squaring", "n": 11012, "dtype": "int32", "layers": 10, "p": 0.7,
         "lookback": 2},
        # many families at once: sizes log-uniform from a household to a county, one graph replay per batch
        {"name": "batch_128_i32", "kind": "batch", "count": 128, "lo": 16, "hi": 4096},
        # the canonical vertex order of a closed sparse graph, and the graph renumbered by it
        {"name": "order_300007_i64", "kind": "order", "n": 300_007, "dtype": "int64", "layers": 13, "p": 0.7,
         "lookback": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closure"] * 4 + ["product", "insert", "dag", "squaring", "batch", "order"])
    if kind == "closure":
        dtype = rng.choice(["int32", "int32", "int64"])
        numbering = rng.choice(["lower", "lower", "upper", "any"])
        top = {"lower": 8192, "upper": 6000, "any": 4000}[numbering]
        n = _log(rng, 100, top if dtype == "int32" else top // 2)
        return _closure(None, n, dtype, numbering, max(3, min(24, math.ceil(math.log2(n)) + rng.randint(-2, 8))),
                        rng.choice([0.7, 0.75, 0.8]), rng.randint(1, 4))
    if kind == "product":
        n = _log(rng, 200, 6000)
        dtype = rng.choice(["int32", "int64"])
        if dtype == "int64":
            n = min(n, 3000)
        m, q = (max(1, int(n * rng.uniform(0.3, 1.0))) for _ in range(2))
        return {"kind": "product", "m": m, "k": n, "n": q, "dtype": dtype, "layers": max(3, math.ceil(math.log2(n))),
                "p": 0.75, "lookback": rng.randint(1, 4)}
    if kind == "insert":
        return {"kind": "insert", "n": _log(rng, 32, 4095), "edges": rng.randint(1, 64), "dtype": "int32"}
    if kind == "dag":
        plan = rng.random() < 0.5
        n = _log(rng, 442, 700_000 if plan else 200_000)
        return {"kind": "dag", "n": n, "dtype": rng.choice(["int32", "int64"]),
                "layers": max(4, min(15, math.ceil(math.log2(n)) + rng.randint(-3, 1))), "p": rng.choice([0.7, 0.75]),
                "lookback": rng.randint(1, 2), "plan": plan}
    if kind == "squaring":
        n = _log(rng, 442, 15000)
        return {"kind": "squaring", "n": n, "dtype": rng.choice(["int32", "int64"]),
                "layers": max(4, math.ceil(math.log2(n)) - rng.randint(2, 5)), "p": 0.7, "lookback": rng.randint(1, 3)}
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(20, 120), "lo": 16, "hi": _log(rng, 200, 3500)}
    n = _log(rng, 3000, 280_000)
    return {"kind": "order", "n": n, "dtype": rng.choice(["int32", "int64"]),
            "layers": max(4, min(13, math.ceil(math.log2(n)) - rng.randint(2, 6))), "p": 0.7, "lookback": 1}


# ---- inputs -----------------------------------------------------------------
def _spec(case, n):
    return synth.PedigreeSpec(n, case["layers"], case["p"], case["lookback"])


def _numbered(A, numbering, seed):
    if numbering == "upper":
        return synth.reverse_vertices(A)
    return synth.shuffle_vertices(A, seed) if numbering == "any" else A


def _matrix(case, n, seed, numbering="lower"):
    return _numbered(synth.dense_pedigree(_spec(case, n), seed, dtype=np.dtype(case["dtype"])), numbering, seed)


def _csr(case, seed):
    """One pedigree per case, its vertices renumbered by the seed within each
    layer: every seed's matrices differ, and all closures have one size."""
    n, layers = case["n"], case["layers"]
    rng = np.random.Generator(np.random.PCG64(seed))
    bounds = np.linspace(0, n, max(1, min(layers, n)) + 1).round().astype(np.int64)
    p = np.concatenate([lo + rng.permutation(hi - lo) for lo, hi in zip(bounds[:-1], bounds[1:])])
    A = synth.csr_pedigree(_spec(case, n), 0, dtype=np.dtype(case["dtype"]))[p][:, p]
    A.sort_indices()
    return A


def _insertions(case, seed):
    """The graph of a serving request stream and the parent edges a request
    adds: child in the later half, parent before it, of the sex the
    relationship needs, so that no edge closes a cycle."""
    n = case["n"]
    spec = synth.component_spec(n)
    is_red = synth.pedigree_edges(spec, seed)[0]
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    edges = []
    while len(edges) < case["edges"]:
        a = int(rng.integers(max(1, n // 2), n))
        rel = 2 if rng.random() < 0.5 else 3
        cand = np.nonzero(is_red[:a] == (rel == 2))[0]
        if cand.size:
            edges.append((a, int(cand[int(rng.integers(0, cand.size))]), rel))
    return synth.dense_pedigree(spec, seed), edges


def _batch_sizes(case):
    return synth.batched_sizes(case["count"], case["lo"], case["hi"], 0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        sizes = _batch_sizes(case)
        parts = [synth.component_edges(synth.component_spec(int(s)), synth.component_seed(seed, i))
                 for i, s in enumerate(sizes)]
        b = BatchedClosure(sizes, tri=1)
        b.load_edges([d for d, _ in parts], [e for _, e in parts])
        return {"kind": kind, "batch": b, "input": b.pool.clone()}
    et = elem_type(np.dtype(case["dtype"]))
    if kind == "closure":
        A = _matrix(case, case["n"], seed, case["numbering"])
        return {"kind": kind, "A": torch.from_numpy(A).cuda(), "et": et}
    if kind == "product":
        W = dense.fw_closure(torch.from_numpy(_matrix(case, case["k"], seed)).cuda(), et)[0]
        return {"kind": kind, "A": W[:case["m"], :].contiguous(), "B": W[:, :case["n"]].contiguous(), "et": et}
    if kind == "insert":
        A, edges = _insertions(case, seed)
        R = dense.fw_closure(torch.from_numpy(A).cuda(), et)[0].contiguous()
        return {"kind": kind, "R": R, "edges": edges, "et": et}
    S = _csr(case, seed)
    if kind == "dag" and case["plan"]:
        A = sd.from_scipy(S, np.dtype(case["dtype"]))
        plan = sd.DagPlan(case["n"], A.data.dtype, int(128 * S.nnz), S.nnz)
        return {"kind": "dag_plan", "A": A, "plan": plan}
    if kind in ("dag", "squaring"):
        return {"kind": kind, "A": CSRMatrixGPU.from_cpu(S)}
    C, _ = sd.dag_closure(sd.from_scipy(S, np.dtype(case["dtype"])))
    return {"kind": kind, "C": C}


# ---- the calls --------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "closure":
        W, out = dense.fw_closure(state["A"], state["et"])
        return {"W": W, "diameter": out.diameter}
    if kind == "product":
        C, st = dense.matmul(state["A"], state["B"], state["et"])
        return {"C": C, "events": int(st.events)}
    if kind == "insert":
        R, st = dense.edge_compose_many(state["R"], state["edges"], state["et"])
        return {"R": R, "events": int(st.events), "cycle": int(st.flags) & 4}
    if kind == "dag_plan":
        C, info = sd.dag_closure(state["A"], plan=state["plan"])
        return {"indptr": C.indptr, "indices": C.indices, "data": C.data, "diameter": info.diameter_candidates}
    if kind in ("dag", "squaring"):
        C, d = (transitive_closure_dag_gpu if kind == "dag" else transitive_closure_gpu)(state["A"])
        return {"indptr": C.indptr, "indices": C.indices, "data": C.data, "diameter": d}
    if kind == "batch":
        b = state["batch"]
        b.stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(b.stream):
            b.pool.copy_(state["input"])
        b.run(graph=True)
        outs = b.outcomes()
        return {"pool": b.pool,  # every component, each in its zero-padded square
                "diameter": np.array([o.diameter for o in outs], dtype=np.int64)}
    perm, P, counts = canonical_order_device(state["C"])
    return {"perm": perm, "indptr": P.indptr, "indices": P.indices, "data": P.data, "sizes": counts}


# ---- the work a pass cannot do without ---------------------------------------
def _ancestors(case):
    """Closure entries per vertex, roughly: a vertex d layers down is its own
    entry and has (2p)^g ancestors g generations up, a generation being
    (lookback + 1) / 2 layers."""
    per, step = 2.0 * case["p"], (case["lookback"] + 1) / 2.0
    total = 0.0
    for d in range(case["layers"]):
        total += sum(per ** g for g in range(int(d / step) + 1))
    return min(total / case["layers"], case["n"] / 2.0)


def work(case):
    kind = case["kind"]
    if kind == "closure":
        # the matrix read and written; a product and a minimum per cell
        e = np.dtype(case["dtype"]).itemsize
        return {"bytes": 2.0 * e * case["n"] ** 2, "flops": 2.0 * case["n"] ** 2}
    if kind == "product":
        e = np.dtype(case["dtype"]).itemsize
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": float(e) * (m * k + k * n + m * n), "flops": 2.0 * m * n}
    if kind == "insert":
        return {"bytes": 8.0 * case["n"] ** 2, "flops": 2.0 * case["n"] * case["edges"]}
    if kind == "batch":
        cells = float(sum(int(s) ** 2 for s in _batch_sizes(case)))
        return {"bytes": 8.0 * cells, "flops": 2.0 * cells}
    e = 4 + np.dtype(case["dtype"]).itemsize
    nnz_in = case["n"] * (1 + 2 * case["p"])
    nnz_out = case["n"] * _ancestors(case)
    if kind == "order":
        return {"bytes": 2.0 * (e * nnz_out + 8 * case["n"]) + 4.0 * case["n"], "flops": nnz_out}
    # the input read and the closure written
    return {"bytes": e * (nnz_in + nnz_out) + 16.0 * case["n"], "flops": 2.0 * nnz_out}


# ---- the same results in 64 bits ----------------------------------------------
def _msb(y):
    """floor(log2 y) of an int64 array of values >= 1 (exact below 2**53)."""
    return np.frexp(y.astype(np.float64))[1].astype(np.int64) - 1


def _join(x, y):
    """The AVOS product of two values >= 2: y's bits below its top one appended to x."""
    return ((x - 1) << _msb(y)) + y


def _naive(A):
    """The closure by the naive k-i-j loop, only over present operands, and
    floor(log2) of the largest value any cell ever held.  None where a value
    leaves the exact range of the float logarithm."""
    W = A.astype(np.int64)
    top = int(W.max(initial=0))
    for k in range(W.shape[0]):
        rows = np.nonzero(W[:, k])[0]
        cols = np.nonzero(W[k])[0]
        rows, cols = rows[rows != k], cols[cols != k]
        if rows.size == 0 or cols.size == 0:
            continue
        at = np.ix_(rows, cols)
        new = _join(W[rows, k][:, None], W[k, cols][None, :])
        old = W[at]
        new = np.where((old == 0) | (new < old), new, old)
        W[at] = new
        top = max(top, int(new.max()))
    return (W, top.bit_length() - 1 if top > 0 else 0) if top < 2 ** 52 else None


def exact(case, seed):
    kind = case["kind"]
    if kind == "closure":
        r = _naive(_matrix(case, case["n"], seed, case["numbering"]))
        return None if r is None else {"W": r[0], "diameter": r[1]}
    if kind == "product":
        r = _naive(_matrix(case, case["k"], seed))
        if r is None or r[1] > 25:
            return None
        A, B = r[0][:case["m"]], r[0][:, :case["n"]]
        C = np.zeros((case["m"], case["n"]), dtype=np.int64)
        for k in range(case["k"]):
            rows, cols = np.nonzero(A[:, k])[0], np.nonzero(B[k])[0]
            x, y = A[rows, k][:, None], B[k, cols][None, :]
            new = _join(np.abs(x), np.abs(y))
            # an identity on the right keeps an x of its own colour, one on
            # the left keeps every y but the other identity
            new = np.where(y == -1, np.where(x % 2 == 0, x, 0), new)
            new = np.where(y == 1, np.where(x % 2 == 1, x, 0), new)
            new = np.where(np.abs(x) == 1, np.where((np.abs(y) > 1) | (x == y), y, 0), new)
            at = np.ix_(rows, cols)
            old = C[at]
            C[at] = np.where((old == 0) | ((new != 0) & (new < old)), new, old)
        return {"C": C, "events": 0}
    if kind == "batch":
        parts, ds = [], []
        for i, size in enumerate(_batch_sizes(case)):
            r = _naive(synth.dense_pedigree(synth.component_spec(int(size)), synth.component_seed(seed, i)))
            if r is None:
                return None
            pad = max(1, (int(size) + 127) // 128) * 128 - int(size)
            parts.append(np.pad(r[0], ((0, pad), (0, pad))).reshape(-1))
            ds.append(r[1])
        return {"pool": np.concatenate(parts), "diameter": np.array(ds, dtype=np.int64)}
    return None  # whole numbers, and minutes of work in plain numpy
