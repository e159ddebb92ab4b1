"""Edge compositions queued one launch an edge, against the out-of-place
composition applied edge by edge."""
import numpy as np
import pytest

from redblackgraph_amd import _lib, dense, synth
from redblackgraph_amd._dtypes import elem_type

pytestmark = pytest.mark.gpu


def _edges(n, kind, rng):
    """Edges (alpha, beta, rel) from a vertex to an earlier one: no cycles in a
    lower triangular closure."""
    if kind == "chain":  # each edge's source is the next one's target or source
        v = np.sort(rng.choice(n, min(n, 40), replace=False))
        return [(int(b), int(a), int(rng.integers(2, 4))) for a, b in zip(v[:-1], v[1:])]
    if kind == "same":  # one source again and again: its row was just replaced
        return [(n - 1, int(b), 2 + int(q % 2)) for q, b in enumerate(rng.choice(n - 1, min(n - 1, 20), replace=False))]
    if kind == "down":  # sources from the last to the first: every later row reaches them
        v = np.sort(rng.choice(np.arange(1, n), min(n - 1, 40), replace=False))[::-1]
        return [(int(a), int(rng.integers(0, a)), int(rng.integers(2, 4))) for a in v]
    v = rng.integers(1, n, 50)
    return [(int(a), int(rng.integers(0, a)), int(rng.integers(2, 4))) for a in v]


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("kind", ["chain", "same", "down", "random"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 700, 4096, 4097, 5003])
def test_edges_one_launch_each(n, kind, dtype):
    rng = np.random.default_rng(n)
    layers = max(2, min(10, int(np.log2(n)) + 1))
    A = synth.dense_pedigree(synth.PedigreeSpec(n, layers, 0.6, 1), n, dtype=dtype)
    et = elem_type(dtype)
    R = dense.fw_closure(_lib.to_device(np.tril(A)), et)[0].contiguous()
    edges = _edges(n, kind, rng)
    if n > 4000:
        edges = edges[:12]
    want, events, flags = R, 0, 0
    for a, b, rel in edges:
        want, st = dense.edge_compose(want, a, b, rel, et)
        events, flags = events | int(st.events), flags | int(st.flags)
    before = R.clone()
    got, st = dense.edge_compose_many(R, edges, et)
    assert bool((R == before).all())
    assert bool((got == want).all())
    assert int(st.events) == events and int(st.flags) == flags
    inplace, st = dense.edge_compose_many(R, edges, et, inplace=True)
    assert bool((inplace == want).all()) and int(st.flags) == flags
    none, st = dense.edge_compose_many(before, [], et)
    assert bool((none == before).all()) and int(st.flags) == 0


def _full(n, density, dt, seed):
    """A lower triangular matrix with that share of its cells below the
    diagonal present, made on the device."""
    t = _lib.torch()
    g = t.Generator(device="cuda").manual_seed(seed)
    R = t.zeros((n, n), dtype=dt, device="cuda")
    for i in range(0, n, 4096):
        k = min(4096, n - i)
        R[i:i + k] = (t.rand((k, n), device="cuda", generator=g) < density) * \
            t.randint(2, 900, (k, n), device="cuda", generator=g, dtype=dt)
    R = t.tril(R, -1)
    R.fill_diagonal_(1)
    return R


def _one_by_one(R, edges, et):
    events = flags = 0
    for a, b, rel in edges:
        R, st = dense.edge_compose(R, a, b, rel, et)
        events |= int(st.events)
        flags |= int(st.flags)
    return R, events, flags


@pytest.mark.parametrize("dt", ["int32", "int64"])
@pytest.mark.parametrize("n,density", [(1, 1.0), (63, 1.0), (255, 0.5), (256, 1.0), (257, 0.5), (1023, 0.3),
                                       (1025, 1.0), (4097, 0.02), (12_000, 0.01), (24_001, 0.0005)])
def test_edges_into_full_rows(dt, n, density):
    """Spans of lefts, chunks of columns and their remainders, against one edge
    at a time by its own kernels: repeated, chained and crossing sources."""
    t = _lib.torch()
    et = elem_type(np.dtype(dt))
    R = _full(n, density, getattr(t, dt), n)
    rng = np.random.default_rng(n)
    edges = [(int(rng.integers(n // 2, n)), int(rng.integers(0, n // 2 + 1)), int(rng.integers(2, 4))) for _ in range(5)]
    edges += [(edges[-1][0], 0, 3), (n - 1, edges[0][0], 2), (edges[0][0], edges[0][1], 0)]
    want, events, flags = _one_by_one(R, edges, et)
    got, st = dense.edge_compose_many(R, edges, et)
    assert t.equal(got, want)
    assert (int(st.events), int(st.flags) & _lib.F_CYCLE) == (events, flags & _lib.F_CYCLE)


def test_edges_into_full_rows_cost_less_than_one_by_one():
    """Updating in place what each edge changes is cheaper than a copy of the
    matrix for each, also where rows and columns are full (about a half; with
    the columns' workgroups alone it took twice the time)."""
    t = _lib.torch()
    et = elem_type(np.int32)
    R = _full(4095, 0.3, t.int32, 1)
    rng = np.random.default_rng(3)
    edges = [(int(rng.integers(2047, 4095)), int(rng.integers(0, 2047)), 2) for _ in range(16)]

    def ms(fn):
        best = []
        for _ in range(6):
            a, b = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    assert ms(lambda: dense.edge_compose_many(R, edges, et)) < ms(lambda: _one_by_one(R, edges, et))


def test_edges_of_any_iterable():
    """Edges come from a generator, an array or rows of one, and each has three
    numbers."""
    t = _lib.torch()
    et = elem_type(np.int32)
    R = _full(300, 0.1, t.int32, 2)
    edges = [(290, 10, 2), (200, 20, 3), (299, 200, 2)]
    want, _ = dense.edge_compose_many(R, edges, et)
    for form in ((e for e in edges), np.array(edges), [np.array(e, dtype=np.uint8 if max(e) < 256 else np.int64) for e in edges],
                 map(list, edges), dict.fromkeys(edges), zip(*zip(*edges))):
        got, _ = dense.edge_compose_many(R, form, et)
        assert t.equal(got, want)
    for wrong in ([(290, 10)], [(290, 10, 2, 1)], [(290, 10), (2, 200, 20, 3)], [290, 10, 2]):
        with pytest.raises((TypeError, ValueError)):
            dense.edge_compose_many(R, wrong, et)
