"""Levels that mix long and short closure rows, against the oracle."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from redblackgraph_amd import _lib
from redblackgraph_amd import sparse_dev as sd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    return oracle


def _check(orc, S, vdt, **kw):
    S = sp.csr_matrix(S).astype(vdt)
    C, info = sd.dag_closure(sd.canonicalize(sd.from_scipy(S, vdt)), **kw)
    ptr, idx, val = (x.cpu().numpy() for x in (C.indptr, C.indices, C.data))
    want = orc.dag_closure(S, 8 * np.dtype(vdt).itemsize)
    np.testing.assert_array_equal(ptr, want.indptr)
    np.testing.assert_array_equal(idx, want.indices)
    np.testing.assert_array_equal(val, want.data)
    assert (info.cand_max, info.final_max, info.nnz) == (want.cand_max, want.final_max, len(want.data))
    return info


@pytest.mark.parametrize("vdt", [np.int32, np.int64])
@pytest.mark.parametrize("n", [2000, 400_000])
def test_long_rows_between_short_ones(orc, vdt, n):
    """Level 1 holds rows of one to three candidates and, between them, rows of
    600: a short row behind a long one must not land in the long row's place."""
    rng = np.random.default_rng(n)
    sinks = n // 2
    rows, cols = [], []
    for v in range(sinks, n):
        k = 600 if v % 97 == 5 else 1 + v % 3
        c = rng.choice(sinks, k, replace=False)
        rows += [v] * k
        cols += list(c)
    S = sp.csr_matrix((rng.integers(2, 4, len(rows)), (rows, cols)), shape=(n, n))
    info = _check(orc, S, vdt)
    assert info.nlevels == 2 and info.cycle_vertex == -1


def _layered(n, per, fan, rng, values=(2, 4)):
    """Vertices numbered sinks first, `per` a level, `fan` successors in the
    level below, and a diagonal."""
    rows, cols = [np.arange(n)], [np.arange(n)]
    v = np.arange(per, n)
    for _ in range(fan):
        rows.append(v)
        cols.append((v // per - 1) * per + rng.integers(0, per, v.size))
    r, c = np.concatenate(rows), np.concatenate(cols)
    _, first = np.unique(r * n + c, return_index=True)
    r, c = r[first], c[first]
    return sp.csr_matrix((np.where(r == c, rng.choice([-1, 1], r.size), rng.integers(*values, r.size)), (r, c)),
                         shape=(n, n))


@pytest.mark.parametrize("vdt", [np.int32, np.int64])
@pytest.mark.parametrize("n,per,fan", [(1, 1, 1), (5, 1, 1), (63, 9, 1), (1000, 100, 3), (8192, 2048, 2),
                                       (8193, 2048, 2), (32_640, 5000, 2), (32_641, 5000, 2), (900, 90, 9)])
def test_sizes_of_the_one_workgroup_levels(orc, vdt, n, per, fan):
    S = _layered(n, per, fan, np.random.default_rng(n))
    info = _check(orc, S, vdt)
    assert info.nlevels == -(-n // per)
    perm = np.random.default_rng(1).permutation(n)  # any numbering
    _check(orc, S[perm][:, perm], vdt)


@pytest.mark.parametrize("levels", [249, 250, 251, 300])
def test_levels_past_the_one_workgroup_limit(orc, levels):
    """Deeper graphs take the rounds, with a plan (no wait) as without."""
    n = 3 * levels  # three chains of ones: no product grows
    v = np.arange(3, n)
    S = sp.csr_matrix((np.ones(v.size, np.int64), (v, v - 3)), shape=(n, n))
    A = sd.canonicalize(sd.from_scipy(S.astype(np.int64), np.int64))
    plan = sd.DagPlan(n, A.data.dtype, 400 * n, A.nnz)
    first, i1 = sd.dag_closure(A, plan=plan)
    again, i2 = sd.dag_closure(A, plan=plan)
    assert i1.nlevels == i2.nlevels == levels
    assert sd.csr_equal(first, again)
    want = orc.dag_closure(S, 64)
    np.testing.assert_array_equal(sd.to_scipy(first).toarray(), want.toarray(n))


@pytest.mark.parametrize("known", [False, True])
def test_cycles_and_small_buffers(known):
    """A cycle is named and a full arena grows, also with a plan whose level
    count is known."""
    n = 2000
    S = _layered(n, 200, 2, np.random.default_rng(2))
    A = sd.canonicalize(sd.from_scipy(S, np.int64))
    plan = sd.DagPlan(n, A.data.dtype, 400_000, A.nnz + 10)
    want, full = sd.dag_closure(A, plan=plan if known else None)
    tight = sd.DagPlan(n, A.data.dtype, full.arena // 10, A.nnz)
    if known:
        tight.levels, tight.out_nnz, tight.kinds = plan.levels, plan.out_nnz, plan.kinds
    got, info = sd.dag_closure(A, plan=tight)
    assert sd.csr_equal(got, want) and info.cycle_vertex == -1
    B = S.tolil()
    B[0, n - 1] = 2  # the first level reaches the last
    B = sd.canonicalize(sd.from_scipy(sp.csr_matrix(B), np.int64))
    C, info = sd.dag_closure(B, plan=plan if known else None)
    assert (C is None) == (info.cycle_vertex >= 0)
    reach = want.indices.cpu().numpy()[int(want.indptr[n - 1]):int(want.indptr[n])]
    assert (C is None) == (0 in reach)
    # a workspace without the predecessor lists is refused as before
    t = _lib.torch()
    bare = sd.DagPlan(n, A.data.dtype, 400_000, 0)
    from redblackgraph_amd.dense import status
    for rounds in (8, -plan.levels if known else 8):
        st = status()
        st.reset(None)
        _lib.call("rbg_dag_closure_i64", _lib.ptr(A.indptr), _lib.ptr(A.indices), _lib.ptr(A.data), n,
                  _lib.ptr(bare.ws), int(_lib.load().rbg_dag_workspace_bytes(n, 0)), _lib.ptr(bare.arena_cols),
                  _lib.ptr(bare.arena_vals), bare.arena_cols.numel(), rounds, None, 64, st.p,
                  _lib.stream_handle(None))
        s = st.read()
        assert not s.aux[7]
        assert rounds < 0 or s.flags & _lib.F_CAPACITY
    t.cuda.synchronize()


@pytest.mark.parametrize("vdt", [np.int32, np.int64])
@pytest.mark.parametrize("n", [6000, 40_000])
@pytest.mark.parametrize("direct", [0, 1, 5])
def test_long_rows_of_two_lists(orc, vdt, n, direct):
    """Rows of one and two successors whose candidates reach from one wave's
    share past the workgroup's, with shared columns, products that vanish
    (values -1 and 1) and direct entries inside and outside the lists."""
    rng = np.random.default_rng(direct)
    sinks, mid, top = 3000, [], []
    lengths = [1, 3, 255, 256, 257, 400, 500, 511, 512, 640, 1022, 1023, 1024, 1025, 1500, 2040]
    rows, cols = [], []

    def add(v, c):
        rows.extend([v] * len(c))
        cols.extend(int(x) for x in c)

    for q, k in enumerate(lengths):
        for rep in range(2):
            v = sinks + len(mid)
            mid.append(k)
            add(v, rng.choice(sinks, k, replace=False))
    for a in range(len(mid)):
        for b in (a, a ^ 1, (a + 7) % len(mid), (a + 13) % len(mid)):
            v = sinks + len(mid) + len(top)
            top.append((a, b))
            c = {sinks + a, sinks + b} | set(rng.choice(sinks, direct, replace=False).tolist())
            add(v, sorted(c))
    order = rng.permutation(sinks + len(mid) + len(top)) if direct == 1 else np.arange(n)
    rows, cols = np.array(rows), np.array(cols)
    if direct == 1:
        rows, cols = order[rows], order[cols]
    S = sp.csr_matrix((rng.choice([-1, 1, 2, 3], rows.size), (rows, cols)), shape=(n, n))
    info = _check(orc, S, vdt)
    assert info.nlevels == 3


def _row_lengths(lengths, n=3000):
    """A sink per vertex but the last ones, which have rows of the given
    numbers of entries (the diagonal among them)."""
    S = sp.eye(n, dtype=np.int64).tolil()
    for q, k in enumerate(lengths):
        S[n - 1 - q, :k - 1] = 2
    return S.tocsr()


def _calls(monkeypatch, name):
    said = []
    call = _lib.call

    def counted(fn, *args):
        if fn.startswith(name):
            said.append(fn)
        return call(fn, *args)

    monkeypatch.setattr(_lib, "call", counted)
    return said


# the squares of rows of more than 7 entries sum to at most 65,536
@pytest.mark.parametrize("lengths,rounds", [([7] * 2000, False), ([256], False), ([257], True), ([1500], True),
                                            ([64] * 16, False), ([64] * 16 + [8], True), ([8] * 1024, False),
                                            ([8] * 1025, True), ([100] * 16, True)])
def test_long_rows_are_the_rounds(orc, monkeypatch, lengths, rounds):
    """Which launches close a graph shows in its plan's kinds, and the plan's
    next closure takes the same ones at once."""
    S = _row_lengths(lengths)
    A = sd.canonicalize(sd.from_scipy(S, np.int64))
    plan = sd.DagPlan(A.n_rows, A.data.dtype, 400_000, A.nnz)
    want = orc.dag_closure(S, 64).toarray(A.n_rows)
    said = _calls(monkeypatch, "rbg_dag_closure")
    for _ in range(3):
        C, _ = sd.dag_closure(A, plan=plan)
        assert [bool(k & 4) for k in plan.kinds] == [rounds] * plan.levels
        np.testing.assert_array_equal(sd.to_scipy(C).toarray(), want)
    assert len(said) == 3


def test_closed_graph_closed_again(orc):
    """A closure is its own closure, and has rows too long for the launches of
    small graphs."""
    from redblackgraph_amd import synth
    S = synth.csr_pedigree(synth.PedigreeSpec(2000, 11, 0.7, 1), 0)
    C, _ = sd.dag_closure(sd.from_scipy(S, np.int64))
    plan = sd.DagPlan(C.n_rows, C.data.dtype, 64 * C.nnz, C.nnz)
    for _ in range(2):
        again, _ = sd.dag_closure(C, plan=plan)
        assert sd.csr_equal(again, C) and all(k & 4 for k in plan.kinds)


@pytest.mark.parametrize("graph", ["deep", "long rows", "pedigree"])
def test_rounds_without_a_wait(monkeypatch, graph):
    """A level count alone closes any graph of so many levels without a wait;
    a deep graph's plan does it by one call as well."""
    from redblackgraph_amd import synth
    from redblackgraph_amd.dense import status
    n = 900
    if graph == "deep":
        v = np.arange(3, n)
        S = sp.csr_matrix((np.ones(v.size, np.int64), (v, v - 3)), shape=(n, n))
    elif graph == "long rows":
        S = _row_lengths([300, 200], n)
    else:
        S = synth.csr_pedigree(synth.PedigreeSpec(n, 10, 0.7, 1), 0)
    A = sd.canonicalize(sd.from_scipy(S.astype(np.int64), np.int64))
    plan = sd.DagPlan(n, A.data.dtype, 400 * n, A.nnz)
    said = _calls(monkeypatch, "rbg_dag_closure")
    want, _ = sd.dag_closure(A, plan=plan)
    got, _ = sd.dag_closure(A, plan=plan)
    assert sd.csr_equal(got, want) and len(said) == 2
    st = status()
    st.reset(None)
    _lib.call("rbg_dag_closure_i64", _lib.ptr(A.indptr), _lib.ptr(A.indices), _lib.ptr(A.data), n, _lib.ptr(plan.ws),
              plan.ws.numel(), _lib.ptr(plan.arena_cols), _lib.ptr(plan.arena_vals), plan.arena_cols.numel(),
              -plan.levels, None, 64, st.p, _lib.stream_handle(None))
    s = st.read()
    assert s.aux[7] == 1 and s.aux[6] == plan.levels


def _queued(A, plan, ws_bytes=None, kinds=None, batch=None):
    """The status of a closure queued without a wait."""
    from redblackgraph_amd.dense import status
    st = status()
    st.reset(None)
    kinds = (ctypes.c_uint8 * plan.levels).from_buffer_copy(plan.kinds if kinds is None else kinds)
    _lib.call("rbg_dag_closure_i64", _lib.ptr(A.indptr), _lib.ptr(A.indices), _lib.ptr(A.data), A.n_rows,
              _lib.ptr(plan.ws), plan.ws.numel() if ws_bytes is None else ws_bytes, _lib.ptr(plan.arena_cols),
              _lib.ptr(plan.arena_vals), plan.arena_cols.numel(), -plan.levels if batch is None else batch,
              ctypes.cast(kinds, ctypes.c_void_p), 64, st.p, _lib.stream_handle(None))
    return st.read()


@pytest.mark.parametrize("n,per,fan", [(3, 1, 1), (2000, 200, 2), (9000, 900, 3), (32_640, 4000, 2)])
@pytest.mark.parametrize("from_level", [0, 1, 2])
def test_cycles_are_named_without_a_wait(n, per, fan, from_level):
    """With an earlier graph's levels and kinds, a cycle is reported with a
    vertex on it and the levels below it, as by the rounds; a workspace without
    room for the predecessor lists is refused."""
    S = _layered(n, per, fan, np.random.default_rng(n))
    A = sd.canonicalize(sd.from_scipy(S, np.int64))
    plan = sd.DagPlan(n, A.data.dtype, 1 << 24, A.nnz + 10)
    sd.dag_closure(A, plan=plan)
    s = _queued(A, plan)
    assert s.aux[7] == 1 and s.aux[6] == plan.levels and not s.flags & (_lib.F_CYCLE | _lib.F_CAPACITY)
    if n > 3:  # three vertices' lists fit what the sizes are rounded up by
        s = _queued(A, plan, ws_bytes=int(_lib.load().rbg_dag_workspace_bytes(n, 0)))
        assert not s.aux[7] and s.flags & _lib.F_CAPACITY
    low = from_level * per  # a vertex of that level, and one above it that reaches it
    v = n - 1
    while v >= low + per:
        v = int(S.indices[S.indptr[v]:S.indptr[v + 1]][0])
    top = n - 1
    B = S.tolil()
    B[v, top] = 2
    B = sp.csr_matrix(B)
    B = sd.canonicalize(sd.from_scipy(B, np.int64))
    s = _queued(B, plan)
    C, info = sd.dag_closure(B, plan=plan)
    from scipy.sparse.csgraph import connected_components
    H = sd.to_scipy(B)
    H = sp.csr_matrix((np.abs(H.data), H.indices, H.indptr), shape=H.shape)
    _, comp = connected_components(H, directed=True, connection="strong")
    size = np.bincount(comp)
    if v == top:  # an entry on the diagonal
        assert size.max() == 1 and s.aux[7] == 1 and not s.flags & _lib.F_CYCLE and C is not None
        return
    assert s.flags & _lib.F_CYCLE and not s.aux[7] and size[comp[int(s.aux[0])]] > 1
    assert C is None and size[comp[info.cycle_vertex]] > 1
    # the levels placed: the longest paths among the vertices that reach no cycle
    inside = size[comp] > 1
    bad = inside.copy()
    for _ in range(n):
        more = bad | (np.asarray((H != 0).astype(np.int64) @ bad).ravel() > 0)
        if (more == bad).all():
            break
        bad = more
    assert s.aux[6] == info.nlevels == max((x // per + 1 for x in np.nonzero(~bad)[0]), default=0)


def test_plan_reused_for_another_graph(orc, monkeypatch):
    """Kinds of another graph of the same size cost a small graph no second
    closure, and the plan then holds its own."""
    n = 3000
    rng = np.random.default_rng(4)
    graphs = [_layered(n, 300, 1, rng), _layered(n, 300, 3, rng), _layered(n, 500, 3, rng)]
    As = [sd.canonicalize(sd.from_scipy(S, np.int64)) for S in graphs]
    plan = sd.DagPlan(n, As[0].data.dtype, 1 << 24, max(A.nnz for A in As))
    kinds = []
    for S, A in zip(graphs, As):
        own = sd.DagPlan(n, A.data.dtype, 1 << 24, A.nnz)
        sd.dag_closure(A, plan=own)
        kinds.append((own.levels, own.kinds))
    assert kinds[0][0] == kinds[1][0] > kinds[2][0] and kinds[0][1] != kinds[1][1]
    sd.dag_closure(As[0], plan=plan)
    said = _calls(monkeypatch, "rbg_dag_closure")
    for q in (1, 2):
        C, info = sd.dag_closure(As[q], plan=plan)
        want = orc.dag_closure(graphs[q], 64)
        np.testing.assert_array_equal(C.indptr.cpu().numpy(), want.indptr)
        np.testing.assert_array_equal(C.indices.cpu().numpy(), want.indices)
        np.testing.assert_array_equal(C.data.cpu().numpy(), want.data)
        assert (plan.levels, plan.kinds) == kinds[q] and info.nlevels == kinds[q][0]
    assert len(said) == 2
