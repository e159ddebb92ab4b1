"""The fused squaring step (rbg_csr_square_*) against the AVOS product, the
smallest-|value| merge and the comparison run one after another; and the
permutation of rows with repeated columns."""
import numpy as np
import pytest
import scipy.sparse as sp

from redblackgraph_amd import _lib, synth
from redblackgraph_amd import sparse_dev as sd

pytestmark = pytest.mark.gpu


def _plain(R, upper):
    R2, _ = sd.spgemm(R, R, mask_upper=upper)
    N = sd.avos_sum_csr(R, R2, min_abs=True)
    return None if sd.csr_equal(R, N) else N


def _same(S, dt, upper=False, steps=12):
    R = sd.canonicalize(sd.from_scipy(S, dt))
    for _ in range(steps):
        N, P = sd.square_step(R, upper), _plain(R, upper)
        assert (N is None) == (P is None)
        if N is None:
            return R
        assert sd.csr_equal(N, P)
        R = N
    return R


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("n,layers,lookback", [(1, 1, 1), (2, 2, 1), (65, 5, 2), (1300, 9, 1), (700, 18, 2)])
def test_square_step_pedigrees(dt, n, layers, lookback):
    S = synth.csr_pedigree(synth.PedigreeSpec(n, layers, 0.8, lookback), n, dtype=dt)
    _same(S, dt)
    _same(S.T.tocsr(), dt, upper=True)


@pytest.mark.parametrize("dt", [np.int32, np.int64])
def test_square_step_signs_and_ties(dt):
    """Values -1, 1 and up in any place, cycles included: the merge keeps R's
    entry on ties of the absolute value."""
    rng = np.random.default_rng(3)
    for n, density in ((30, 0.3), (200, 0.03)):
        A = (rng.random((n, n)) < density) * rng.choice([-1, 1, 2, 3, 4, 5], (n, n))
        _same(sp.csr_matrix(A.astype(dt)), dt, steps=2)
        _same(sp.csr_matrix(A.astype(dt)), dt, upper=True, steps=2)


@pytest.mark.parametrize("columns,fused", [(767, True), (768, True), (769, False)])
def test_square_step_row_limit(columns, fused):
    """A row of N with 768 columns stays in the table, one more takes the
    separate kernels."""
    n = 900
    A = np.zeros((n, n), dtype=np.int64)
    A[0, 1] = 2
    A[1, 2:columns + 1] = 3  # row 0 of N: column 1 and row 1's
    R = sd.canonicalize(sd.from_scipy(sp.csr_matrix(A), np.int64))
    t = _lib.torch()
    from redblackgraph_amd.dense import status
    st, temp = status(), sd.glue_temp(n, R.indices.device)
    ptr = t.empty(n + 1, dtype=t.int64, device=R.indices.device)
    _lib.call("rbg_csr_square_count_i64", _lib.ptr(R.indptr), _lib.ptr(R.indices), _lib.ptr(R.data), n, 0,
              _lib.ptr(ptr), _lib.ptr(temp), temp.numel(), 64, st.p, _lib.stream_handle(None))
    s = st.read()
    assert bool(s.flags & _lib.F_CAPACITY) == (not fused)
    if fused:
        assert s.aux[0] != 0 and s.aux[1] == columns + columns - 1 == int(ptr[n])
    assert sd.csr_equal(sd.square_step(R), _plain(R, False))


def test_square_step_many_rows():
    """More rows than the one-workgroup row-pointer scan takes."""
    S = synth.csr_pedigree(synth.PedigreeSpec(70_001, 3, 0.7, 1), 1, dtype=np.int32)
    _same(S, np.int32, steps=1)


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("length", [1, 3, 64, 65, 255, 256, 257, 511, 512, 513, 700])
def test_permute_csr_rows_with_repeated_columns(dt, length):
    """Rows on both sides of the lengths ranked in place; every second one
    repeats columns, and equal columns keep their order."""
    from redblackgraph_amd.sparse.csgraph._ordering import _permute_csr_device
    t = _lib.torch()
    rng = np.random.default_rng(length)
    n = 800
    rows = [np.sort(rng.choice(n, length, replace=bool(r % 2))) for r in range(4)] + [np.zeros(0, np.int64)] * (n - 4)
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    idx = np.concatenate(rows).astype(np.int32)
    val = np.arange(1, idx.size + 1).astype(dt)
    p = rng.permutation(n).astype(np.int32)
    inv = np.argsort(p)
    optr, oidx, oval = _permute_csr_device(_lib.to_device(ptr), _lib.to_device(idx), _lib.to_device(val), n, idx.size,
                                           np.dtype(dt), _lib.to_device(p))
    optr, oidx, oval = optr.cpu().numpy(), oidx.cpu().numpy(), oval.cpu().numpy()
    t.cuda.synchronize()
    for i in range(n):
        cols, vals = inv[idx[ptr[p[i]]:ptr[p[i] + 1]]], val[ptr[p[i]]:ptr[p[i] + 1]]
        order = np.argsort(cols, kind="stable")
        np.testing.assert_array_equal(oidx[optr[i]:optr[i + 1]], cols[order])
        np.testing.assert_array_equal(oval[optr[i]:optr[i + 1]], vals[order])


def _labels(S):
    from redblackgraph_amd.sparse.csgraph._components import _device_labels
    return _device_labels(S).cpu().numpy()


@pytest.mark.parametrize("shape", ["one", "none", "star", "path", "blocks", "pedigree", "shuffled"])
def test_components_one_pass(shape):
    """Labels (the smallest vertex of each component) of graphs whose first
    forests differ: no edges, a star, a path, equal blocks, pedigrees in order
    and shuffled."""
    from scipy.sparse.csgraph import connected_components
    rng = np.random.default_rng(5)
    n = 1 if shape == "one" else 20_011
    if shape in ("one", "none"):
        S = sp.csr_matrix((n, n), dtype=np.int32)
    elif shape == "star":
        S = sp.csr_matrix((np.ones(n - 1, np.int32), (np.arange(1, n), np.zeros(n - 1, int))), shape=(n, n))
    elif shape == "path":
        q = rng.permutation(n)
        S = sp.csr_matrix((np.ones(n - 1, np.int32), (q[:-1], q[1:])), shape=(n, n))
    elif shape == "blocks":
        r, c = rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n)
        keep = r // 50 == c // 50
        S = sp.csr_matrix((np.ones(keep.sum(), np.int32), (r[keep], c[keep])), shape=(n, n))
    else:
        S = synth.csr_pedigree(synth.PedigreeSpec(n, 9, 0.6, 2), 3, dtype=np.int32)
        if shape == "shuffled":
            q = rng.permutation(n)
            S = S[q][:, q].tocsr()
    for _ in range(3):
        lab = _labels(S)
        _, comp = connected_components(S, directed=False)
        least = np.full(comp.max() + 1, n)
        np.minimum.at(least, comp, np.arange(n))
        np.testing.assert_array_equal(lab, least[comp])


def _crowded(dt):
    """Rows of the closure past 1,024 columns: nearly every parent known."""
    return synth.csr_pedigree(synth.PedigreeSpec(4000, 16, 0.95, 1), 0, dtype=dt)


def test_squaring_closure_leaves_the_fused_step_for_good(monkeypatch):
    """Rows only grow: after the first step with a row past the limit the
    fused kernel is not tried again."""
    from redblackgraph_amd.gpu import CSRMatrixGPU, transitive_closure_gpu
    said = []
    call = _lib.call

    def counted(fn, *args):
        if fn.startswith("rbg_csr_square") or fn.startswith("rbg_spgemm"):
            said.append(fn[:16])
        return call(fn, *args)

    S = _crowded(np.int64)
    monkeypatch.setattr(_lib, "call", counted)
    C, _ = transitive_closure_gpu(CSRMatrixGPU.from_cpu(S))
    monkeypatch.undo()
    tried, plain = ([k for k, f in enumerate(said) if f.startswith(p)] for p in ("rbg_csr_square", "rbg_spgemm"))
    assert len(plain) >= 2 and max(tried) < min(plain)
    R = sd.canonicalize(sd.from_scipy(S, np.int64))
    N = _plain(R, False)
    while N is not None:
        R, N = N, _plain(N, False)
    assert sd.csr_equal(C._dev(), R)


@pytest.mark.parametrize("dt", [np.int32, np.int64])
def test_square_count_stops_at_the_limit(dt):
    """Counting a step whose rows pass the limit costs less than half of the
    product that then has to be computed (a tenth or so; a count that went on
    to the end cost as much as the whole step)."""
    from redblackgraph_amd.dense import status
    t = _lib.torch()
    R = sd.canonicalize(sd.from_scipy(_crowded(dt), dt))
    sfx, n = "i32" if dt == np.int32 else "i64", R.n_rows
    st, temp = status(), sd.glue_temp(n, R.indices.device)
    ptr = t.empty(n + 1, dtype=t.int64, device=R.indices.device)

    def count(M):
        _lib.call(f"rbg_csr_square_count_{sfx}", _lib.ptr(M.indptr), _lib.ptr(M.indices), _lib.ptr(M.data), n, 0,
                  _lib.ptr(ptr), _lib.ptr(temp), temp.numel(), 8 * np.dtype(dt).itemsize, st.p, _lib.stream_handle(None))

    def ms(fn):
        best = []
        for _ in range(5):
            a, b = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    declined = 0
    while R is not None:  # the last step, which changes nothing, is declined too
        count(R)
        if st.read().flags & _lib.F_CAPACITY:
            declined += 1
            assert ms(lambda: count(R)) < 0.5 * ms(lambda: _plain(R, False))
        R = _plain(R, False)
    assert declined >= 2


@pytest.mark.parametrize("n", [5, 1024, 1025, 4097, 300_000])
@pytest.mark.parametrize("shape", ["path", "path down", "two paths", "comb", "random"])
def test_components_of_long_paths(n, shape):
    """Vertices in a row, each joined to the one before: first forests as deep
    as the graph, alone, two of them crossing, with teeth, and none."""
    from scipy.sparse.csgraph import connected_components
    rng = np.random.default_rng(n)
    r, c = np.arange(1, n), np.arange(n - 1)
    if shape == "path down":
        r, c = c, r
    elif shape == "two paths":  # even and odd vertices, joined by the last edge
        r, c = np.r_[np.arange(2, n), n - 1], np.r_[np.arange(n - 2), n - 2]
    elif shape == "comb":  # every third vertex hangs from the first third's path
        k = max(1, n // 3)
        r, c = np.r_[np.arange(1, k), np.arange(k, n)], np.r_[np.arange(k - 1), np.arange(n - k) % k]
    elif shape == "random":
        r, c = rng.integers(0, n, n // 2), rng.integers(0, n, n // 2)
    S = sp.csr_matrix((np.ones(len(r), np.int32), (r, c)), shape=(n, n))
    S.sort_indices()
    lab = _labels(S)
    _, comp = connected_components(S, directed=False)
    least = np.full(comp.max() + 1, n)
    np.minimum.at(least, comp, np.arange(n))
    np.testing.assert_array_equal(lab, least[comp])


def test_components_of_a_long_path_cost_no_walk():
    """A path of a million vertices in their order takes about as long as one in
    a shuffled order (a walk down the whole path took ten times)."""
    from redblackgraph_amd.sparse.csgraph._components import _device_labels_dev
    t = _lib.torch()
    n = 1_000_000
    q = np.random.default_rng(1).permutation(n)

    def ms(r, c):
        A = sd.from_scipy(sp.csr_matrix((np.ones(n - 1, np.int32), (r, c)), shape=(n, n)), np.int32)
        best = []
        for _ in range(6):
            a, b = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            a.record()
            _device_labels_dev(A)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    assert ms(np.arange(1, n), np.arange(n - 1)) < 3 * ms(q[1:], q[:-1])


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("n", [1, 31, 33, 262_143, 262_144, 262_209])
def test_sum_of_short_and_empty_rows(dt, n):
    """Either side of the row count from which a wave moves 64 rows: rows of
    none to three entries, columns of both, one and neither matrix."""
    rng = np.random.default_rng(n)

    def some():
        k = rng.integers(0, 4, n)
        return sp.csr_matrix((rng.integers(1, 9, k.sum()).astype(dt), (np.repeat(np.arange(n), k),
                                                                       rng.integers(0, min(n, 5), k.sum()))),
                             shape=(n, n))

    A, B = some(), some()
    C = sd.to_scipy(sd.avos_sum_csr(sd.canonicalize(sd.from_scipy(A, dt)), sd.canonicalize(sd.from_scipy(B, dt))))
    assert C.has_sorted_indices
    a, b = A[:, :5].toarray(), B[:, :5].toarray()
    want = np.where(a == 0, b, np.where(b == 0, a, np.minimum(a, b)))
    np.testing.assert_array_equal(C[:, :5].toarray(), want)
    assert C.nnz == np.count_nonzero(want)
