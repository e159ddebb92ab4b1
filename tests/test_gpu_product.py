"""The dense AVOS product's fast paths against the general kernel."""
import numpy as np
import pytest

from redblackgraph_amd import _lib, dense, synth
from redblackgraph_amd._dtypes import elem_type

pytestmark = pytest.mark.gpu


def _closure(n, layers, lookback, seed, dt, p=0.8):
    A = synth.dense_pedigree(synth.PedigreeSpec(n, layers, p, lookback), seed, dtype=dt)
    return dense.fw_closure(_lib.to_device(A), elem_type(dt))[0].contiguous()


@pytest.mark.parametrize("dt,n", [(np.int32, 700), (np.int64, 700), (np.int64, 1500)])
def test_matmul_fast_repeats(dt, n):
    """rbg_matmul_fast_* on a closure and its transpose (most cells of the
    result present), three runs: every cell the general kernel's."""
    t = _lib.torch()
    W = _closure(n, 14, 3, n, dt)
    B = W.t().contiguous()
    et = elem_type(dt)
    G, g = dense.matmul(W, B, et, force_general=True)
    sfx = "i32" if dt == np.int32 else "i64"
    ws = t.empty(int(_lib.load().rbg_matmul_fast_workspace_bytes(n, n, n, W.element_size())), dtype=t.uint8,
                 device=W.device)
    for _ in range(3):
        C = t.empty_like(W)
        st = dense.status()
        st.reset()
        _lib.call(f"rbg_matmul_fast_{sfx}", _lib.ptr(W), n, _lib.ptr(B), n, _lib.ptr(C), n, n, n, n, _lib.ptr(ws),
                  ws.numel(), st.p, _lib.stream_handle(None))
        assert st.read().flags == 0
        assert int((C != G).sum()) == 0


def _rows(A, B):
    """(taken, C, status) of one rbg_matmul_rows_* call; C starts at 77."""
    t = _lib.torch()
    Ad, Bd = _lib.to_device(A), _lib.to_device(B)
    (M, K), N = A.shape, B.shape[1]
    sfx = "i32" if A.dtype == np.int32 else "i64"
    ws = t.empty(int(_lib.load().rbg_matmul_rows_workspace_bytes(M, K, N, A.itemsize)), dtype=t.uint8, device=Ad.device)
    C = t.full((M, N), 77, dtype=Ad.dtype, device=Ad.device)
    st = dense.status()
    _lib.call(f"rbg_matmul_rows_{sfx}", _lib.ptr(Ad), K, _lib.ptr(Bd), N, _lib.ptr(C), N, M, K, N, _lib.ptr(ws),
              ws.numel(), st.p, _lib.stream_handle(None))
    s = st.read()
    return bool(s.aux[5]), C.cpu().numpy(), s


def _few(rng, rows, cols, per_row, dt, hi=200):
    """``per_row`` entries in every row: values 2..hi, and some of 1 and -1."""
    A = np.zeros((rows, cols), dtype=dt)
    for r in range(rows):
        at = rng.choice(cols, min(per_row, cols), replace=False)
        A[r, at] = rng.choice(np.r_[-1, 1, np.arange(2, hi)], at.size)
    return A


# rows and columns off the vectors and waves, more entries of a row than a
# wave has lanes, and more columns than one pass of a workgroup's LDS holds
@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("M,K,N,pa,pb", [(1, 1, 1, 1, 1), (3, 70, 5, 4, 1), (65, 130, 257, 9, 3), (40, 300, 1030, 3, 70),
                                         (200, 1000, 999, 130, 3), (70, 90, 16384, 2, 5), (33, 64, 17001, 1, 140)])
def test_matmul_rows_vs_oracle(orc, dt, M, K, N, pa, pb):
    rng = np.random.default_rng(M + K + N)
    A, B = _few(rng, M, K, pa, dt), _few(rng, K, N, pb, dt)
    taken, C, s = _rows(A, B)
    ref, ev = orc.matmul(A, B)
    pairs = int((A != 0).sum(0) @ (B != 0).sum(1))
    assert taken == (64 * pairs <= M * K * N)
    if taken:
        assert ev == 0 and not s.flags & _lib.F_NEED_GENERAL
        np.testing.assert_array_equal(C, ref)
    else:
        assert (C == 77).all()


@pytest.mark.parametrize("dt", [np.int32, np.int64])
def test_matmul_rows_declines(dt):
    rng = np.random.default_rng(1)
    A = _few(rng, 300, 300, 3, dt)
    W = A.copy()
    W[7] = 5  # a full row: more than a quarter
    assert not _rows(A, W)[0] and not _rows(W, A)[0]
    W = A.copy()
    W[5, 6] = -7
    taken, C, s = _rows(W, A)
    assert not taken and s.flags & _lib.F_PRECOND_FAIL and (C == 77).all()


@pytest.mark.parametrize("dt,bits", [(np.int32, 32), (np.int64, 64)])
def test_matmul_rows_overflow(orc, dt, bits):
    """The widest products that fit, and the first that does not: the facade
    then raises what the general kernel finds."""
    A, B = np.zeros((300, 300), dtype=dt), np.zeros((300, 300), dtype=dt)
    A[3, 5], B[5, 9] = 1 << (bits // 2), 1 << (bits // 2 - 2)
    taken, C, s = _rows(A, B)
    assert taken and s.flags == 0 and int(C[3, 9]) == 1 << (bits - 2)
    B[5, 9] = 1 << (bits // 2 - 1)
    taken, _, s = _rows(A, B)
    assert taken and s.flags & _lib.F_NEED_GENERAL
    et = elem_type(dt)
    C2, s2 = dense.matmul(_lib.to_device(A), _lib.to_device(B), et)
    C3, s3 = dense.matmul(_lib.to_device(A), _lib.to_device(B), et, force_general=True)
    assert s2.events == s3.events != 0
    np.testing.assert_array_equal(C2.cpu().numpy(), C3.cpu().numpy())


@pytest.mark.parametrize("dt,n", [(np.int32, 1100), (np.int64, 700)])
def test_matmul_of_closures_vs_general(dt, n):
    W = _closure(n, 12, 3, 5, dt)
    et = elem_type(dt)
    C, s = dense.matmul(W, W, et)
    G, g = dense.matmul(W, W, et, force_general=True)
    assert bool((C == G).all()) and s.events == g.events == 0 and s.flags == 0


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("M,K,N", [(1 << 20, 4, 4), (3, 5, 1 << 20), (300, 300, 300)])
def test_matmul_by_shape(orc, dt, M, K, N):
    """Products that the shape leaves to the blocked kernels, and one that it
    does not, by the facade."""
    rng = np.random.default_rng(M)
    A = ((rng.random((M, K)) < 0.2) * rng.integers(2, 90, (M, K))).astype(dt)
    B = ((rng.random((K, N)) < 0.2) * rng.integers(2, 90, (K, N))).astype(dt)
    for diagonal in (True, False):
        if not diagonal:  # inside the fast kernels' domain
            np.fill_diagonal(A, 0)
            np.fill_diagonal(B, 0)
        C, st = dense.matmul(_lib.to_device(A), _lib.to_device(B), elem_type(dt))
        ref, ev = orc.matmul(A, B)
        assert int(st.events) == ev == 0
        np.testing.assert_array_equal(C.cpu().numpy(), ref)


def test_matmul_without_room_for_the_entries(orc, monkeypatch):
    """Where the entries' workspace does not fit the memory the product takes
    the kernels that need none of it."""
    t = _lib.torch()
    rng = np.random.default_rng(1)
    n = 300
    A, B = _few(rng, n, n, 3, np.int32), _few(rng, n, n, 4, np.int32)
    size = int(_lib.load().rbg_matmul_rows_workspace_bytes(n, n, n, 4))
    empty = t.empty
    refused = []

    def no_room(shape, *args, **kw):
        if shape == size and kw.get("dtype") == t.uint8:
            refused.append(shape)
            raise t.OutOfMemoryError("no room")
        return empty(shape, *args, **kw)

    Ad, Bd = _lib.to_device(A), _lib.to_device(B)
    monkeypatch.setattr(t, "empty", no_room)
    C, st = dense.matmul(Ad, Bd, elem_type(np.int32))
    monkeypatch.undo()
    ref, ev = orc.matmul(A, B)
    assert refused and int(st.events) == ev
    np.testing.assert_array_equal(C.cpu().numpy(), ref)
