"""Device-level dense operations: Floyd-Warshall closure, AVOS product,
relational composition.  Inputs and outputs are torch tensors resident on the
GPU, in the widened device domain (see _dtypes).  The reference-shaped API in
core.py wraps these.
"""
from __future__ import annotations

import ctypes
import threading
from dataclasses import dataclass

from . import _lib
from ._dtypes import ElemType, msb

FW_TILE = 128
ROWS_MAX_N = 32640  # rbg_fw_rows_max_n(): the largest order rbg_fw_rows_* takes
ROWS_ANY_MAX_N = 16384  # and the largest with entries above the diagonal
_tls = threading.local()


def _workspace(npad: int, elem: int):
    """The calling thread's snapshot workspace (one per thread and device:
    threads run closures on their own streams and must not share it)."""
    t = _lib.torch()
    dev = _lib.device()
    return _cached_bytes("ws_cache", (dev.index, npad, elem),
                         lambda: int(_lib.load().rbg_fw_tri_workspace_bytes(npad, elem)), t, dev)


def _cached_bytes(name: str, key: tuple, nbytes, t, dev):
    """The calling thread's byte buffer for ``key``; another key replaces it."""
    cache = getattr(_tls, name, None)
    if cache is None:
        cache = {}
        setattr(_tls, name, cache)
    ws = cache.get(key)
    if ws is None:
        ws = t.empty(nbytes(), dtype=t.uint8, device=dev)
        cache.clear()
        cache[key] = ws
    return ws


_ROWS_SIDES = {1: "lower", 2: "upper", 3: "full"}


def _rows_closure(src, work, n: int, npad: int, st: _lib.Status, stream):
    """rbg_fw_rows_* / rbg_fw_rows_any_*: the closure from the rows' direct
    entries.  Returns (closed or not, the schedule the entries' sides stand
    for or None when they are not known, status); status None where there is
    no room for the workspace."""
    t = _lib.torch()
    dev = _lib.device()
    elem = work.element_size()
    try:
        ws = _cached_bytes("rows_cache", (dev.index, n, elem),
                           lambda: int(_lib.load().rbg_fw_rows_workspace_bytes(n, elem)), t, dev)
    except t.OutOfMemoryError:
        return False, None, None
    sfx = "i32" if elem == 4 else "i64"
    sh = _lib.stream_handle(stream)
    _lib.call(f"rbg_fw_rows_{sfx}", _lib.ptr(src), n, src.stride(0), _lib.ptr(work), npad, _lib.ptr(ws), ws.numel(),
              st.p, sh)
    s = st.read(stream)
    if s.aux[5] > 1:
        try:
            largest = t.empty_like(work)
        except t.OutOfMemoryError:
            s.aux[5] = 0
        else:
            _lib.call(f"rbg_fw_rows_any_{sfx}", n, _lib.ptr(work), _lib.ptr(largest), npad, _lib.ptr(ws), ws.numel(),
                      st.p, sh)
            s = st.read(stream)
            if s.flags & _lib.F_NEED_GENERAL:
                s.aux[5] = s.flags = 0
    closed, sched = bool(s.aux[5]), _ROWS_SIDES.get(int(s.aux[6]))
    s.aux[5] = s.aux[6] = 0
    return closed, sched, s


def padded_order(n: int) -> int:
    return max(FW_TILE, ((n + FW_TILE - 1) // FW_TILE) * FW_TILE)


@dataclass
class FwOutcome:
    status: _lib.RbgStatus
    npad: int
    mode: str  # "fast" | "general"
    # the schedule that the entries' sides stand for: "full" | "lower" | "upper"
    # (closed from the rows' entries, else by the blocked schedules; "lower" is
    # then the persistent closure) | "lower-steps" (one launch per pivot step)
    schedule: str = "full"

    @property
    def diameter(self) -> int:
        return msb(self.status.diameter_max)

    def key_kij(self, key: int):
        n = self.npad
        return key // (n * n), (key // n) % n, key % n


def _run(work, et: ElemType, mode: int, st: _lib.Status, stream, tri: int = 0):
    t = _lib.torch()
    npad = work.shape[0]
    elem = work.element_size()
    ws = _workspace(npad, elem)
    fn = "rbg_fw_dense_tri_i32" if work.dtype == t.int32 else "rbg_fw_dense_tri_i64"
    _lib.call(fn, _lib.ptr(work), npad, npad, et.width, int(et.unsigned), mode, tri,
              _lib.ptr(ws), ws.numel(), st.p, _lib.stream_handle(stream))


def status() -> _lib.Status:
    """A per-thread reusable status block (device + pinned host mirror)."""
    st = getattr(_tls, "status", None)
    if st is None:
        st = _lib.Status()
        _tls.status = st
    return st


_TRI = {"full": 0, "lower": 1, "upper": 2, "lower-steps": 3}


def fw_closure(W, et: ElemType, stream=None, force_general: bool = False, schedule: str = "auto"):
    """Close an n x n device matrix.  Returns (closed n x n tensor, FwOutcome).

    The input tensor is not modified.  Runs the fast kernels when the input is
    inside their domain (rbg_fw_precheck) and falls back to the general kernels
    otherwise -- both on the GPU.  schedule "auto" takes the triangular
    schedule when the precheck finds every off-diagonal entry on one side of
    the diagonal (a pedigree numbered parents first is lower triangular), else
    the full one; "full" forces the full schedule (the results are the same).
    With "auto" an acyclic matrix of few entries per row (a pedigree, in any
    numbering) is closed from its rows' direct entries (rbg_fw_rows_*), with
    the schedule its entries' sides stand for.  Other lower triangular
    closures run as one persistent launch; "steps" keeps
    one launch per pivot step there (the same results again).
    """
    if schedule not in ("auto", "full", "steps"):
        raise ValueError(f"unknown schedule {schedule!r}")
    t = _lib.torch()
    n = W.shape[0]
    npad = padded_order(n)

    def fresh():
        if npad == n:
            return W.clone()
        w = t.zeros((npad, npad), dtype=W.dtype, device=W.device)
        w[:n, :n] = W
        return w

    st = status()
    fast = et.native and not force_general
    sched = "full"
    if fast:
        src = W if (W.stride(1) == 1 and W.stride(0) >= n) else W.contiguous()
        work = t.empty((npad, npad), dtype=W.dtype, device=W.device)
        known = None  # the schedule, where the rows' scan has found it
        if schedule == "auto" and 0 < n <= ROWS_MAX_N:
            closed, known, s = _rows_closure(src, work, n, npad, st, stream)
            if closed and not s.flags & _lib.F_NEED_GENERAL:
                return work[:n, :n], FwOutcome(s, npad, "fast", known)
            if closed or (s is not None and s.flags & _lib.F_PRECOND_FAIL):
                fast = False
    st.reset(stream)
    if fast:
        # one pass: copy, fast-domain check and encoding (rbg_fw_load_*)
        fn = "rbg_fw_load_i32" if work.dtype == t.int32 else "rbg_fw_load_i64"
        _lib.call(fn, _lib.ptr(src), n, src.stride(0), _lib.ptr(work), npad, st.p, _lib.stream_handle(stream))
        if known is not None:
            sched = known
        else:
            s = st.read(stream)
            if s.flags & _lib.F_PRECOND_FAIL:
                fast = False
                st.reset(stream)
            elif schedule in ("auto", "steps"):
                if not s.flags & _lib.F_HAS_UPPER:
                    sched = "lower" if schedule == "auto" else "lower-steps"
                elif not s.flags & _lib.F_HAS_LOWER:
                    sched = "upper"
    if not fast:
        work = fresh()
        sched = "full"
    _run(work, et, 2 if fast else 1, st, stream, _TRI[sched])
    s = st.read(stream)
    if fast and s.flags & _lib.F_STALLED:
        # a wait of the persistent closure ran out: the same schedule, one
        # launch per pivot step, on the original input
        work = fresh()
        st.reset(stream)
        sched = "lower-steps"
        _run(work, et, 0, st, stream, _TRI[sched])
        s = st.read(stream)
    mode = "fast" if fast else "general"
    # A cycle makes a diagonal value >= 2, after which products through the
    # pivot cell (skipped by the fast kernels) can raise events of their own:
    # the error path reruns in general mode, which records every event.
    if fast and (s.flags & _lib.F_NEED_GENERAL or s.cycle_count):
        work = fresh()
        st.reset(stream)
        _run(work, et, 1, st, stream)
        s = st.read(stream)
        mode = "general"
        sched = "full"
    return work[:n, :n], FwOutcome(s, npad, mode, sched)


# Products with fewer multiply-adds than this take the general kernel directly
# (the fast paths' scan of the operands costs more than it saves).
MATMUL_FAST_MIN_TERMS = 1 << 24


def matmul(A, B, et: ElemType, stream=None, force_general: bool = False):
    """C = A (x) B for device matrices (M x K) and (K x N).  Native-width
    operands with few entries (closures) take rbg_matmul_rows_* where their
    shape is one for it (rbg_matmul_rows_fits); others inside
    the fast domain (rbg_matmul_precheck's rules) rbg_matmul_fast_*; others,
    and a fast run whose MSB guard fails, take the general kernel with the
    full arithmetic and events."""
    t = _lib.torch()
    M, K = A.shape
    K2, N = B.shape
    assert K == K2
    C = t.empty((M, N), dtype=A.dtype, device=A.device)
    st = status()
    sfx = "i32" if A.dtype == t.int32 else "i64"
    sh = _lib.stream_handle(stream)
    A = A.contiguous()
    B = B.contiguous()
    if et.native and not force_general and M * K * N >= MATMUL_FAST_MIN_TERMS:
        ws = None
        if _lib.load().rbg_matmul_rows_fits(M, K, N, A.element_size()):
            size = int(_lib.load().rbg_matmul_rows_workspace_bytes(M, K, N, A.element_size()))
            try:
                ws = t.empty(size, dtype=t.uint8, device=A.device)
            except t.OutOfMemoryError:
                pass
        if ws is not None:
            # from the operands' entries, where they are few
            _lib.call(f"rbg_matmul_rows_{sfx}", _lib.ptr(A), K, _lib.ptr(B), N, _lib.ptr(C), N, M, K, N,
                      _lib.ptr(ws), ws.numel(), st.p, sh)
            s = st.read(stream)
            taken = bool(s.aux[5])
            s.aux[5] = 0
            if taken and not s.flags & _lib.F_NEED_GENERAL:
                s.flags = 0
                return C, s
            blocked = not taken and not s.flags & _lib.F_PRECOND_FAIL
            del ws
        else:
            st.reset(stream)
            _lib.call(f"rbg_matmul_precheck_{sfx}", _lib.ptr(A), K, M, K, st.p, sh)
            _lib.call(f"rbg_matmul_precheck_{sfx}", _lib.ptr(B), N, K, N, st.p, sh)
            blocked = not st.read(stream).flags & _lib.F_PRECOND_FAIL
        if blocked:
            ws = t.empty(int(_lib.load().rbg_matmul_fast_workspace_bytes(M, K, N, A.element_size())),
                         dtype=t.uint8, device=A.device)
            st.reset(stream)
            _lib.call(f"rbg_matmul_fast_{sfx}", _lib.ptr(A), K, _lib.ptr(B), N, _lib.ptr(C), N, M, K, N,
                      _lib.ptr(ws), ws.numel(), st.p, sh)
            s = st.read(stream)
            if not s.flags & _lib.F_NEED_GENERAL:
                return C, s
    st.reset(stream)
    _lib.call(f"rbg_matmul_{sfx}", _lib.ptr(A), K, _lib.ptr(B), N, _lib.ptr(C), N, M, K, N, et.width,
              int(et.unsigned), st.p, sh)
    return C, st.read(stream)


def edge_compose(R, alpha: int, beta: int, rel: int, et: ElemType, stream=None):
    t = _lib.torch()
    n = R.shape[0]
    out = t.empty_like(R)
    st = status()
    st.reset(stream)
    fn = "rbg_edge_compose_i32" if R.dtype == t.int32 else "rbg_edge_compose_i64"
    _lib.call(fn, _lib.ptr(R.contiguous()), n, alpha, beta, int(rel), _lib.ptr(out), et.width,
              int(et.unsigned), st.p, _lib.stream_handle(stream))
    return out, st.read(stream)


def edge_compose_many(R, edges, et: ElemType, stream=None, inplace: bool = False):
    """Apply edge compositions one after another without host round trips:
    each edge reads the previous result.  The compositions run in place on
    one copy of R (R itself too when ``inplace``), touching only the rows
    that reach each edge's source.  Returns (closure, status); status.flags
    has RBG_F_CYCLE when some edge would have closed a cycle, and the result
    is then meaningless."""
    t = _lib.torch()
    n = R.shape[0]
    st = status()
    st.reset(stream)
    fn = "rbg_edge_compose_many_i32" if R.dtype == t.int32 else "rbg_edge_compose_many_i64"
    sh = _lib.stream_handle(stream)
    cur = R if (inplace and R.is_contiguous()) else R.contiguous().clone()
    scratch = t.empty(int(_lib.load().rbg_edge_compose_scratch_bytes(n)), dtype=t.uint8, device=R.device)
    listed = [int(x) for a, b, rel in edges for x in (a, b, rel)]
    flat = (ctypes.c_int64 * len(listed))(*listed)
    _lib.call(fn, _lib.ptr(cur), n, flat, len(listed) // 3, _lib.ptr(scratch), et.width, int(et.unsigned), st.p, sh)
    return cur, st.read(stream)


def vertex_compose(u, R, v, color: int, et: ElemType, stream=None):
    t = _lib.torch()
    n = R.shape[0]
    out = t.zeros((n + 1, n + 1), dtype=R.dtype, device=R.device)
    st = status()
    st.reset(stream)
    fn = "rbg_vertex_compose_i32" if R.dtype == t.int32 else "rbg_vertex_compose_i64"
    _lib.call(fn, _lib.ptr(u.contiguous()), _lib.ptr(R.contiguous()), _lib.ptr(v.contiguous()), int(color), n,
              _lib.ptr(out), et.width, int(et.unsigned), st.p, _lib.stream_handle(stream))
    return out, st.read(stream)
