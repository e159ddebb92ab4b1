"""The dense closure from the rows' direct entries (rbg_fw_rows_*): which
matrices it takes, and W, diameter and status against the oracle's naive loop
and the blocked full schedule, at the edges of its slabs, slots and levels."""
import numpy as np
import pytest

from redblackgraph_amd import _lib, dense, synth
from redblackgraph_amd._dtypes import elem_type

pytestmark = pytest.mark.gpu


def _rows(A, lda=None):
    """(schedule or None, W, status) of one closure from the rows."""
    t = _lib.torch()
    n = A.shape[0]
    big = np.zeros((n, lda or n), dtype=A.dtype)
    big[:, :n] = A
    src = _lib.to_device(big)[:, :n]
    npad = dense.padded_order(n)
    work = t.full((npad, npad), 77, dtype=src.dtype, device=src.device)
    closed, side, s = dense._rows_closure(src, work, n, npad, dense.status(), None)
    side = side if closed else None
    return side, work[:n, :n].cpu().numpy(), s


def _full(A):
    W, out = dense.fw_closure(_lib.to_device(A), elem_type(A.dtype), schedule="full")
    return W.cpu().numpy(), out


def _slots(n):
    return max(8, min(n // 12, 24), min(n // 40, 200))


def _with_extra_entries(n, per_row, dt, seed):
    """A lower triangular matrix with ``per_row`` entries in every row that has
    room for them, values 2..5, and few levels: entries lie in the first half."""
    rng = np.random.default_rng(seed)
    A = np.zeros((n, n), dtype=dt)
    A[np.arange(n), np.arange(n)] = rng.choice([-1, 0, 1], n)
    for i in range(n // 2, n):
        A[i, rng.choice(n // 2, per_row, replace=False)] = rng.integers(2, 6, per_row)
    for i in range(1, n // 2):
        A[i, rng.integers(0, max(1, i // 2))] = 2
    return A


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("n,lda", [(1, None), (2, None), (17, None), (31, 33), (32, 32), (33, 36), (129, None),
                                   (300, 301), (513, 516), (1100, None)])
def test_rows_closure_vs_oracle(orc, dt, n, lda):
    A = synth.dense_pedigree(synth.PedigreeSpec(n, min(n, 12), 0.8, 3), 3 + n, dtype=dt)
    if n > 20:
        A[7, 7] = 0  # a vertex without a colour
    closed, W, s = _rows(A, lda)
    ref = orc.warshall(A)
    assert closed == "lower" and s.flags == 0 and s.events == 0 and s.cycle_count == 0
    np.testing.assert_array_equal(W, ref.W)
    Wf, out = _full(A)
    np.testing.assert_array_equal(W, Wf)
    assert s.diameter_max == out.status.diameter_max
    assert dense.msb(s.diameter_max) == ref.diameter


@pytest.mark.parametrize("dt,n", [(np.int32, 256), (np.int32, 1500), (np.int64, 640)])
def test_rows_closure_slot_limit(dt, n):
    """Rows with as many entries as there are slots are closed here, one more
    sends the matrix to the blocked schedules; the results are the same."""
    full = _with_extra_entries(n, _slots(n), dt, 1)
    closed, W, s = _rows(full)
    Wf, out = _full(full)
    assert closed == "lower" and s.diameter_max == out.status.diameter_max
    np.testing.assert_array_equal(W, Wf)
    over = _with_extra_entries(n, _slots(n) + 1, dt, 1)
    closed, W, _ = _rows(over)
    assert closed is None and (W == 77).all()
    W2, out2 = dense.fw_closure(_lib.to_device(over), elem_type(dt))
    Wf, outf = _full(over)
    assert out2.schedule == "lower" and out2.status.diameter_max == outf.status.diameter_max
    np.testing.assert_array_equal(W2.cpu().numpy(), Wf)


def _chain(n, dt):
    A = np.diag(np.full(n, -1, dtype=dt))
    A[np.arange(1, n), np.arange(n - 1)] = 2
    return A


def _shortcut_chain(n, dt):
    """A chain whose every row also names vertex i - 2, i - 4, ...: n levels,
    values that stay small."""
    A = _chain(n, dt)
    for i in range(n):
        for q in range(1, 7):
            if i - (1 << q) >= 0:
                A[i, i - (1 << q)] = 2
    return A


def test_rows_closure_level_limit():
    for n, closed_ref in ((63, "lower"), (64, "lower"), (65, None)):
        A = _shortcut_chain(n, np.int64)
        closed, W, s = _rows(A)
        assert closed == closed_ref
        Wf, out = _full(A)
        W2, out2 = dense.fw_closure(_lib.to_device(A), elem_type(np.int64))
        np.testing.assert_array_equal(W2.cpu().numpy(), Wf)
        assert out2.status.diameter_max == out.status.diameter_max and out2.schedule == "lower"


@pytest.mark.parametrize("dt,bits", [(np.int32, 32), (np.int64, 64)])
def test_rows_closure_overflow_guard(dt, bits):
    """The longest chain whose values fit is closed; one vertex more overflows
    and comes out of general mode with its events."""
    fits, over = _chain(bits - 1, dt), _chain(bits, dt)
    closed, W, s = _rows(fits)
    Wf, out = _full(fits)
    assert closed == "lower" and s.flags == 0
    np.testing.assert_array_equal(W, Wf)
    closed, _, s = _rows(over)
    assert s.flags & _lib.F_NEED_GENERAL
    W2, out2 = dense.fw_closure(_lib.to_device(over), elem_type(dt))
    Wf, outf = _full(over)
    assert out2.mode == outf.mode == "general" and out2.status.events == outf.status.events != 0
    np.testing.assert_array_equal(W2.cpu().numpy(), Wf)


@pytest.mark.parametrize("i,j,v", [(40, 3, 1), (40, 3, -1), (40, 3, -5), (40, 40, 2), (40, 40, -3)])
def test_rows_closure_declines_values(i, j, v):
    A = synth.dense_pedigree(synth.PedigreeSpec(70, 6, 0.8, 3), 1)
    A[i, j] = v
    closed, W, s = _rows(A)
    assert closed is None and s.flags & _lib.F_PRECOND_FAIL and (W == 77).all()


@pytest.mark.parametrize("dt,n,layers,lookback,seed", [
    (np.int32, 5, 3, 1, 1), (np.int32, 130, 7, 3, 1), (np.int32, 150, 12, 3, 1), (np.int32, 300, 9, 1, 0),
    (np.int64, 700, 18, 2, 1), (np.int32, 700, 18, 4, 1), (np.int64, 513, 30, 3, 2), (np.int32, 1100, 11, 4, 0)])
@pytest.mark.parametrize("numbering", ["upper", "any"])
def test_rows_closure_any_numbering_vs_oracle(orc, dt, n, layers, lookback, seed, numbering):
    """Upper triangular and shuffled pedigrees: W, and the exact largest value
    the naive loop's cells ever held (pedigrees with several paths between two
    vertices, where it depends on the numbering)."""
    A = synth.dense_pedigree(synth.PedigreeSpec(n, layers, 0.8, lookback), seed, dtype=dt)
    A = synth.reverse_vertices(A) if numbering == "upper" else synth.shuffle_vertices(A, seed)
    side, W, s = _rows(A)
    assert side == ("upper" if not np.tril(A, -1).any() else "full") and s.flags == 0
    ref = orc.warshall(A)
    np.testing.assert_array_equal(W, ref.W)
    Wf, out = _full(A)
    assert s.diameter_max == out.status.diameter_max and dense.msb(s.diameter_max) == ref.diameter


def _detour(n, long, dt):
    """Two paths from the last vertex but one to vertex 0: ``long`` edges
    through low numbers, found first, and two edges through the last vertex;
    the other vertices stand alone."""
    A = np.diag(np.full(n, -1, dtype=dt))
    walk = [n - 2] + list(range(long - 1, 0, -1)) + [0]
    for a, b in zip(walk[:-1], walk[1:]):
        A[a, b] = 2
    A[n - 2, n - 1] = 2
    A[n - 1, 0] = 2
    return A


@pytest.mark.parametrize("dt,n,long", [(np.int32, 20, 6), (np.int32, 300, 20), (np.int64, 300, 40)])
def test_rows_closure_any_first_value_above_final(orc, dt, n, long):
    """A cell whose first value is the largest ever held and not its last."""
    A = _detour(n, long, dt)
    side, W, s = _rows(A)
    ref = orc.warshall(A)
    assert side == "full" and s.diameter_max == 1 << long > W.max()
    np.testing.assert_array_equal(W, ref.W)
    assert dense.msb(s.diameter_max) == ref.diameter == long


@pytest.mark.parametrize("dt", [np.int32, np.int64])
def test_rows_closure_any_random_acyclic(orc, dt):
    """Random acyclic matrices, several paths between most vertices, in random
    numberings."""
    for seed in range(24):
        rng = np.random.default_rng(seed)
        n = int(rng.integers(9, 60))
        A = np.tril((rng.random((n, n)) < 0.12) * rng.integers(2, 6, (n, n)), -1).astype(dt)
        A[np.arange(n), np.arange(n)] = rng.choice([-1, 1], n)
        A = synth.shuffle_vertices(A, seed)
        side, W, s = _rows(A)
        if side is None:  # more entries in a row than slots, or values past the guard
            continue
        np.testing.assert_array_equal(W, orc.warshall(A).W)
        assert s.diameter_max == _full(A)[1].status.diameter_max


def test_rows_closure_declines_cycles():
    A = synth.dense_pedigree(synth.PedigreeSpec(140, 7, 0.8, 3), 1)
    kid = int(np.nonzero(A[139, :139])[0][0])
    A[kid, 139] = 2
    side, _, s = _rows(A)
    assert side is None
    W2, out2 = dense.fw_closure(_lib.to_device(A), elem_type(np.int32))
    Wf, outf = _full(A)
    assert out2.mode == outf.mode == "general"
    assert out2.status.cycle_last_key == outf.status.cycle_last_key


@pytest.mark.parametrize("what", ["workspace", "second matrix"])
@pytest.mark.parametrize("numbering", ["lower", "any"])
def test_closure_without_room_for_the_rows(monkeypatch, what, numbering):
    """Where the rows' workspace or the second matrix does not fit the memory
    the blocked schedules close the matrix, as they did before."""
    t = _lib.torch()
    n = 700
    A = synth.dense_pedigree(synth.PedigreeSpec(n, 10, 0.8, 2), 5)
    if numbering == "any":
        A = synth.shuffle_vertices(A, 3)
    et = elem_type(np.int32)
    Ad = _lib.to_device(A)
    want, full = dense.fw_closure(Ad, et, schedule="full")
    size = int(_lib.load().rbg_fw_rows_workspace_bytes(n, 4))
    empty, like = t.empty, t.empty_like
    refused = []

    def no_room(shape, *args, **kw):
        if what == "workspace" and shape == size and kw.get("dtype") == t.uint8:
            refused.append(shape)
            raise t.OutOfMemoryError("no room")
        return empty(shape, *args, **kw)

    def no_second(x, *args, **kw):
        if what == "second matrix":
            refused.append(tuple(x.shape))
            raise t.OutOfMemoryError("no room")
        return like(x, *args, **kw)

    dense._tls.__dict__.pop("rows_cache", None)
    monkeypatch.setattr(t, "empty", no_room)
    monkeypatch.setattr(t, "empty_like", no_second)
    W, out = dense.fw_closure(Ad, et)
    monkeypatch.undo()
    assert t.equal(W, want) and (out.mode, out.diameter) == (full.mode, full.diameter)
    assert bool(refused) == (what == "workspace" or numbering == "any")
    assert out.schedule == ("lower" if numbering == "lower" else "full")


def _closed(A):
    """(closed from the rows or not, W) of the rows' launches alone, and the
    whole closure against the full schedule's."""
    t = _lib.torch()
    et = elem_type(A.dtype)
    n, npad = len(A), dense.padded_order(len(A))
    Ad = _lib.to_device(A)
    work = t.empty((npad, npad), dtype=Ad.dtype, device=Ad.device)
    closed, sched, st = dense._rows_closure(Ad, work, n, npad, dense.status(), None)
    want, full = dense.fw_closure(Ad, et, schedule="full")
    got, out = dense.fw_closure(Ad, et)
    assert t.equal(got, want) and (out.mode, out.diameter) == (full.mode, full.diameter)
    if closed:
        assert t.equal(work[:n, :n], want) and int(st.diameter_max) == int(out.status.diameter_max)
    return closed


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("many,closed", [(4096, True), (4097, False), (6000, False)])
def test_rows_closure_cells_above_the_largest_value(dt, many, closed):
    """A chain of ten, and vertices that reach its head both at once and by
    the whole chain: the longer way's value is above every final one, a cell
    for each; up to 4,096 such cells have their first values looked up."""
    m = 10
    n = m + 1 + many
    A = np.zeros((n, n), dtype=dt)
    i = np.arange(1, m + 1)
    A[i, i - 1] = 3
    A[m + 1:, m] = 3
    A[m + 1:, 0] = 2
    A[np.arange(n), np.arange(n)] = 1
    assert _closed(synth.shuffle_vertices(A, 1)) == closed


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("depth,closed", [(8, True), (9, True), (10, False)])
def test_rows_closure_vertices_between(dt, depth, closed):
    """A vertex that reaches another at once and through a binary tree: up to
    1,024 vertices between the two are looked through for the first value."""
    tree = 2 ** (depth + 1) - 1  # vertex 0 its root
    leaf, j = tree, tree + 1
    A = np.zeros((tree + 2, tree + 2), dtype=dt)
    v = np.arange(2 ** depth - 1)
    A[v, 2 * v + 1] = 2
    A[v, 2 * v + 2] = 3
    A[2 ** depth - 1:tree, leaf] = 2
    A[leaf, j] = 3
    A[0, j] = 2
    A[np.arange(tree + 2), np.arange(tree + 2)] = -1
    assert (tree - 1 + 1 <= 1024) == closed
    assert _closed(synth.shuffle_vertices(A, 2)) == closed


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("n,layers,lookback", [(40, 5, 1), (100, 7, 3), (700, 10, 2), (1500, 24, 4), (3000, 12, 1)])
def test_rows_closure_takes_pedigrees(dt, n, layers, lookback):
    """Pedigrees are closed from their rows in every numbering."""
    A = synth.dense_pedigree(synth.PedigreeSpec(n, layers, 0.8, lookback), n, dtype=dt)
    for M in (A, synth.reverse_vertices(A), synth.shuffle_vertices(A, 1), synth.shuffle_vertices(A, 2)):
        assert _closed(M)


@pytest.mark.parametrize("dt", [np.int32, np.int64])
@pytest.mark.parametrize("n,layers,entries,tried", [(1200, 6, 8, True), (1200, 14, 12, False), (300, 6, 10, True),
                                                    (300, 20, 12, False)])
def test_rows_closure_of_many_paths(monkeypatch, dt, n, layers, entries, tried):
    """Rows of many entries: with few levels closed from them in every
    numbering, with many only where it is lower triangular, and then the passes
    for the other numberings are not run in vain."""
    rng = np.random.default_rng(n)
    bounds = np.linspace(0, n, layers + 1).astype(int)
    A = np.zeros((n, n), dtype=dt)
    for lo, hi in zip(bounds[1:-1], bounds[2:]):
        for i in range(lo, hi):
            A[i, rng.integers(0, lo, entries)] = rng.integers(2, 4, entries)
    A[np.arange(n), np.arange(n)] = -1
    assert _closed(A)
    said, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda fn, *args: (said.append(fn), call(fn, *args))[1])
    assert _closed(synth.shuffle_vertices(A, 3)) == _closed(synth.reverse_vertices(A)) == tried
    assert any(fn.startswith("rbg_fw_rows_any") for fn in said) == tried
