"""Batches whose components part ways: some closed from their rows' entries,
some too dense, too deep or not triangular, by every schedule, run eagerly and
as graph replays, against one matrix at a time."""
import numpy as np
import pytest

from redblackgraph_amd import _lib, dense, synth
from redblackgraph_amd._dtypes import elem_type
from redblackgraph_amd.batched import BatchedClosure

pytestmark = pytest.mark.gpu


def _pedigree(n, seed):
    return synth.dense_pedigree(synth.PedigreeSpec(n, max(2, int(np.ceil(np.log2(n))) if n > 2 else 2), 0.8, 1), seed)


def _dense_lower(n):
    """Every row has entries in the 30 columns before it: past the slots of a
    row, and deeper than the level limit where n > 64."""
    A = np.zeros((n, n), dtype=np.int32)
    for i in range(n):
        A[i, max(0, i - 30):i] = 2 + np.arange(i - max(0, i - 30)) % 2
        A[i, i] = 1 if i % 2 else -1
    return A


def _chain(n):
    """More levels than the rows' closure takes, two entries a row."""
    A = np.zeros((n, n), dtype=np.int32)
    i = np.arange(n)
    A[i, i] = -1
    A[i[1:], i[:-1]] = 2
    A[i[20:], i[:-20]] = 3
    return A


def _close(mats, tri, persistent):
    sizes = np.array([len(m) for m in mats])
    b = BatchedClosure(sizes, tri=tri, persistent=persistent)
    try:
        b.load_dense(mats)
        src = b.pool.clone()
        _lib.torch().cuda.synchronize()
        got, told = [], []
        for graph in (False, False, True, True, False):
            with _lib.torch().cuda.stream(b.stream):
                b.pool.copy_(src)
            b.run(graph=graph)
            b.stream.synchronize()
            told.append(b.rows_closed())
            got.append([b.result(i).cpu().numpy().copy() for i in range(len(mats))])
            outs = [(o.mode, o.diameter) for o in b.outcomes()]
            got[-1].append(outs)
        return got, told
    finally:
        b.close()


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("kind", ["closable", "mixed", "none"])
def test_batch_components_part_ways(kind, persistent):
    mats = {"closable": [_pedigree(n, 3 + n) for n in (1, 16, 127, 128, 129, 700, 1500)],
            "mixed": [_pedigree(300, 1), _dense_lower(200), _pedigree(64, 2), _chain(150), _pedigree(900, 4)],
            "none": [_dense_lower(130), _chain(140)]}[kind]
    mats = [np.tril(m) for m in mats]
    got, told = _close(mats, 1, persistent)
    want = [True] * len(mats) if kind == "closable" else None
    et = elem_type(np.int32)
    alone = [dense.fw_closure(_lib.to_device(m), et, schedule="steps") for m in mats]
    for run, t in zip(got, told):
        if want:
            assert list(t) == want
        if kind == "none":
            assert not t.any()
        for i in range(len(mats)):
            np.testing.assert_array_equal(run[i], alone[i][0].cpu().numpy())
            assert run[-1][i] == (alone[i][1].mode, alone[i][1].diameter)
    if kind == "mixed":
        assert told[0].any() and not told[0].all()


def _alone(mats):
    et = elem_type(np.int32)
    out = [dense.fw_closure(_lib.to_device(m), et, schedule="steps") for m in mats]
    return [w.cpu().numpy() for w, _ in out], [(o.mode, o.diameter) for _, o in out]


def _check(b, mats, want):
    b.stream.synchronize()
    assert [(o.mode, o.diameter) for o in b.outcomes()] == want[1]
    for i in range(len(mats)):
        np.testing.assert_array_equal(b.result(i).cpu().numpy(), want[0][i])


_INPUTS = {"closable": [_pedigree(200, 5), _pedigree(150, 6)], "mixed": [_pedigree(200, 7), _chain(150)],
           "none": [_dense_lower(200), _chain(150)]}
_INPUTS = {k: [np.tril(m) for m in v] for k, v in _INPUTS.items()}


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("graph", [False, True])
def test_batch_input_changes_between_runs(graph, persistent):
    """What one run found says nothing about the next one's input."""
    want = {k: _alone(v) for k, v in _INPUTS.items()}
    b = BatchedClosure([200, 150], tri=1, persistent=persistent)
    try:
        for kind in ("closable", "mixed", "closable", "none", "closable", "mixed", "mixed", "closable"):
            b.load_dense(_INPUTS[kind])
            b.run(graph=graph)
            _check(b, _INPUTS[kind], want[kind])
            np.testing.assert_array_equal(b.rows_closed(), {"closable": [1, 1], "mixed": [1, 0], "none": [0, 0]}[kind])
    finally:
        b.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("launches", [1, 2, 3])
def test_batch_recorded_by_its_caller(launches, graph):
    """A run recorded into the caller's own graph queues every launch, and what
    it found is not taken for the answer of a later direct run."""
    t = _lib.torch()
    want = {k: _alone(v) for k, v in _INPUTS.items()}
    b = BatchedClosure([200, 150], tri=1)
    try:
        outer = t.cuda.CUDAGraph()
        t.cuda.synchronize()
        with t.cuda.graph(outer, stream=b.stream):
            b.run(graph=False)
        for _ in range(launches):
            b.load_dense(_INPUTS["closable"])
            with t.cuda.stream(b.stream):
                outer.replay()
            _check(b, _INPUTS["closable"], want["closable"])
        for kind in ("none", "mixed", "closable", "none"):
            b.load_dense(_INPUTS[kind])
            b.run(graph=graph)
            _check(b, _INPUTS[kind], want[kind])
        b.load_dense(_INPUTS["mixed"])
        with t.cuda.stream(b.stream):
            outer.replay()
        _check(b, _INPUTS["mixed"], want["mixed"])
    finally:
        b.close()


@pytest.mark.parametrize("persistent", [False, True])
def test_rows_closed_names_the_callers_components(persistent):
    """Components in no order of size: the flags are in the caller's order."""
    mats = [_pedigree(60, 1), _dense_lower(200), _pedigree(900, 2), _chain(130), _pedigree(300, 3), _dense_lower(500),
            _pedigree(1500, 4), _chain(150)]
    mats = [np.tril(m) for m in mats]
    _, told = _close(mats, 1, persistent)
    for t in told:
        assert list(t) == [True, False, True, False, True, False, True, False]
