"""Levels that mix long and short closure rows, against the oracle."""
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

