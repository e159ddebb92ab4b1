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
