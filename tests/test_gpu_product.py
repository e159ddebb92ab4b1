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
