"""The C ABI: librbg_hip.so loads and exports every symbol include/rbg_hip.h
declares, and the Python binding declares the same set.  CPU only (no
compute calls)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    syms = set()
    for name in sorted(os.listdir(os.path.join(ROOT, "include"))):
        if not name.endswith(".h"):
            continue
        text = open(os.path.join(ROOT, "include", name)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        syms |= set(re.findall(r"\b(rbg_\w+)\s*\(", text))
    return syms


def test_header_declares_functions():
    assert len(header_symbols()) >= 15


def test_library_exports_every_declared_symbol():
    from redblackgraph_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail("librbg_hip.so is not built (python -m redblackgraph_amd.build)")
    lib = ctypes.CDLL(_lib.LIB_PATH)
    missing = [s for s in sorted(header_symbols()) if not hasattr(lib, s)]
    assert not missing, missing


def test_binding_matches_header():
    from redblackgraph_amd import _lib
    assert set(_lib.SIGNATURES) == header_symbols()


def test_host_scalar_entry_points():
    import redblackgraph_amd as rb
    assert rb.avos_product(9223372036854775807, 2) == 18446744073709551614
    with pytest.raises(OverflowError):
        rb.avos_product(4294967296, 4294967296)
    with pytest.raises(OverflowError):
        rb.avos_product(9223372036854775807, 3)
    assert rb.avos_sum(-1, 1) == -1


@pytest.mark.parametrize("elem", [4, 8])
@pytest.mark.parametrize("M,K,N", [(1 << 22, 4, 4), (4, 1 << 22, 1), (1 << 20, 1, 16), (1000, 63, 70), (300, 300, 300)])
def test_matmul_rows_workspace_of_narrow_operands(elem, M, K, N):
    """No more room than the operands' own entries can take, but for what the
    arrays' starts are rounded up by."""
    from redblackgraph_amd import _lib
    need = _lib.load().rbg_matmul_rows_workspace_bytes(M, K, N, elem)
    assert need <= (4 + elem) * (M * K + K * N) + 4 * (M + K) + 2048 + 7 * 256


@pytest.mark.parametrize("elem", [4, 8])
def test_matmul_shapes_for_the_entries(elem):
    """Shapes measured: many short rows of C, or few very long ones, are the
    blocked kernels' whatever the operands hold; closures and their blocks, and
    short rows with many terms, are tried from the entries."""
    from redblackgraph_amd import _lib
    fits = _lib.load().rbg_matmul_rows_fits
    for shape in ((1 << 22, 4, 4), (1 << 20, 16, 16), (1 << 18, 64, 64), (1 << 17, 32, 32), (4, 4, 1 << 22),
                  (64, 64, 1 << 18)):
        assert fits(*shape, elem) == 0, shape
    for shape in ((300, 300, 300), (1000, 3000, 2000), (8192, 8192, 8192), (20_000, 2000, 20_000), (64, 1 << 18, 64),
                  (4096, 64, 64), (256, 4096, 4096), (1 << 16, 256, 256), (32_000, 32_000, 32_000)):
        assert fits(*shape, elem) == 1, shape


@pytest.mark.parametrize("sfx,elem", [("i32", 4), ("i64", 8)])
def test_rows_closure_refuses_a_row_stride_past_its_indices(sfx, elem):
    """The close pass counts 16-byte units of the matrix in 32 bits: a stride
    that carries n rows past them is an argument error, with no launch."""
    from redblackgraph_amd import _lib
    L = _lib.load()
    n = 32_640
    fake = 1 << 20  # never read: the arguments are refused
    room = int(L.rbg_fw_rows_workspace_bytes(n, elem))
    stride = (1 << 32) // n * (16 // elem) // 128 * 128
    over = stride + 256
    for npad in (over, 1 << 31):
        assert getattr(L, f"rbg_fw_rows_{sfx}")(fake, n, n, fake, npad, fake, room, fake, None) == -1
    over = (1 << 32) // 16_384 * (16 // elem) // 128 * 128 + 256
    assert getattr(L, f"rbg_fw_rows_any_{sfx}")(16_384, fake, fake, over, fake, room, fake, None) == -1
