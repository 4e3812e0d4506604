"""CPU checks of the dispatch rules: which kernel a GEMM takes on a chip of 256
CUs, through the library's host-only test hooks (no GPU, no context)."""
import ctypes

import pytest

F16, BF16, F32 = 2, 3, 5


@pytest.fixture(scope="module")
def lib():
    from vibe_compiler_amd import backend

    return backend.load()


def formal_rows(lib, fmt, m, k, n, batch=1, lt=0, rt=0, cus=256):
    u32 = ctypes.c_uint32
    return lib.wafer_internal_formal_rows(u32(fmt), u32(m), u32(k), u32(n), u32(batch), lt, rt, u32(cus))


@pytest.mark.parametrize("fmt,m,k,n,batch,normal,transposed", [
    (F32, 128, 512, 8192, 1, 8, 0), (F32, 1000, 1024, 300, 1, 4, 0), (F32, 256, 1024, 300, 8, 8, 0),
    (F32, 32, 512, 8192, 8, 8, 8), (F32, 33, 512, 8192, 8, 8, 0), (F32, 16, 512, 2048, 8, 4, 4),
    (F32, 24, 512, 2048, 8, 4, 0), (F32, 2, 512, 8192, 8, 1, 1), (BF16, 256, 128, 2048, 1, 8, 0),
    (BF16, 256, 512, 2048, 1, 8, 8), (BF16, 32, 16, 8192, 1, 4, 4), (BF16, 33, 16, 8192, 1, 4, 0),
    (F16, 256, 16, 2048, 1, 8, 0), (F16, 256, 48, 2048, 1, 8, 8), (F16, 16, 700, 300, 1, 1, 1)])
def test_formal_rows_of_a_transposed_lhs(lib, fmt, m, k, n, batch, normal, transposed):
    """The register-chain kernel serves a transposed lhs only where it is the
    faster one: few rows, or 16 bits over a long k.  No transposed rhs."""
    assert formal_rows(lib, fmt, m, k, n, batch) == normal
    assert formal_rows(lib, fmt, m, k, n, batch, lt=1) == transposed
    assert formal_rows(lib, fmt, m, k, n, batch, rt=1) == formal_rows(lib, fmt, m, k, n, batch, lt=1, rt=1) == 0
