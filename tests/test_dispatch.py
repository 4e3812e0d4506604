"""CPU checks of the dispatch rules: which kernel a GEMM takes on a chip of 256
CUs, through the library's host-only test hooks (no GPU, no context)."""
import ctypes

import pytest

F16, BF16, F32 = 2, 3, 5
# operand kinds, epilogues and kernels of the MFMA GEMMs (gemm_common.h, gemm_mfma.hip)
K_BF16, K_F16, K_I8 = 0, 1, 2
OUT_F32, OUT_NARROW, OUT_I8, OUT_SWIGLU, OUT_RES = range(5)
STREAM, TILE4, WAVE8, SPLIT = range(4)


@pytest.fixture(scope="module")
def lib():
    from vibe_compiler_amd import backend

    return backend.load()


def gemm_route(lib, m, n, k, out=OUT_NARROW, kind=K_BF16, acc=False, cus=256):
    """(kernel, tile rows, tile columns, splits) of m x n outputs over k elements; n counts a SwiGLU's two products."""
    r = (ctypes.c_int * 4)()
    lib.wafer_internal_gemm_route(kind, out, m, n, k * (1 if kind == K_I8 else 2), cus, int(acc), r)
    return tuple(r)


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


@pytest.mark.parametrize("m,features,k,route", [
    (256, 5504, 14336, (TILE4, 128, 128, 1)), (2048, 1024, 14336, (TILE4, 128, 128, 1)),
    (128, 16384, 12288, (TILE4, 128, 128, 1)), (256, 16384, 14336, (TILE4, 128, 128, 1)),
    (300, 11008, 12288, (WAVE8, 256, 256, 1)), (777, 16384, 12288, (WAVE8, 256, 256, 1)),
    (512, 11008, 10240, (WAVE8, 256, 256, 1)), (777, 11008, 14336, (TILE4, 256, 256, 1)),
    (777, 14336, 4096, (TILE4, 256, 256, 1)), (1024, 14336, 4096, (TILE4, 256, 224, 1)),
    (1024, 14336, 14336, (TILE4, 256, 224, 1)), (16, 14336, 4096, (STREAM, 0, 0, 1))])
def test_swiglu_takes_the_tile_it_was_priced_on(lib, m, features, k, route):
    """Past K 12288 a SwiGLU product keeps the 128x128 tiles that its cost names
    (they went to the 8-wave kernel, which has 256x256 SwiGLU tiles only); 256x256
    tiles take the 8-wave kernel over rows of 3 or 5 times a power of two bytes."""
    for kind in (K_BF16, K_F16):
        assert gemm_route(lib, m, 2 * features, k, OUT_SWIGLU, kind) == route


@pytest.mark.parametrize("m,n,k,kernel", [
    (777, 4096, 2048, TILE4), (777, 4096, 4096, WAVE8), (200, 14336, 4096, WAVE8), (600, 4096, 4096, WAVE8),
    (1024, 4096, 4096, TILE4), (896, 4096, 12288, WAVE8), (900, 4096, 14336, WAVE8)])
@pytest.mark.parametrize("out", [OUT_F32, OUT_NARROW, OUT_RES])
def test_ragged_128_tiles_take_the_8_wave_kernel(lib, m, n, k, kernel, out):
    """128x128 tiles over 16-bit operands from K 4096 on: the 8-wave kernel where
    they do not divide the output, and from K 12288 on everywhere."""
    for kind in (K_BF16, K_F16):
        assert gemm_route(lib, m, n, k, out, kind) == (kernel, 128, 128, 1)
    if kernel == WAVE8 and k < 12288:
        assert gemm_route(lib, m, n, k, OUT_I8, K_I8)[0] == TILE4


@pytest.mark.parametrize("m,n,plain,acc", [
    (300, 4096, (TILE4, 128, 64), (TILE4, 128, 64)), (1024, 4096, (TILE4, 128, 128), (TILE4, 128, 128)),
    (512, 4096, (TILE4, 128, 64), (WAVE8, 128, 128)), (777, 4096, (TILE4, 128, 128), (WAVE8, 128, 128)),
    (4096, 1000, (TILE4, 128, 128), (WAVE8, 128, 128)), (1152, 4096, (TILE4, 128, 192), (WAVE8, 128, 128)),
    (256, 4096, (TILE4, 64, 64), (TILE4, 64, 64)), (777, 6144, (TILE4, 128, 192), (TILE4, 128, 192)), (4096, 4096, (WAVE8, 256, 256), (WAVE8, 256, 256))])
def test_int8_accumulators_keep_the_faster_kernel(lib, m, n, plain, acc):
    """An int8 product whose accumulators are asked for stores them element by
    element: shifted tiles, and 128x64 where whole 128x128 ones serve, are slower so."""
    assert gemm_route(lib, m, n, 4096, OUT_I8, K_I8)[:3] == plain
    assert gemm_route(lib, m, n, 4096, OUT_I8, K_I8, acc=True)[:3] == acc


def test_int8_128_tiles_over_a_short_k(lib):
    for k, kernel in ((512, WAVE8), (1024, WAVE8), (1152, TILE4), (4096, TILE4)):
        assert gemm_route(lib, 1024, 4096, k, OUT_I8, K_I8)[:3] == (kernel, 128, 128)


@pytest.mark.parametrize("fmt,group_size,rows,keys,chunks,group,fused", [
    (BF16, 1, 1024, 17, 16, 1, 0), (BF16, 1, 512, 300, 16, 1, 1), (F16, 1, 512, 2048, 16, 1, 0),
    (BF16, 4, 256, 1, 16, 1, 0), (F16, 1, 32, 4095, 16, 0, 1), (BF16, 8, 256, 1, 16, 0, 0), (BF16, 8, 256, 17, 1, 0, 1),
    (BF16, 8, 128, 17, 16, 0, 1), (BF16, 8, 128, 17, 32, 0, 0), (BF16, 8, 64, 8192, 16, 0, 1),
    (BF16, 8, 64, 8193, 16, 0, 0), (F16, 4, 256, 300, 16, 0, 1), (F16, 1, 1, (1 << 32) - 1, 16, 0, 0)])
def test_decode_append_rule(lib, fmt, group_size, rows, keys, chunks, group, fused):
    """A decode step's new rows are written by the decode kernel only where that
    beats a copy kernel before it: not over large caches or many workgroups."""
    u32 = ctypes.c_uint32
    assert lib.wafer_internal_append_in_kernel(u32(fmt), u32(group_size), u32(rows), u32(keys), u32(chunks), group,
                                               u32(256)) == fused
