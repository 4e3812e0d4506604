"""GPU tests of the MFMA GEMMs by row count: the weight-streaming kernel of few
rows, at the edges of its 16-row tiles and of its column tiles, and with K
that is not a whole 128-byte unit or leaves some of a workgroup's waves
without one; and every tile of the 4-wave and 8-wave kernels and the K split, each
checked to be the one the dispatch takes.

Against float64 on the same inputs: an f32 sum of K products in any order is
within K 2^-24 sum |a| |b| of the exact one.  A 16-bit output adds half an ulp:
BF16 has 8 significant bits and F16 has 11, so that is at most 2^-8 and 2^-11 of
the value (just above a power of two), and 2^-25 below F16's normal range.  The fused
epilogues and the int8 GEMM are held bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hip():
    from vibe_compiler_amd import backend

    ctx = backend.Context(0)
    yield ctx
    ctx.close()


@pytest.fixture(scope="module")
def B():
    from vibe_compiler_amd import backend

    return backend


def _check(got, a, b, half_ulp):
    """got [m, n] against a [m, k] . b [n, k]^T in float64, element by element."""
    a, b = a.double(), b.double()
    ref, mag = a @ b.t(), a.abs() @ b.abs().t()
    bound = a.shape[1] * 2.0 ** -24 * mag
    bound = bound + half_ulp * (ref.abs() + bound) + (2.0 ** -25 if half_ulp else 0.0)
    over = (got.double() - ref).abs() - bound
    assert float(over.max()) <= 0, float(over.max())


ROWS = [(1, 128, 4096, 3), (15, 130, 96, 2), (16, 16, 32, 3), (17, 4096, 160, 3), (31, 33, 8192, 2), (32, 8192, 96, 3),
        (33, 1000, 544, 2), (48, 10272, 64, 3), (63, 20, 2080, 3), (64, 12288, 128, 2), (64, 640, 1024, 3)]
# few outputs of more rows (64 x 32 tiles, SwiGLU 64 x 64), and more of them with
# n of every alignment
TILES = [(200, 4100, 128, 3), (65, 64, 128, 3), (127, 72, 256, 2), (100, 16400, 128, 3), (129, 130, 192, 2), (300, 4100, 128, 3),
         (300, 6145, 256, 2), (1000, 6148, 128, 3), (300, 28648, 64, 2), (300, 28656, 128, 3), (130, 60, 256, 3),
         (1000, 500, 96, 2), (120, 4096, 2080, 3)]


# every kernel and tile of more rows, by its route (kernel, tile rows, tile
# columns, splits; test_dispatch.py): whole grids, and grids whose last row,
# column or both the tile does not divide, BF16 and F16 in turn
TILE4, WAVE8, SPLIT = 1, 2, 3
ROUTES = [
    (64, 64, TILE4, (65, 4100, 64), (65, 4160, 192), (128, 4100, 64), (200, 4096, 4096)),
    (64, 128, TILE4, (65, 8200, 128), (320, 6144, 64), (65, 11008, 64), (192, 8200, 64)),
    (128, 64, TILE4, (129, 6148, 64), (256, 4160, 64), (129, 6144, 128), (128, 8200, 64)),
    (128, 128, TILE4, (200, 8200, 64), (384, 6144, 192), (129, 11008, 64), (256, 8200, 64), (700, 4100, 2048)),
    (128, 192, TILE4, (257, 11008, 64), (384, 12288, 64), (257, 12288, 128), (512, 8200, 64), (700, 6148, 4096)),
    (256, 256, TILE4, (16448, 320, 64), (768, 8192, 64), (1024, 6148, 128), (1000, 6145, 64)),
    # 8 waves: long K, 64-byte K stages, and products narrower than every tile
    (128, 128, WAVE8, (384, 6144, 12288), (129, 11008, 4096), (256, 8200, 4096), (700, 4100, 14336), (16448, 32, 64),
     (65, 4100, 32), (384, 1536, 96), (129, 3072, 4128), (128, 4100, 32), (1024, 4096, 96)),
    (256, 256, WAVE8, (1024, 12288, 32), (1024, 12288, 96)),
    (256, 256, SPLIT, (768, 1536, 10240), (512, 4096, 14336), (768, 3072, 8192)),
]
ROUTED = [(*s, 3 if (i + s[0]) % 2 else 2, (kernel, bm, bn)) for bm, bn, kernel, *shapes in ROUTES
          for i, s in enumerate(shapes)]
# the same of SwiGLU products (n features)
SWIGLU_ROUTES = [
    (64, 128, TILE4, (400, 2080, 64), (320, 3072, 64), (65, 5504, 128)),
    (128, 64, TILE4, (256, 2080, 64), (129, 3072, 64)),
    (128, 128, TILE4, (500, 2080, 64), (384, 3072, 64), (129, 5504, 64), (512, 2080, 128), (129, 5504, 12352)),
    (128, 192, TILE4, (257, 5504, 64), (384, 6144, 64), (257, 6144, 128), (384, 5504, 64)),
    (256, 224, TILE4, (512, 7168, 64), (512, 7168, 192)),
    (256, 256, TILE4, (768, 4096, 64), (1536, 2080, 64), (777, 5520, 128)),
    (256, 256, WAVE8, (768, 4096, 192), (1536, 2080, 192), (777, 5520, 320), (768, 768, 32), (65, 5504, 96),
     (256, 2080, 32)),
]
SWIGLU_ROUTED = [(*s, 3 if (i + s[0]) % 2 else 2, (kernel, bm, bn)) for bm, bn, kernel, *shapes in SWIGLU_ROUTES
                 for i, s in enumerate(shapes)]


def _route(B, m, n, k, swiglu=False):
    import ctypes

    r = (ctypes.c_int * 4)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    B.load().wafer_internal_gemm_route(0, 3 if swiglu else 1, m, n, 2 * k, cus, 0, r)
    return tuple(r)[:3]


@pytest.mark.parametrize("m,n,k,fmt", ROWS + TILES)
def test_gemm_rows_vs_float64(hip, B, m, n, k, fmt):
    print("[gemm rows]", m, n, k, fmt, flush=True)
    _rows(hip, B, m, n, k, fmt)


@pytest.mark.parametrize("m,n,k,fmt,route", ROUTED)
def test_gemm_routes_vs_float64(hip, B, m, n, k, fmt, route):
    print("[gemm route]", m, n, k, fmt, route, flush=True)
    assert _route(B, m, n, k) == route
    split = route[0] == SPLIT
    _rows(hip, B, m, n, k, fmt, swiglu=False, shifts=(0,) if split else (0, 1))


@pytest.mark.parametrize("m,n,k,fmt,route", SWIGLU_ROUTED)
def test_swiglu_routes_vs_plain(hip, B, m, n, k, fmt, route):
    print("[swiglu route]", m, n, k, fmt, route, flush=True)
    assert _route(B, m, 2 * n, k, swiglu=True) == route
    dt = torch.bfloat16 if fmt == B.BF16 else torch.float16
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + k)
    _swiglu(hip, B, (torch.randn(m, k, generator=g, device="cuda")).to(dt),
            (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dt), g, m, n, k, fmt)


def _rows(hip, B, m, n, k, fmt, swiglu=True, shifts=(0, 1)):
    dt, half_ulp = (torch.bfloat16, 2.0 ** -8) if fmt == B.BF16 else (torch.float16, 2.0 ** -11)
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + k)
    a = torch.randn(m, k, generator=g, device="cuda").to(dt)
    b = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dt)
    out = torch.full((m * n + 512,), 7.5, device="cuda")
    hip.gemm_mfma(a, b, out, m, k, n, in_fmt=fmt, out_fmt=B.F32, rhs_t=True)
    _check(out[:m * n].view(m, n), a, b, 0.0)
    assert torch.all(out[m * n:] == 7.5)
    # an output that no vector store is aligned for
    for shift in shifts:
        outn = torch.full((m * n + 512,), 7.5, dtype=dt, device="cuda")
        view = outn[shift:shift + m * n]
        hip.gemm_mfma(a, b, view, m, k, n, in_fmt=fmt, out_fmt=fmt, rhs_t=True)
        _check(view.view(m, n), a, b, half_ulp)
        assert torch.all(outn[:shift] == 7.5) and torch.all(outn[shift + m * n:] == 7.5)
    # the narrowed product plus a residual, in place, is the Add command's sum
    r = torch.randn(m, n, generator=g, device="cuda").to(dt)
    ref = torch.empty_like(r)
    hip.elementwise("Add", fmt, view.clone().view(m, n), ref, r)
    hip.gemm_mfma_residual(a, b, r, r, m, k, n, in_fmt=fmt, rhs_t=True)
    assert torch.equal(r.view(torch.int16), ref.view(torch.int16))
    if swiglu and n % 16 == 0:
        _swiglu(hip, B, a, b, g, m, n, k, fmt)


def _swiglu(hip, B, a, b, g, m, n, k, fmt):
    """The SwiGLU of n features (gate weights b) is the two narrowed products and the region, bit for bit."""
    wu = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(a.dtype)
    gate, up, ref, got = (torch.empty(m, n, dtype=a.dtype, device="cuda") for _ in range(4))
    hip.gemm_mfma(a, b, gate, m, k, n, in_fmt=fmt, out_fmt=fmt, rhs_t=True)
    hip.gemm_mfma(a, wu, up, m, k, n, in_fmt=fmt, out_fmt=fmt, rhs_t=True)
    hip.silu_mul(gate, up, ref, fmt=fmt)
    packed = torch.empty(2 * n, k, dtype=a.dtype, device="cuda")
    hip.interleave_gate_up(b, wu, packed)
    hip.gemm_mfma_swiglu(a, packed, got, m, k, n, in_fmt=fmt)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(1, 100, 64), (16, 4096, 1024), (33, 1001, 4160), (64, 12288, 192),
                                   (65, 100, 256), (300, 1000, 1024), (301, 4103, 128), (777, 6151, 128),
                                   # 4-wave tiles 64x64, 64x128, 128x64, 128x128, 128x192 and the 8-wave kernel
                                   # (64-byte stages, a short K, whole 256x256)
                                   (65, 4100, 128), (192, 8200, 128), (129, 6148, 128), (384, 6144, 2048),
                                   (200, 8200, 128), (512, 8200, 128), (257, 12288, 128), (300, 4103, 4160),
                                   (1024, 4096, 192), (384, 6144, 128), (1024, 12288, 64), (1024, 12288, 128)])
@pytest.mark.parametrize("rt", [False, True])
def test_gemm_i8_rows_bit_exact(hip, B, m, n, k, rt):
    print("[gemm i8 rows]", m, n, k, rt, flush=True)
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    b = rng.integers(-127, 128, (n, k)).astype(np.int8)
    scale = rng.uniform(0.001, 0.01, n).astype(np.float32)
    acc_ref = a.astype(np.int64) @ b.astype(np.int64).T
    y = torch.zeros(m * n + 64, dtype=torch.bfloat16, device="cuda")
    acc = torch.zeros(m * n + 64, dtype=torch.int32, device="cuda")
    rhs = b if rt else np.ascontiguousarray(b.T)
    hip.gemm_i8(torch.from_numpy(a).cuda(), torch.from_numpy(rhs).cuda(), torch.from_numpy(scale).cuda(), y, m, k, n,
                acc_out=acc, rhs_t=rt)
    assert np.array_equal(acc[:m * n].view(m, n).cpu().numpy(), acc_ref)
    yref = torch.from_numpy(acc_ref.astype(np.float32) * scale).to(torch.bfloat16)
    assert torch.equal(y[:m * n].view(m, n).cpu(), yref)
    hip.gemm_i8(torch.from_numpy(a).cuda(), torch.from_numpy(rhs).cuda(), torch.from_numpy(scale).cuda(), y.zero_(), m, k,
                n, rhs_t=rt)  # without the accumulators: the staged stores
    assert torch.equal(y[:m * n].view(m, n).cpu(), yref)
    assert torch.all(acc[m * n:] == 0) and torch.all(y[m * n:] == 0)


@pytest.mark.parametrize("m,k,n,batch,fmt,lt", [
    (1, 40, 57400, 1, 5, 0), (2, 5, 65000, 1, 5, 1), (3, 1000, 1000, 1, 3, 0), (9, 17, 130, 1, 2, 1), (16, 300, 700, 1, 2, 0),
    (130, 512, 2000, 1, 5, 0), (127, 31, 2001, 1, 5, 1), (300, 80, 1500, 1, 5, 1), (129, 63, 1030, 1, 3, 1),
    (257, 33, 2047, 1, 2, 0), (65, 15, 64, 120, 5, 0), (5, 48, 100, 300, 3, 1)])
def test_formal_gemm_rows_bit_exact(hip, B, oracle, m, k, n, batch, fmt, lt):
    """The formal GEMM's register chains at the edges of their row tiles, 64
    columns and 16-k chunks (fewer k than one chunk, a partial last one), with
    zeros of both signs, an infinity and a NaN among the operands, a partial sum
    and both lhs orientations, bit for bit against the oracle."""
    print("[formal rows]", m, k, n, batch, fmt, lt, flush=True)
    rng = np.random.default_rng(m + 3 * k + n)
    a = rng.standard_normal((batch, m, k)).astype(np.float32)
    b = rng.standard_normal((batch, k, n)).astype(np.float32)
    a[:, 0] = -0.0
    b[:, :, -1] = 0.0
    b[:, :, 0] = np.inf
    b[0, k // 2, n // 2] = np.nan
    psum = rng.standard_normal((batch, m, n)).astype(np.float32)
    store = {5: lambda x: x, 3: lambda x: oracle.f32_to_bf16(x).reshape(x.shape),
             2: lambda x: x.astype(np.float16).view(np.uint16)}[fmt]
    ah, bh = store(a), store(b)
    al = np.ascontiguousarray(ah.transpose(0, 2, 1)) if lt else ah
    ref = oracle.gemm_formal(fmt, fmt, al, bh, m, k, n, batch=batch, psum=psum, lhs_t=bool(lt))
    dev = lambda x: torch.from_numpy(x.view(np.int16) if x.dtype == np.uint16 else x).cuda()  # noqa: E731
    out = torch.zeros(batch * m * n + 64, dtype=torch.float32 if fmt == 5 else torch.int16, device="cuda")
    hip.gemm(dev(al), dev(bh), out, m, k, n, batch=batch, in_fmt=fmt, out_fmt=fmt, psum=dev(psum), lhs_t=bool(lt))
    got = out.cpu().numpy()
    assert np.array_equal(got[:-64].view(np.uint32 if fmt == 5 else np.uint16), ref.ravel().view(np.uint32 if fmt == 5 else np.uint16))
    assert not got[-64:].any()
