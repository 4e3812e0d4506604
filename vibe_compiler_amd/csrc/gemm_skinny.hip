// gemm_skinny.hip -- MFMA GEMMs of few rows (decode steps, short prompts):
// y [m, n] = a [m, K] . bt [n, K]^T with m at most 64, or few outputs, bf16 / f16
// (f32 accumulate) and int8 (exact int32 accumulate).
//
// What bounds it is the weight bt, read once from HBM, and then the
// activations, which every workgroup reads again from L2.  The tile kernels
// of gemm_mfma.hip compute 128 or 256 rows whatever m is and leave most CUs
// idle (n 4096: 32 workgroups, each walking all of K behind stage barriers).
// Here a workgroup of 4 waves takes 16 NT columns of the output and all m
// rows, and its waves take K in turn (unit u, 128 bytes of every row, to wave
// u % 4).  Each wave keeps a ring of D units of its own in LDS, filled by
// buffer_load ... lds D - 1 units ahead, and waits on its own vmcnt only: no
// barrier until the waves' partial sums meet in LDS and are added in wave
// order.  The LDS pass is what makes the loads whole 128-byte row pieces: in
// the MFMA operand layout 16 consecutive lanes hold 16 rows, and loading that
// straight into VGPRs ran at about 6.3 TB/s for weights and activations
// together, whether they came from HBM or from L2 (m 16, the 4096 -> 28672
// gate/up product: 58.5 us against 40.0).  The weights are the A operand, so a
// lane ends up with 4 consecutive output columns.
//
// Measured on one box, weights cold (us; the tile kernels before -> here; the
// weights alone take 7.9 / 5.2 / 36.7 / 18.4 us at 6.4 TB/s):
//   m    4096->6144     4096->4096     4096->28672 SwiGLU   14336->4096 + residual
//   1    30.0 -> 11.7   29.3 -> 8.2    108.4 -> 40.8        93.1 -> 22.0
//   16   30.4 -> 14.0   29.7 -> 9.3    108.7 -> 40.0        96.9 -> 25.8
//   64   33.1 -> 22.7   32.0 -> 13.3   113.4 -> 55.4        114.5 -> 40.5
// Non-temporal weight loads: 49.0 -> 46.5 us (gate/up) and 25.9 -> 22.0 us
// (14336->4096) at m 1.
//
// The order of the sum of one output depends on K alone (not on m, n, or the
// epilogue) for every product that this kernel serves, so the fused epilogues
// keep the bits of the unfused calls.  It is not the k order of the tile kernels:
// a row's bits differ between m 64 and 65 where n is large, and again where the
// few-output rule ends.
//
// More rows on few columns take the same kernel on tiles of 64 x 32 (SwiGLU: 64 x
// 64, the two products' columns), wherever those are one round of workgroups at
// most: twice the workgroups of 64 x 64 tiles and rings three units deep, so more
// bytes in flight on more CUs, and no stage barrier (64 x 64 tiles here were no
// faster than the tile kernel's).  Against that kernel (us): 128 x 4096, K 4096
// 21.0 -> 16.3; 128 x 4096 with residual, K 14336 74 -> 52; int8 300 x 1389, K
// 3520 21.8 -> 11.5; 256 x 2048, K 1024 6.9 -> 6.0.
//
// Rows past m, columns past n and K past its end read as zero (buffer range)
// and are not stored.
#include "gemm_common.h"

namespace wafer {
namespace {

constexpr int SKINNY_WAVES = 4;
constexpr int SKINNY_ROWS = 64;
constexpr int NON_TEMPORAL = 2;  // buffer load policy: the weights are read once

template <int KIND> struct Acc4 { typedef f32x4 T; };
template <> struct Acc4<KIND_I8> { typedef i32x4 T; };

template <int KIND>
__device__ inline typename Acc4<KIND>::T mfma16(u32x4 a, u32x4 b, typename Acc4<KIND>::T c) {
  if constexpr (KIND == KIND_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else if constexpr (KIND == KIND_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  else
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0,
                                                 0);
}

template <int KIND>
__device__ inline uint16_t narrow16(float v) {
  return KIND == KIND_F16 ? narrow_f16(v) : (uint16_t)bf16x2_rne(v, v);
}
template <int KIND>
__device__ inline float widen16(uint16_t h) {
  return KIND == KIND_F16 ? widen_f16(h) : bf16_to_f32(h);
}

template <int KIND, int OUT, int MT, int NT, int D>
__global__ __launch_bounds__(64 * SKINNY_WAVES) void gemm_nt_skinny_kernel(GemmArgs args) {
  typedef typename Acc4<KIND>::T acc_t;
  constexpr int W = SKINNY_WAVES, TILES = MT * NT;
  constexpr int PER = 2 * (MT + NT), SLOT = PER * 1024;  // DMA instructions and bytes per unit
  static_assert(OUT != OUT_SWIGLU || NT % 2 == 0, "a gate tile and its up tile");
  static_assert(W * TILES * 1024 <= W * D * SLOT, "the fold reuses the ring");
  static_assert((D - 1) * PER <= 63, "vmcnt counts every move in flight");
  __shared__ __align__(1024) uint8_t lds[W * D * SLOT];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * (16 * MT);
  const int kb = args.kbytes;
  const int units = (kb + 127) / 128, iters = (units + W - 1) / W;

  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(args.bt + (size_t)n0 * kb), 0, min(16 * NT, args.n - n0) * kb, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(args.a + (size_t)m0 * kb), 0, min(16 * MT, args.m - m0) * kb, 0x00020000);

  // One DMA instruction moves 8 rows x 128 bytes: lane l fills chunk position
  // l % 8 of row l / 8, so it loads the chunk that the swizzle (chunk ^ (row
  // >> 1) & 7, conflict-free fragment reads) puts there; the second
  // instruction of a 16-row tile has rows 8 .. 15 and its own swizzle.
  uint32_t voff[2];
  int chunk[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 8 * h + lane / 8;
    chunk[h] = ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    voff[h] = (uint32_t)(row * kb + chunk[h]);
  }
  uint8_t *const ring = lds + wv * (D * SLOT);
  // unit `u` of K (bytes 128 u .. +127 of every row) into ring slot `slot`;
  // chunks past K take an offset outside both ranges and read as zero
  auto issue = [&](int u, int slot) __attribute__((always_inline)) {
    uint8_t *const dst = ring + slot * SLOT;
    const int k0 = u * 128;
    uint32_t vo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) vo[h] = k0 + chunk[h] < kb ? voff[h] + (uint32_t)k0 : 0x80000000u;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int t = q / 2, h = q % 2;  // tiles 0 .. NT-1 weights, then activations
      const uint32_t v = vo[h] + (uint32_t)((t < NT ? t : t - NT) * 16 * kb);
      auto *const d = (__attribute__((address_space(3))) void *)(dst + q * 1024);
      if (t < NT)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, d, 16, v, 0, 0, NON_TEMPORAL);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, d, 16, v, 0, 0, 0);
    }
  };
  acc_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;

  // fragment of k-step s: row l16 of the tile, chunk 4 s + g
  int foff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) foff[s] = l16 * 128 + (((4 * s + g) ^ ((l16 >> 1) & 7)) << 4);

#pragma unroll
  for (int d = 0; d < D - 1; ++d) issue(wv + d * W, d);
  int slot = 0, fill = D - 1;
  for (int it = 0; it < iters; ++it) {
    // slot `fill` held the previous unit, whose fragments are in registers
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(wv + (it + D - 1) * W, fill);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * PER) : "memory");
    const uint8_t *const src = ring + slot * SLOT;
    u32x4 wf[2][NT], xf[2][MT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < NT; ++j) wf[s][j] = *(const u32x4 *)(src + j * 2048 + foff[s]);
#pragma unroll
      for (int i = 0; i < MT; ++i) xf[s][i] = *(const u32x4 *)(src + (NT + i) * 2048 + foff[s]);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma16<KIND>(wf[s][j], xf[s][i], acc[i][j]);
    fill = slot;
    slot = slot + 1 == D ? 0 : slot + 1;
  }
  // moves of units past the last still fly: drain before the ring is reused
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  acc_t(*const part)[TILES][64] = (acc_t(*)[TILES][64])lds;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) part[wv][i * NT + j][lane] = acc[i][j];
  __syncthreads();

  // the fold: lane (l16, g) of a tile holds row m0 + 16 i + l16, columns
  // n0 + 16 j + 4 g .. +3
  auto fold = [&](int tile, int ln) __attribute__((always_inline)) {
    acc_t s = part[0][tile][ln];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const acc_t p = part[w][tile][ln];
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] += p[r];
    }
    return s;
  };
  if constexpr (OUT == OUT_SWIGLU) {
    // tile pair (gate, up): features n0 / 2 + 4 g .. +3
    const int nf = args.n / 2;
    const bool vec = nf % 4 == 0 && ((uintptr_t)args.y & 7) == 0;
    for (int q = threadIdx.x; q < TILES / 2 * 64; q += 64 * W) {
      const int t = q >> 6, ln = q & 63;  // pair t: row tile t / (NT / 2), column tiles 2 (t % (NT / 2)), + 1
      const int row = m0 + 16 * (t / (NT / 2)) + (ln & 15), f0 = n0 / 2 + 16 * (t % (NT / 2)) + 4 * (ln >> 4);
      if (row >= args.m || f0 >= nf) continue;
      const acc_t gt = fold(2 * t, ln), up = fold(2 * t + 1, ln);
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = narrow16<KIND>(silu_mul_1(widen16<KIND>(narrow16<KIND>((float)gt[r])),
                                         widen16<KIND>(narrow16<KIND>((float)up[r]))));
      uint16_t *y = (uint16_t *)args.y + (size_t)row * nf + f0;
      if (vec) {
        const u32x2 v = {o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16)};
        *(u32x2 *)y = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (f0 + r < nf) y[r] = o[r];
      }
    }
  } else {
    const bool vec = args.n % 4 == 0 && ((uintptr_t)args.y & (OUT == OUT_F32 ? 15 : 7)) == 0 &&
                     (OUT != OUT_NARROW_RES || ((uintptr_t)args.res & 7) == 0);
    for (int q = threadIdx.x; q < TILES * 64; q += 64 * W) {
      const int t = q >> 6, ln = q & 63;
      const int row = m0 + 16 * (t / NT) + (ln & 15), col = n0 + 16 * (t % NT) + 4 * (ln >> 4);
      if (row >= args.m || col >= args.n) continue;
      const acc_t s = fold(t, ln);
      const size_t o = (size_t)row * args.n + col;
      const int cols = vec ? 4 : min(4, args.n - col);
      if constexpr (OUT == OUT_F32) {
        float *y = (float *)args.y + o;
        if (vec) {
          const f32x4 v = {(float)s[0], (float)s[1], (float)s[2], (float)s[3]};
          *(f32x4 *)y = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r < cols) y[r] = (float)s[r];
        }
      } else {
        uint16_t v[4];
        if constexpr (OUT == OUT_NARROW) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = narrow16<KIND>((float)s[r]);
        } else if constexpr (OUT == OUT_NARROW_RES) {
          uint16_t res[4] = {0, 0, 0, 0};
          if (vec) {
            const u32x2 rv = *(const u32x2 *)(args.res + o);
#pragma unroll
            for (int r = 0; r < 4; ++r) res[r] = (uint16_t)(rv[r >> 1] >> (16 * (r & 1)));
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (r < cols) res[r] = args.res[o + r];
          }
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = narrow16<KIND>(widen16<KIND>(narrow16<KIND>((float)s[r])) + widen16<KIND>(res[r]));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int32_t a32 = (int32_t)s[r];
            if (r < cols) {
              if (args.acc_out) args.acc_out[o + r] = a32;
              const float d = (float)a32 * args.scale[col + r];
              v[r] = (uint16_t)bf16x2_rne(d, d);
            }
          }
        }
        uint16_t *y = (uint16_t *)args.y + o;
        if (vec) {
          const u32x2 w = {v[0] | ((uint32_t)v[1] << 16), v[2] | ((uint32_t)v[3] << 16)};
          *(u32x2 *)y = w;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r < cols) y[r] = v[r];
        }
      }
    }
  }
}

// ring depth that keeps a workgroup's LDS at 80 KiB (two per CU) where two
// units at least fit: 5 units at most (one tile of each)
constexpr int ring_depth(int mt, int nt) {
  const int d = 80 / (SKINNY_WAVES * 2 * (mt + nt));
  return d < 2 ? 2 : d;
}

template <int KIND, int OUT, int MT, int NT, int D = ring_depth(MT, NT)>
int launch_cols(hipStream_t st, const GemmArgs &args) {
  hipLaunchKernelGGL((gemm_nt_skinny_kernel<KIND, OUT, MT, NT, D>),
                     dim3((unsigned)((args.n + 16 * NT - 1) / (16 * NT)), (unsigned)((args.m + 16 * MT - 1) / (16 * MT))),
                     dim3(64 * SKINNY_WAVES), 0, st, args);
  return launch_status("gemm_nt_skinny_kernel");
}

// Column tiles per workgroup: more of them read the activations fewer times,
// fewer of them give more workgroups.  Measured at K 4096 (us, NT 1 / 2 / 4):
// n 4096, m 16: 9.3 / 11.9 / 14.8; n 8192, m 16: 15.4 / 16.0 / 17.7, m 32:
// 18.5 / 16.5 / 19.7; n 12288, m 1: 18.9 / 23.7 / 19.0, m 16: 21.6 / 24.4 /
// 19.7 (two workgroups fit a CU: 384 of them make a second round three
// quarters empty), m 64: 34.3 / 31.9 / 26.9; n 16384, m 64: 44.6 / 35.6 / 28.8.
template <int KIND, int OUT, int MT>
int launch_rows(hipStream_t st, const GemmArgs &args, int cus) {
  const long tiles = (args.n + 15) / 16;
  if (2 * tiles >= 5L * cus) return launch_cols<KIND, OUT, MT, 4>(st, args);
  if (OUT == OUT_SWIGLU || (MT > 1 && 4 * tiles >= 7L * cus)) return launch_cols<KIND, OUT, MT, 2>(st, args);
  if constexpr (OUT != OUT_SWIGLU) return launch_cols<KIND, OUT, MT, 1>(st, args);
}

}  // namespace

bool gemm_is_skinny(int m, int n, int cus) {
  return m <= SKINNY_ROWS || (long)((m + 63) / 64) * ((n + 31) / 32) <= cus;
}

template <int KIND, int OUT>
int launch_gemm_skinny(hipStream_t st, GemmArgs args, int cus) {
  if (args.m > SKINNY_ROWS)
    return launch_cols<KIND, OUT, 4, OUT == OUT_SWIGLU ? 4 : 2, OUT == OUT_SWIGLU ? 2 : 3>(st, args);
  if (args.m <= 16) return launch_rows<KIND, OUT, 1>(st, args, cus);
  if (args.m <= 32) return launch_rows<KIND, OUT, 2>(st, args, cus);
  return launch_rows<KIND, OUT, 4>(st, args, cus);
}

#define SKINNY_INSTANCE(K, O) template int launch_gemm_skinny<K, O>(hipStream_t, GemmArgs, int);
SKINNY_INSTANCE(KIND_BF16, OUT_F32)
SKINNY_INSTANCE(KIND_BF16, OUT_NARROW)
SKINNY_INSTANCE(KIND_BF16, OUT_NARROW_RES)
SKINNY_INSTANCE(KIND_BF16, OUT_SWIGLU)
SKINNY_INSTANCE(KIND_F16, OUT_F32)
SKINNY_INSTANCE(KIND_F16, OUT_NARROW)
SKINNY_INSTANCE(KIND_F16, OUT_NARROW_RES)
SKINNY_INSTANCE(KIND_F16, OUT_SWIGLU)
SKINNY_INSTANCE(KIND_I8, OUT_I8_DEQUANT)

}  // namespace wafer
