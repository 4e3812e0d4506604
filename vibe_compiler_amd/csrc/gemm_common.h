// gemm_common.h -- what the MFMA GEMM files share: operand kinds, epilogue
// selectors, the kernel arguments, and the f16 widening / narrowing of the
// epilogues.
#pragma once

#include "common.h"

namespace wafer {

enum { KIND_BF16 = 0, KIND_F16 = 1, KIND_I8 = 2 };

// Epilogue selectors.
// OUT_SWIGLU (bf16 or f16): the rhs rows come in 32-row groups, 16 gate rows
// then the 16 up rows of the same features, and y[m, f] =
// T(silu_mul(T(gate), T(up))) over N/2 features, T the storage format (the narrowed
// products, then the silu_mul region).  In a 32x32 MFMA tile the gate
// values of 16 features sit in lanes l32 < 16 and their up values in lanes
// l32 + 16; one v_permlane16_swap per register pair brings both to one
// lane (swiglu_pair).
// OUT_NARROW_RES: the narrowed product plus a residual tensor of the same
// format and shape, y = Add(narrow(acc), res) -- the GEMM's narrow output
// followed by the CT Add command, bit for bit (y may be res itself: every
// element is read before it is written, by the same lane).
enum { OUT_F32 = 0, OUT_NARROW = 1, OUT_I8_DEQUANT = 2, OUT_SWIGLU = 3, OUT_NARROW_RES = 4 };

// f32 -> f16 by v_cvt_f16_f32 in the default round-to-nearest-even mode, with
// gradual underflow and overflow to +-inf; a NaN narrows to the canonical
// 0x7e00 as f32_to_f16 does.
__device__ inline uint16_t narrow_f16(float x) {
  x = f32_rounded(x);
  return x != x ? (uint16_t)0x7e00u : __builtin_bit_cast(uint16_t, (_Float16)x);
}

struct GemmArgs {
  const uint8_t *a;    // [M, K] elements, K-contiguous
  const uint8_t *bt;   // [N, K] ([K, N] for the BKN int8 kernel)
  void *y;             // [M, N]
  int32_t *acc_out;    // int8 only, optional [M, N]
  const float *scale;  // int8 only, [N]
  int m, n, kbytes;    // K in bytes
  int tiles_m, tiles_n;  // ceil(M / BM), ceil(N / BN)
  const uint16_t *res;   // OUT_NARROW_RES only, [M, N]
  // split-K (4-wave kernel only): ksplit > 1 workgroups per tile each take
  // kbytes / ksplit of K and store f32 partial tiles to part [ksplit, M, N],
  // which a fold launch adds in split order
  int ksplit;
  float *part;
};

// GEMMs of few rows or few outputs (gemm_skinny.hip): true where the weight-
// streaming kernel serves a product of m x n (of one of the two products of a
// SwiGLU, so that it sums as the two plain calls do), and its launch.
bool gemm_is_skinny(int m, int n, int cus);
template <int KIND, int OUT> int launch_gemm_skinny(hipStream_t st, GemmArgs args, int cus);

}  // namespace wafer
