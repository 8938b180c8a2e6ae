// fp32 products on the bf16 matrix cores (gfx950): each fp32 operand is split into three bf16
// parts and the product is the sum of the six leading part products.
//
// a = a0 + a1 + a2 with a0 = bf16(a), a1 = bf16(a - a0), a2 = a - a0 - a1 (round to nearest even):
// a bf16 holds 8 significant bits, so the remainder after two parts has at most 8 and the split is
// exact.  |a1| <= 2^-8 |a| and |a2| <= 2^-16 |a|, so
//   a b = a0 b0 + (a0 b1 + a1 b0) + (a0 b2 + a1 b1 + a2 b0) + O(2^-24 |a b|)
// The dropped terms, of random sign, are below the fp32 rounding of a sum: over the radial network's and
// the message linear's sizes the errors against float64 are 0.4 to 0.9 times those of fp32 FMAs (2-norm;
// the largest entry's alike).  A sum that one product dominates can err by 1.7 times 2^-24, an FMA by 1.
// The matrix core
// multiplies bf16 exactly and accumulates in fp32.  Its dense bf16 peak is 16 times the fp32 one
// (2.5 PFLOP/s and 157 TFLOP/s), so six part products cost 3/8 of the fp32 instructions' time.
//
// Operands are split times 2^24: the last bit of the smallest fp32 number (2^-149) is then a normal
// bf16 (2^-125), so that no part loses bits to subnormals (split unscaled, an operand below 2^-110 lost
// its third part and one near 2^-126 was off by 1e-3).  Both scalings are exact; results are multiplied by
// 2^-48 (kSplitUnscale).
//
// Operands of 2^103 and more, results of 2^80 and more, infinities and NaNs leave a NaN or an infinity
// in the accumulators (inf - inf in the split); the kernels look for non-finite results and evaluate
// those again with plain fp32 FMAs, so the results are the fp32 ones there too.
#pragma once
#include "ictc_common.hpp"

namespace ictc {

using bf16x2 = __bf16 __attribute__((ext_vector_type(2)));
using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
using f32x2 = float __attribute__((ext_vector_type(2)));
using f32x16 = float __attribute__((ext_vector_type(16)));

// Eight consecutive reduction entries of one row (or column): a lane's operand of
// v_mfma_f32_32x32x16_bf16, in three parts.
struct Split8 {
  bf16x8 p[3];
};

constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

__device__ __forceinline__ Split8 split8(const float* v) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    f32x2 x{v[i] * kSplitScale, v[i + 1] * kSplitScale};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const bf16x2 b = __builtin_convertvector(x, bf16x2);
      s.p[q][i] = b[0];
      s.p[q][i + 1] = b[1];
      if (q < 2) {
        x[0] -= static_cast<float>(b[0]);
        x[1] -= static_cast<float>(b[1]);
      }
    }
  }
  return s;
}

// The part products, smallest first.
constexpr int kSplitProducts = 6;
constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

// acc[t][c] += 2^48 a[t] b[c] over 16 reduction steps: lane l supplies row (column) l % 32 and steps
// 8 (l / 32) .. + 8, and receives D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32], i = 0..15.  Consecutive
// instructions go to different accumulators (a dependent one waits out its predecessor's passes).
// Long reductions give the five small part products accumulators of their own (lo, added once at
// the end), so that the main ones round once per 16 steps; short ones pass the same twice.
template <int T, int C>
__device__ __forceinline__ void mfma_split(const Split8 (&a)[T], const Split8 (&b)[C], f32x16 (&hi)[T][C],
                                           f32x16 (&lo)[T][C]) {
#pragma unroll
  for (int q = 0; q < kSplitProducts; ++q)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        f32x16& acc = q < kSplitProducts - 1 ? lo[t][c] : hi[t][c];
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t].p[kSplitA[q]], b[c].p[kSplitB[q]], acc, 0, 0, 0);
      }
}

// The accumulators of scaled operands to the products' scale, in place (infinities and NaNs stay).
__device__ __forceinline__ void unscale(f32x16& v) {
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] *= kSplitUnscale;
}

__device__ __forceinline__ int mfma_row(int i, int half) { return 8 * (i / 4) + 4 * half + i % 4; }

// Whether any lane of the wave holds a non-finite value (the sum of v * 0 is 0 or NaN).
__device__ __forceinline__ bool any_nonfinite(const f32x16& v) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s = fmaf(v[i], 0.f, s);
  return __ballot(!(s == 0.f)) != 0;
}

}  // namespace ictc
