// Symmetric-contraction plans: one specialisation per (lmax, target_lmax, correlation),
// generated by csrc/gen_sc.py (straight-line chain evaluation, see that file).
//
// The generated code is written once over a scalar V with the operations below.
// V = float evaluates the chains; V = Dual carries a tangent t alongside every value
// (x + eps t, eps^2 = 0), so the same code yields directional derivatives: the
// forward becomes a JVP, the VJP a Hessian-vector product, the weight features their
// derivative along t.  Weights and cotangents stay plain float.
#pragma once
#include <hip/hip_runtime.h>

namespace ictc {
namespace sc {

struct Dual {
  float v, d;
  __device__ Dual() = default;
  __device__ constexpr Dual(float value) : v(value), d(0.f) {}  // NOLINT: constants lift implicitly
  __device__ constexpr Dual(float value, float tangent) : v(value), d(tangent) {}
};

__device__ __forceinline__ Dual operator*(Dual a, Dual b) { return {a.v * b.v, fmaf(a.v, b.d, a.d * b.v)}; }
__device__ __forceinline__ Dual operator*(float a, Dual b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ Dual operator*(Dual a, float b) { return {a.v * b, a.d * b}; }
__device__ __forceinline__ Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }

// a * b + c for every mix of float and Dual operands that the generated code forms
__device__ __forceinline__ float sfma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ Dual sfma(float a, float b, Dual c) { return {fmaf(a, b, c.v), c.d}; }
__device__ __forceinline__ Dual sfma(float a, Dual b, float c) { return {fmaf(a, b.v, c), a * b.d}; }
__device__ __forceinline__ Dual sfma(float a, Dual b, Dual c) { return {fmaf(a, b.v, c.v), fmaf(a, b.d, c.d)}; }
__device__ __forceinline__ Dual sfma(Dual a, Dual b, Dual c) {
  return {fmaf(a.v, b.v, c.v), fmaf(a.v, b.d, fmaf(a.d, b.v, c.d))};
}

// what a float-valued result keeps: the value, or the tangent of a Dual
__device__ __forceinline__ float part(float a) { return a; }
__device__ __forceinline__ float part(Dual a) { return a.d; }

// opaque to the optimiser: stops loop-invariant hoisting of work on the input copy
__device__ __forceinline__ void launder(float& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void launder(Dual& a) {
  asm volatile("" : "+v"(a.v));
  asm volatile("" : "+v"(a.d));
}

// Sums of the weight features over several nodes, one LDS column per lane ([KTOT][64] floats of the wave):
// the generated assignment phi[p * Cs] = v adds v to the lane's sum of column p.  Cs stays the
// compile-time stride, so that every column has an immediate LDS offset.
struct LdsSums {
  float* p;
  struct Ref {
    float* at;
    __device__ __forceinline__ void operator=(float v) const { *at += v; }
  };
  __device__ __forceinline__ Ref operator[](int i) const { return {p + i}; }
};

// the stride of a node's phi row, opaque like the inputs (row addresses formed inside their step)
__device__ __forceinline__ void launder(int& stride, float*) { asm volatile("" : "+s"(stride)); }
__device__ __forceinline__ void launder(int&, LdsSums) {}

template <int L, int T, int K>
struct Plan;

}  // namespace sc
}  // namespace ictc
