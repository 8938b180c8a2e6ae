// The radial network's last layer, gates = h W^T (h [E, 64], W [N, 64], N = paths * channels; reference
// mace_ictc/models/pure_cartesian_ictd_fix.py:1545-1553), its input adjoint gh = g W and its weight
// adjoint dW = g^T h, on the bf16 matrix cores with fp32 operands split into three parts
// (split_bf16.hpp).  E is edge-sized (1e3 .. 1e6), so each product moves one [E, N] fp32 tensor
// (1.24 GB at E = 105,634, N = 2,944) and should take the time of that stream.
//
// Measured at E = 105,634, N = 2,944, each product by itself in a replayed graph (rocBLAS / hipBLASLt fp32 before):
// gates 288 (408) us = 4.3 TB/s written, input adjoint 311 (373) us = 4.0 TB/s read, weight adjoint 293 (515: split
// products and a remainder) us = 4.3 TB/s read.  The six part products would take 95 us at the matrix cores' peak;
// one after the other in a training pass the matrix cores are busy 41, 39 and 47 % of the time.
// Errors against float64 (2-norm): 1.1e-7 (1.4e-7), 3.3e-7 (9.7e-7), 1.1e-6 (3.1e-6).
//
// Every kernel: 256 threads, v_mfma_f32_32x32x16_bf16.  The operand that all edges share (W, or h for
// the weight adjoint) is split once per block into LDS, in the instruction's operand order
// [part][octet of reduction steps][column], double-buffered with one barrier per chunk; the other
// operand goes from global memory straight into the operand registers of the one wave that uses it.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "split_bf16.hpp"

namespace ictc {
namespace {

constexpr int kGh = 64;                  // hidden width
constexpr int kGWaves = 4;
constexpr int kGThreads = kWave * kGWaves;
constexpr int kGPad = kGh + 1;           // columns per octet row (16-byte units): staggers the octets' banks

// A [64 reduction steps x 64 columns] operand in three parts.
struct OperandTile {
  bf16x8 v[3][8][kGPad];
};

__device__ __forceinline__ void put(OperandTile& t, int octet, int col, const float* w) {
  const Split8 s = split8(w);
#pragma unroll
  for (int q = 0; q < 3; ++q) t.v[q][octet][col] = s.p[q];
}

__device__ __forceinline__ Split8 get(const OperandTile& t, int octet, int col) {
  Split8 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.p[q] = t.v[q][octet][col];
  return s;
}

// LDS written and read by the lanes of one wave: the accesses of a wave complete in order; this
// keeps the compiler from reordering them.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.f;
  return v;
}

// ------------------------------------------------------------------------------------- gates
// out[e, n] = sum_c h[e, c] W[n, c].  A wave keeps 64 edges' split h in registers (96 VGPRs) for the
// whole launch and walks the columns; W arrives in chunks of 64 columns.  Each store instruction
// writes 256 contiguous bytes of two rows.
constexpr int kFwRows = 64;
template <bool VEC>
struct WeightRows {   // the thread's two octets of a 64-column chunk of W, along the hidden width
  float v[2][8];
  __device__ __forceinline__ static int octet(int t) { return VEC ? t & 7 : t >> 6; }
  __device__ __forceinline__ static int column(int t) { return VEC ? t >> 3 : t & 63; }
  __device__ __forceinline__ void load(const float* __restrict__ w, int64_t wsn, int64_t wsk, int n0, int N) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = threadIdx.x + kGThreads * i;
      int n = n0 + column(t);
      n = n < N ? n : N - 1;             // columns past N repeat the last one; their results are not stored
      const float* __restrict__ p = w + n * wsn + 8 * octet(t) * wsk;
      if constexpr (VEC) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = a[j], v[i][4 + j] = b[j];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = p[j * wsk];
      }
    }
  }
  __device__ __forceinline__ void store(OperandTile& tile) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = threadIdx.x + kGThreads * i;
      // columns in the order even, odd: a lane of the product then owns two neighbouring columns
      put(tile, octet(t), 32 * (column(t) & 1) + column(t) / 2, v[i]);
    }
  }
};

// PAIR: the output rows are 8-byte aligned (a lane's two columns in one store).
template <bool VEC, bool PAIR>
__global__ void __launch_bounds__(kGThreads, 2)
gates_forward_kernel(const float* __restrict__ h, const float* __restrict__ w, int64_t wsn, int64_t wsk,
                     float* __restrict__ out, int64_t ldo, int64_t E, int N, int chunks_per_block) {
  __shared__ OperandTile tile[2];
  const int lane = threadIdx.x & (kWave - 1), r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kGWaves + wave) * kFwRows;
  const int nchunks = (N + kGh - 1) / kGh;
  const int c0 = blockIdx.y * chunks_per_block;
  const int c1 = c0 + chunks_per_block < nchunks ? c0 + chunks_per_block : nchunks;
  WeightRows<VEC> wr;
  wr.load(w, wsn, wsk, c0 * kGh, N);
  Split8 a[4][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t er = row0 + 32 * t + r, e = er < E ? er : E - 1;   // rows past E repeat the last one, not stored
    const float* __restrict__ p = h + e * kGh + 8 * half;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float v[8];
      const f32x4 x = *reinterpret_cast<const f32x4*>(p + 16 * k), y = *reinterpret_cast<const f32x4*>(p + 16 * k + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = x[j], v[4 + j] = y[j];
      a[k][t] = split8(v);
    }
  }
  wr.store(tile[c0 & 1]);
  __syncthreads();
  const int rows = row0 >= E ? 0 : E - row0 < kFwRows ? static_cast<int>(E - row0) : kFwRows;   // wave-uniform
  const uint32_t ld = static_cast<uint32_t>(ldo) * 4u;
  const rsrc_t ro = make_rsrc(rows > 0 ? out + row0 * ldo : nullptr, rows * ld);
  for (int ch = c0; ch < c1; ++ch) {
    const bool more = ch + 1 < c1;
    if (more) wr.load(w, wsn, wsk, (ch + 1) * kGh, N);
    f32x16 acc[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) acc[t][ct] = zero16();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const Split8 b[2] = {get(tile[ch & 1], 2 * k + half, r), get(tile[ch & 1], 2 * k + half, 32 + r)};
      mfma_split(a[k], b, acc, acc);
    }
    const int n = ch * kGh + 2 * r;      // the lane's columns n, n + 1
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (any_nonfinite(acc[t][0]) || any_nonfinite(acc[t][1])) {   // see split_bf16.hpp: again in fp32
        for (int i = 0; i < 16; ++i) {
          const int er = 32 * t + mfma_row(i, half);
          const int64_t e = row0 + er < E ? row0 + er : E - 1;
          for (int ct = 0; ct < 2; ++ct) {
            const float* __restrict__ wp = w + (n + ct < N ? n + ct : N - 1) * wsn;
            float v = 0.f;
            for (int k = 0; k < kGh; ++k) v = fmaf(h[e * kGh + k], wp[k * wsk], v);
            buf_store<1>(ro, n + ct < N ? er * ld + (n + ct) * 4u : 0xFFFFFFF0u, Vec<1>{{v}});
          }
        }
      } else if (PAIR && rows == kFwRows && (ch + 1) * kGh <= N) {   // whole tile: row offsets in SGPRs
        const uint32_t voff = 4u * half * ld + n * 4u;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const f32x2 v{acc[t][0][i] * kSplitUnscale, acc[t][1][i] * kSplitUnscale};
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), ro, voff,
                                                (32 * t + mfma_row(i, 0)) * ld, kNonTemporal);
        }
      } else {
        uint32_t step = ld;                  // opaque: the 32 row offsets are formed here, not kept through the loop
        asm volatile("" : "+s"(step));
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct)
            buf_store<1>(ro, n + ct < N ? (32 * t + mfma_row(i, half)) * step + (n + ct) * 4u : 0xFFFFFFF0u,
                         Vec<1>{{acc[t][ct][i] * kSplitUnscale}});
      }
    }
    if (more) wr.store(tile[(ch + 1) & 1]);
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------ input adjoint
// gh[e, c] = sum_n g[e, n] W[n, c]: the reduction runs along the rows of the [E, N] operand (two
// chunks in flight per wave measured the same as one).  A wave
// owns 32 edges and all 64 columns; per 32-step chunk its lanes read 128 contiguous bytes of eight rows
// per instruction, one chunk ahead, and pass them through the wave's own LDS rows to the lanes
// that need them (read by operand lanes directly, four instructions would share each line and the
// lines in flight of a CU exceed its L1: 637 us at E = 105,634, N = 2,944).
constexpr int kIgSteps = 32;

struct StepTile {
  bf16x8 v[3][kIgSteps / 8][kGh];
};

// 16-byte piece p (of eight) of row r of a wave's 32 x 32 staging area, in units of four floats: the
// pieces of a row are rotated so that the operand reads of eight neighbouring rows meet all banks.
__device__ __forceinline__ int stage_slot(int r, int p) { return r * 8 + (p ^ (r & 7)); }

// Four blocks per CU (128 VGPRs, 40 KB of LDS): the 826 blocks of E = 105,634 are then resident at once
// (at three per CU a second round of 58 blocks doubled the time).  Above E = 131,072 a second round begins here: 365
// us at 131,072, 401 at 131,200 (library 466, 480).
__global__ void __launch_bounds__(kGThreads, 4)
gates_input_grad_kernel(const float* __restrict__ g, int64_t ldg, const float* __restrict__ w, int64_t wsn, int64_t wsk,
                        float* __restrict__ out, int64_t E, int N) {
  __shared__ StepTile tile[2];
  __shared__ __align__(16) f32x4 sG[kGWaves][32 * kIgSteps / 4];
  const int lane = threadIdx.x & (kWave - 1), r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kGWaves + wave) * 32;
  const int nchunks = (N + kIgSteps - 1) / kIgSteps;
  const int rows = row0 >= E ? 0 : E - row0 < 32 ? static_cast<int>(E - row0) : 32;   // wave-uniform
  const uint32_t ld = static_cast<uint32_t>(ldg) * 4u;
  // rows past E lie beyond the descriptor and read 0
  const rsrc_t rg = make_rsrc(rows > 0 ? g + row0 * ldg : nullptr, rows * ld);
  const rsrc_t rw = make_rsrc(w, static_cast<uint32_t>(((N - 1) * wsn + (kGh - 1) * wsk + 1) * 4));
  const int lr = lane >> 3, lp = lane & 7;               // the lane's row (of eight) and 16-byte piece
  const int wc = threadIdx.x & 63, wo = threadIdx.x >> 6;   // its octet of W: column, octet of steps
  const uint32_t wvoff = static_cast<uint32_t>((8 * wo * wsn + wc * wsk) * 4), wstep = static_cast<uint32_t>(wsn) * 4u;
  const uint32_t goff = lr * ld + lp * 16u;
  float wv[8];
  f32x4 gv[4];
  auto fetch_w = [&](int ch) {
    const int n0 = ch * kIgSteps;
    if (n0 + kIgSteps <= N) {
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = buf_load_vs(rw, wvoff, (n0 + j) * wstep);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        wv[j] = buf_load<1>(rw, n0 + 8 * wo + j < N ? wvoff + (n0 + j) * wstep : 0xFFFFFFF0u).v[0];
    }
  };
  auto fetch_g = [&](int ch) {
    const bool in = ch * kIgSteps + 4 * lp < N;          // N is a multiple of 4
    const uint32_t off = in ? goff + ch * (kIgSteps * 4u) : 0xFFFFFFF0u - 24u * ld;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Vec<4> t = buf_load<4, kNonTemporal>(rg, off + 8u * i * ld);
      gv[i] = f32x4{t.v[0], t.v[1], t.v[2], t.v[3]};
    }
  };
  auto store_w = [&](StepTile& t) {
    const Split8 s = split8(wv);
#pragma unroll
    for (int q = 0; q < 3; ++q) t.v[q][wo][wc] = s.p[q];
  };
  fetch_w(0);
  fetch_g(0);
  store_w(tile[0]);
  __syncthreads();
  f32x16 hi[1][2] = {{zero16(), zero16()}}, lo[1][2] = {{zero16(), zero16()}};
  f32x4* __restrict__ sg = sG[wave];
  for (int ch = 0; ch < nchunks; ++ch) {
    const bool more = ch + 1 < nchunks;
#pragma unroll
    for (int i = 0; i < 4; ++i) sg[stage_slot(8 * i + lr, lp)] = gv[i];
    if (more) {
      fetch_g(ch + 1);
      fetch_w(ch + 1);
    }
    wave_lds_order();                                    // the wave's own rows, in order
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const f32x4 x = sg[stage_slot(r, 4 * k + 2 * half)], y = sg[stage_slot(r, 4 * k + 2 * half + 1)];
      float u[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) u[j] = x[j], u[4 + j] = y[j];
      const Split8 a[1] = {split8(u)};
      Split8 b[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int q = 0; q < 3; ++q) b[ct].p[q] = tile[ch & 1].v[q][2 * k + half][32 * ct + r];
      mfma_split(a, b, hi, lo);
    }
    if (more) store_w(tile[(ch + 1) & 1]);
    __syncthreads();
  }
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int i = 0; i < 16; ++i) hi[0][ct][i] = (hi[0][ct][i] + lo[0][ct][i]) * kSplitUnscale;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const int c = 32 * ct + r;
    const bool redo = any_nonfinite(hi[0][ct]);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t row = row0 + mfma_row(i, half);
      if (row < E) {
        float v = hi[0][ct][i];
        if (redo) {
          v = 0.f;
          for (int n = 0; n < N; ++n) v = fmaf(g[row * ldg + n], w[n * wsn + c * wsk], v);
        }
        out[row * kGh + c] = v;
      }
    }
  }
}

// ----------------------------------------------------------------------------- weight adjoint
// dW[n, c] = sum_e g[e, n] h[e, c].  A block owns 256 columns of g (64 per wave) and a range of edges;
// the reduction index is the edge, so a lane's g operand is eight rows of one column: each load
// instruction reads two whole 128-byte lines.  h is split into LDS 32 edges at a time.  Partials per
// edge range are summed in range order by gates_weight_sum_kernel.
constexpr int kWgCols = 256;
constexpr int kWgEdges = 32;

struct HiddenTile {
  bf16x8 v[3][kWgEdges / 8][kGPad];
};

__global__ void __launch_bounds__(kGThreads, 2)
gates_weight_grad_kernel(const float* __restrict__ g, int64_t ldg, const float* __restrict__ h, float* __restrict__ ws,
                         int64_t E, int N, int64_t per_range) {
  __shared__ HiddenTile tile[2];
  const int lane = threadIdx.x & (kWave - 1), r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n0 = blockIdx.x * kWgCols + 64 * wave;
  const int64_t e0 = blockIdx.y * per_range, e1 = e0 + per_range < E ? e0 + per_range : E;
  const int hc = threadIdx.x & 63, ho = threadIdx.x >> 6;   // the thread's octet of h: column, octet of edges
  const uint32_t ld = static_cast<uint32_t>(ldg) * 4u;
  uint32_t voff[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int n = n0 + 32 * t + r;
    voff[t] = 8u * half * ld + (n < N ? n : N - 1) * 4u;   // columns past N repeat the last one; not stored
  }
  const uint32_t hoff = (8u * ho * kGh + hc) * 4u;
  float hv[8], gv[2][2][8];
  // Rows of a whole chunk: uniform row offsets in SGPRs.  The last, partial chunk of a range: rows past
  // its end lie beyond the descriptors and read 0 (offsets in the checked operand).
  auto fetch_h = [&](int64_t eb) {
    const int64_t n = e1 - eb < kWgEdges ? e1 - eb : kWgEdges;
    const rsrc_t rh = make_rsrc(h + eb * kGh, static_cast<uint32_t>(n) * kGh * 4u);
#pragma unroll
    for (int j = 0; j < 8; ++j) hv[j] = buf_load<1>(rh, hoff + j * kGh * 4u).v[0];
  };
  auto fetch_g = [&](int64_t eb, int k) {
    const int64_t n = e1 - eb < kWgEdges ? e1 - eb : kWgEdges;
    const rsrc_t rg = make_rsrc(g + eb * ldg, static_cast<uint32_t>(n) * ld);
    if (n == kWgEdges) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) gv[t][k][j] = buf_load_vs<kNonTemporal>(rg, voff[t], (16 * k + j) * ld);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) gv[t][k][j] = buf_load<1, kNonTemporal>(rg, voff[t] + (16 * k + j) * ld).v[0];
    }
  };
  auto store_h = [&](HiddenTile& t) {
    const Split8 s = split8(hv);
#pragma unroll
    for (int q = 0; q < 3; ++q) t.v[q][ho][hc] = s.p[q];
  };
  f32x16 acc[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) acc[t][ct] = zero16();
  // One step ahead: while the 24 matrix instructions of a 16-edge step run, the next step's g values
  // are split (the interleave asked for below), so that the two pipes work at the same time.
  Split8 a[2];
  auto split_g = [&](int k, Split8 (&to)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) to[t] = split8(gv[t][k]);
  };
  auto step = [&](const HiddenTile& t, int k) {
    Split8 s[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int q = 0; q < 3; ++q) s[ct].p[q] = t.v[q][2 * k + half][32 * ct + r];
    mfma_split(a, s, acc, acc);
  };
  fetch_h(e0);
#pragma unroll
  for (int k = 0; k < 2; ++k) fetch_g(e0, k);
  store_h(tile[0]);
  split_g(0, a);
  __syncthreads();
  int b = 0;
  for (int64_t eb = e0; eb < e1; eb += kWgEdges, b ^= 1) {
    const bool more = eb + kWgEdges < e1;
    const int64_t nb = more ? eb + kWgEdges : eb;   // past the end: this chunk again, unused
    Split8 next[2];
    fetch_h(nb);
    fetch_g(nb, 0);
    split_g(1, next);
    step(tile[b], 0);
#pragma unroll
    for (int q = 0; q < 4 * kSplitProducts; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one matrix instruction
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);   // four VALU instructions
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) a[t] = next[t];
    fetch_g(nb, 1);
    split_g(0, next);
    step(tile[b], 1);
#pragma unroll
    for (int q = 0; q < 4 * kSplitProducts; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) a[t] = next[t];
    if (more) store_h(tile[b ^ 1]);
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      unscale(acc[t][ct]);
      const bool redo = any_nonfinite(acc[t][ct]);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int n = n0 + 32 * t + mfma_row(i, half), c = 32 * ct + r;
        if (n < N) {
          float v = acc[t][ct][i];
          if (redo) {
            v = 0.f;
            for (int64_t e = e0; e < e1; ++e) v = fmaf(g[e * ldg + n], h[e * kGh + c], v);
          }
          ws[(static_cast<int64_t>(blockIdx.y) * N + n) * kGh + c] = v;
        }
      }
    }
}

// out[n, c] = sum over the ranges' partials in order, four threads per entry in a fixed interleave.
__global__ void __launch_bounds__(256)
gates_weight_sum_kernel(const float* __restrict__ ws, int ranges, int N, float* __restrict__ out, int64_t osn,
                        int64_t osk) {
  __shared__ float part[3][kGh];
  const int c = threadIdx.x & 63, p = threadIdx.x >> 6, n = blockIdx.x;
  const int64_t step = static_cast<int64_t>(N) * kGh;
  const float* __restrict__ src = ws + static_cast<int64_t>(n) * kGh + c;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  int k = p;
  for (; k + 12 < ranges; k += 16)
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] += src[(k + 4 * j) * step];
  for (; k < ranges; k += 4) s[0] += src[k * step];
  const float v = (s[0] + s[1]) + (s[2] + s[3]);
  if (p > 0) part[p - 1][c] = v;
  __syncthreads();
  if (p == 0) out[n * osn + c * osk] = ((v + part[0][c]) + part[1][c]) + part[2][c];
}

// Edge ranges of a weight-adjoint launch: two resident blocks per CU over the column blocks, and at
// least 128 edges each.
int weight_grad_ranges(int64_t E, int64_t N) {
  const int64_t cols = (N + kWgCols - 1) / kWgCols;
  const int64_t want = (2 * static_cast<int64_t>(compute_units())) / cols, most = (E + 127) / 128;
  const int64_t k = want < most ? want : most;
  return static_cast<int>(k < 1 ? 1 : k);
}

// Column chunks per block of a forward launch: the split of the columns with the fewest rounds of
// resident blocks (two per CU), each costing its chunks and about one and a half more for the block's
// own rows.
int64_t forward_chunks(int64_t rows, int64_t nchunks) {
  const int64_t slots = 2 * static_cast<int64_t>(compute_units());
  int64_t best = nchunks, cost = INT64_MAX;
  for (int64_t split = 1; split <= nchunks; ++split) {
    const int64_t per = (nchunks + split - 1) / split, blocks = rows * ((nchunks + per - 1) / per);
    const int64_t c = (blocks + slots - 1) / slots * (2 * per + 3);
    if (c < cost) cost = c, best = per;
  }
  return best;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Widths and edge counts the kernels index with 32 bits per wave (32 rows of the [E, N] tensor).
bool gates_sizes_ok(int64_t E, int64_t N, int64_t ld) {
  return E >= 0 && N >= 1 && N <= (1 << 20) && ld >= N && ld <= (1 << 22) && E <= (static_cast<int64_t>(1) << 31);
}

// A weight whose elements lie within a 32-bit byte offset of its base.
bool weight_ok(int64_t N, int64_t wsn, int64_t wsk) {
  return wsn >= 0 && wsk >= 0 && wsn <= (1 << 28) && wsk <= (1 << 22) && (N - 1) * wsn + (kGh - 1) * wsk < (1 << 29);
}

}  // namespace
}  // namespace ictc

extern "C" int ictc_hip_gates_forward(const float* hidden, const float* weight, int64_t weight_row_stride,
                                      int64_t weight_col_stride, float* out, int64_t out_row_stride, int64_t edges,
                                      int64_t width, hipStream_t stream) {
  using namespace ictc;
  if (!gates_sizes_ok(edges, width, out_row_stride) || !weight_ok(width, weight_row_stride, weight_col_stride))
    return ICTC_ERR_INVALID_ARGUMENT;
  if (edges == 0) return ICTC_OK;
  if (!hidden || !weight || !out) return ICTC_ERR_INVALID_ARGUMENT;
  if (!aligned16(hidden)) return ICTC_ERR_UNSUPPORTED;
  const int64_t rows = (edges + kFwRows * kGWaves - 1) / (kFwRows * kGWaves), nchunks = (width + kGh - 1) / kGh;
  const int64_t per = forward_chunks(rows, nchunks);
  const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>((nchunks + per - 1) / per));
  const bool vec = weight_col_stride == 1 && weight_row_stride % 4 == 0 && aligned16(weight);
  const bool pair = out_row_stride % 2 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kGThreads), 0, stream, hidden, weight, weight_row_stride, weight_col_stride,
                       out, out_row_stride, edges, static_cast<int>(width), static_cast<int>(per));
  };
  if (vec && pair) launch(gates_forward_kernel<true, true>);
  else if (vec) launch(gates_forward_kernel<true, false>);
  else if (pair) launch(gates_forward_kernel<false, true>);
  else launch(gates_forward_kernel<false, false>);
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}

extern "C" int ictc_hip_gates_input_grad(const float* grad, int64_t grad_row_stride, const float* weight,
                                         int64_t weight_row_stride, int64_t weight_col_stride, float* out,
                                         int64_t edges, int64_t width, hipStream_t stream) {
  using namespace ictc;
  if (!gates_sizes_ok(edges, width, grad_row_stride) || !weight_ok(width, weight_row_stride, weight_col_stride))
    return ICTC_ERR_INVALID_ARGUMENT;
  if (edges == 0) return ICTC_OK;
  if (!grad || !weight || !out) return ICTC_ERR_INVALID_ARGUMENT;
  if (!aligned16(grad) || grad_row_stride % 4 != 0 || width % 4 != 0) return ICTC_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>((edges + 32 * kGWaves - 1) / (32 * kGWaves)));
  hipLaunchKernelGGL(gates_input_grad_kernel, grid, dim3(kGThreads), 0, stream, grad, grad_row_stride, weight,
                     weight_row_stride, weight_col_stride, out, edges, static_cast<int>(width));
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}

extern "C" int64_t ictc_hip_gates_weight_grad_workspace(int64_t edges, int64_t width) {
  if (!ictc::gates_sizes_ok(edges, width, width)) return -ICTC_ERR_INVALID_ARGUMENT;
  return edges == 0 ? 0 : ictc::weight_grad_ranges(edges, width) * width * ictc::kGh;
}

extern "C" int ictc_hip_gates_weight_grad(const float* grad, int64_t grad_row_stride, const float* hidden,
                                          float* workspace, int64_t workspace_floats, float* out,
                                          int64_t out_row_stride, int64_t out_col_stride, int64_t edges, int64_t width,
                                          hipStream_t stream) {
  using namespace ictc;
  if (!gates_sizes_ok(edges, width, grad_row_stride) || !out) return ICTC_ERR_INVALID_ARGUMENT;
  if (edges > 0 && (!grad || !hidden || !workspace)) return ICTC_ERR_INVALID_ARGUMENT;
  int ranges = edges == 0 ? 0 : weight_grad_ranges(edges, width);
  if (workspace_floats < ranges * width * kGh) return ICTC_ERR_INVALID_ARGUMENT;
  if (edges > 0) {
    const int64_t per = ((edges + ranges - 1) / ranges + kWgEdges - 1) / kWgEdges * kWgEdges;
    ranges = static_cast<int>((edges + per - 1) / per);   // every launched range holds edges
    const dim3 grid(static_cast<unsigned>((width + kWgCols - 1) / kWgCols), static_cast<unsigned>(ranges));
    hipLaunchKernelGGL(gates_weight_grad_kernel, grid, dim3(kGThreads), 0, stream, grad, grad_row_stride, hidden,
                       workspace, edges, static_cast<int>(width), per);
    if (hipGetLastError() != hipSuccess) return ICTC_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(gates_weight_sum_kernel, dim3(static_cast<unsigned>(width)), dim3(256), 0, stream, workspace,
                     ranges, static_cast<int>(width), out, out_row_stride, out_col_stride);
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}
