// Per-degree channel linear on the matrix cores (gfx950): the path-preserving message linear of the
// MACE interaction (reference mace_ictc/models/pure_cartesian_ictd_fix.py:629-661,
// PathPreservingLinearSO3; native route ictc_o3/ascendc/linear.py:12-136), applied straight to
// the message kernel's packed output and writing the mul_ir node layout.
//
// Per degree l (d = 2l + 1, K_l = counts[l] * C):
//   x  row n, degree block l:  [counts[l]][d][C]          (ir_mul, the message output)
//   y  row n, degree block l:  [O][d]                     (mul_ir, offset O * l^2)
//   forward:     y[n, o, m]            = alpha * sum_{k, c} W_l[o, k C + c] x[n, k, m, c]
//   input grad:  gx[n, k, m, c]        = alpha * sum_o gy[n, o, m] W_l[o, k C + c]
//   mul_ir map:  y[n, o, m]            = alpha * sum_c W_l[o, c] x[n, c, m]   (counts all 1; x
//                                        mul_ir [N, C (L+1)^2], per degree [C][d] at offset C l^2)
// i.e. for the rows rho = n d + m, Y = alpha X W^T and gX = alpha gY W, one GEMM per degree with
// the layout changes folded into the tile loads and stores (no transposed copies, no
// concatenation, the 1/avg_num_neighbors scale as alpha).
//
// Calls that give every CU a block run on the bf16 matrix cores with fp32 operands in three parts (the split
// kernels below; `launch` has the lines), the weight gradient always; smaller calls, and short products of up
// to 64 columns, on fp32 MFMA, in more and smaller blocks:
//
// Tiling: a 256-thread block computes a 64-row x 64-column output tile of one degree (grid.z);
// K is walked in chunks of 32 staged through LDS, then each wave runs v_mfma_f32_16x16x4_f32 over
// its 16 rows and the tile's 4 column tiles.  Operand layout of that instruction: lane l supplies
// A[l % 16][k_l] and B[k_l][l % 16] and receives D[4 (l / 16) + v][l % 16], v = 0..3, where k_l is
// the instruction's k index l / 16.  Which actual k a lane feeds is free as long as A and B agree:
// here four consecutive MFMAs j = 0..3 cover a 16-wide k group with k = 4 (l / 16) + j, so each
// lane reads its four A (and B) values of a group with one 16-byte LDS read.  Every sum runs in a
// fixed order (bit-identical run to run).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ictc_common.hpp"
#include "ictc_hip.h"
#include "split_bf16.hpp"

namespace ictc {
namespace {

constexpr int kTile = 64;   // rows per block, and columns per block of the forward modes
constexpr int kTileIg = 128;   // columns per block of the input adjoint
constexpr int kKc = 32;     // K per LDS chunk
constexpr int kPitch = kKc + 4;   // LDS row pitch in floats (16-byte aligned rows)

typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct DegreeGeometry {
  int64_t rows;       // N d
  int d;              // 2l + 1
  int k;              // counts[l] * C
  int64_t xoff;       // first float of the degree block in an x row
  int64_t yoff;       // first float of the degree block in a y row
  const float* w;     // [O, k]
};

struct LinearArgs {
  DegreeGeometry g[ICTC_LINEAR_MAX_DEGREES];
  int64_t xwidth, ywidth;
  int channels, out_channels;
  float alpha;
};

// MODE kForward: A = x rows (K = x columns), B^T = W rows, D -> y.  kInputGrad: A = gy rows
// (K = O), B = W, D -> gx columns.  kMulIr: A = mul_ir x rows (K = C, stride d), B^T = W rows,
// D -> y (mul_ir).  kMulIrT: kMulIr with the weights given transposed (B = W [K, O] rows read
// like kInputGrad's, so no transposed copy of W is made).  VEC (channels, and for kInputGrad and
// kMulIrT out_channels, multiples of 32): every
// 32-wide K chunk is full, each K chunk of an x row lies in one path block and weight rows are
// float4-aligned, so operands are fetched into registers one chunk ahead (their loads in flight
// while the MFMAs of the current chunk run); with two LDS buffers
// (NBUF 2) the next chunk is staged into the other buffer right after those MFMAs (one barrier per
// chunk), with one (NBUF 1, half the LDS and so twice the resident blocks) after a second barrier.
// The forward's long K (counts C) takes two buffers, the input adjoint's short K (O) one.
// Without VEC, element by element, one chunk at a time.
enum LinearMode { kForward = 0, kInputGrad = 1, kMulIr = 2, kMulIrT = 3 };

template <int MODE, bool VEC, int NBUF, int TN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NBUF == 1 ? (TN > kTile ? 5 : 8) : 4)))
degree_linear_kernel(const float* __restrict__ in, float* __restrict__ out, const LinearArgs a) {
  constexpr bool FWD = MODE != kInputGrad;      // D -> mul_ir y rows
  constexpr bool BT = MODE == kInputGrad || MODE == kMulIrT;   // B = W rows over K (staged transposed)
  constexpr int NT = TN / 16;                   // 16-column MFMA tiles per wave
  static_assert(BT ? (TN == kTile || TN == kTileIg) : TN == kTile, "column tile");
  constexpr bool STRIDED = MODE != kForward;    // A rows read at stride d over K (mul_ir)
  // the degree's geometry in registers (read once from the kernel arguments)
  const DegreeGeometry g = a.g[blockIdx.z];
  const int d = g.d;
  const int ncols = FWD ? a.out_channels : g.k;   // output columns
  const int kdim = FWD ? g.k : a.out_channels;    // reduction length
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int c0 = blockIdx.y * TN;
  // uniform per block; a degree without path blocks (kdim 0) writes its zero forward rows
  if (r0 >= g.rows || c0 >= ncols) return;
  __shared__ __align__(16) float sA[NBUF][kTile][kPitch];   // [buffer][row][k]
  __shared__ __align__(16) float sB[NBUF][TN][kPitch];      // [buffer][column][k]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int C = a.channels;
  // A staging: thread t holds 8 consecutive k of tile row t / 4
  const int ar = tid >> 2, akq = (tid & 3) * 8;
  const int64_t arho = r0 + ar;
  const bool arow = arho < g.rows;
  const int64_t an = arow ? arho / d : 0;
  const int am = arow ? static_cast<int>(arho - an * d) : 0;
  const float* __restrict__ abase = MODE == kForward   ? in + an * a.xwidth + g.xoff + static_cast<int64_t>(am) * C
                                    : MODE == kInputGrad ? in + an * a.ywidth + g.yoff + am
                                                         : in + an * a.xwidth + g.xoff + am;
  // !FWD B staging: thread t holds weight row k0 + t / 8, columns c0 + CPT (t % 8) .. + CPT - 1
  // (CPT = TN / 8: two or four float4 loads), stored transposed element by element.  The k index
  // of B column col is XOR-swizzled by bsw(col) (a multiple of 8 below 32, so every aligned
  // 4-group of k stays contiguous and in its row; it follows col / 8 for CPT 8, col / 16 for
  // CPT 16, the bits that tell the lanes of one store apart): the transposed stores of a wave
  // then meet at most two lanes per bank, and with the 36-float pitch the 16-byte MFMA operand
  // reads stay conflict-free.
  constexpr int CPT = TN / 8;
  const int wk = tid >> 3, wc = (tid & 7) * CPT;
  auto bsw = [](int col) { return BT ? ((col >> (CPT == 16 ? 4 : 3)) & 3) * 8 : 0; };
  const int wld = MODE == kInputGrad ? g.k : ncols;   // BT: floats per weight row (over the columns)
  f32x4_t acc[NT] = {};
  const int fr = lane & 15, fq = (lane >> 4) * 4;
  auto mfma_chunk = [&](int buf) {
#pragma unroll
    for (int kg = 0; kg < kKc; kg += 16) {
      const f32x4_t av = *reinterpret_cast<const f32x4_t*>(&sA[buf][wave * 16 + fr][kg + fq]);
      if constexpr (NBUF == 1) {
        // one B operand live at a time (the register budget of 8 waves per SIMD); the
        // accumulation chains of the other resident waves fill the MFMA pipe
#pragma unroll
        for (int t = 0; t < NT; t += 2) {
          const f32x4_t bv0 = *reinterpret_cast<const f32x4_t*>(&sB[buf][t * 16 + fr][(kg + fq) ^ bsw(t * 16 + fr)]);
          const f32x4_t bv1 = *reinterpret_cast<const f32x4_t*>(&sB[buf][t * 16 + 16 + fr][(kg + fq) ^ bsw(t * 16 + 16 + fr)]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv0[j], acc[t], 0, 0, 0);
            acc[t + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv1[j], acc[t + 1], 0, 0, 0);
          }
        }
      } else {
        f32x4_t bv[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          bv[t] = *reinterpret_cast<const f32x4_t*>(&sB[buf][t * 16 + fr][(kg + fq) ^ bsw(t * 16 + fr)]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv[t][j], acc[t], 0, 0, 0);
        }
      }
    }
  };
  if constexpr (VEC) {
    // registers of one chunk: A (8 floats of the thread's row), B (8 floats, or CPT of the
    // input adjoint's weight row)
    constexpr int NRB = BT ? CPT / 4 : 2;
    f32x4_t ra0, ra1, rb[NRB];
    // Every K chunk is full under VEC (kdim a multiple of 32), and no load is conditional on the
    // lane: a select or a branch on a loaded value would wait for the load at the fetch instead of
    // at the stage.  Rows past the end read row 0 and columns past the end read the last valid
    // weight columns: their products land in output rows / columns that are never stored.
    auto fetch = [&](int k0) {
      if constexpr (STRIDED) {   // mul_ir row: stride d over K
        const float* p = abase + (k0 + akq) * d;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          ra0[u] = p[u * d];
          ra1[u] = p[(u + 4) * d];
        }
      } else {
        const int blk = k0 / C, c = k0 - blk * C + akq;
        const float* p = abase + blk * d * C + c;
        ra0 = *reinterpret_cast<const f32x4_t*>(p);
        ra1 = *reinterpret_cast<const f32x4_t*>(p + 4);
      }
      if constexpr (!BT) {
        const int col = c0 + ar < ncols ? c0 + ar : ncols - 1;   // weight row col, 8 consecutive k
        const float* p = g.w + static_cast<int64_t>(col) * g.k + k0 + akq;
        rb[0] = *reinterpret_cast<const f32x4_t*>(p);
        rb[1] = *reinterpret_cast<const f32x4_t*>(p + 4);
      } else {
        // ncols is a multiple of 32 under VEC and CPT is 8 or 16: the clamped run of CPT
        // columns stays in range
        const int col = c0 + wc < ncols ? c0 + wc : ncols - CPT;
        const float* p = g.w + static_cast<int64_t>(k0 + wk) * wld + col;
#pragma unroll
        for (int q = 0; q < NRB; ++q) rb[q] = *reinterpret_cast<const f32x4_t*>(p + 4 * q);
      }
    };
    auto stage = [&](int buf) {
      *reinterpret_cast<f32x4_t*>(&sA[buf][ar][akq]) = ra0;
      *reinterpret_cast<f32x4_t*>(&sA[buf][ar][akq + 4]) = ra1;
      if constexpr (!BT) {
        *reinterpret_cast<f32x4_t*>(&sB[buf][ar][akq]) = rb[0];
        *reinterpret_cast<f32x4_t*>(&sB[buf][ar][akq + 4]) = rb[1];
      } else {
#pragma unroll
        for (int q = 0; q < NRB; ++q)
#pragma unroll
          for (int u = 0; u < 4; ++u) sB[buf][wc + 4 * q + u][wk ^ bsw(wc + 4 * q + u)] = rb[q][u];
      }
    };
    if (kdim > 0) {   // uniform
      fetch(0);
      if constexpr (NBUF == 2) {
        // buffer c & 1 holds chunk c; chunk c + 1 is fetched before and staged after chunk c's
        // MFMAs, into the buffer every wave finished reading at the previous barrier
        stage(0);
        __syncthreads();
        int buf = 0;
        for (int k0 = 0; k0 < kdim; k0 += kKc) {
          const bool more = k0 + kKc < kdim;
          if (more) fetch(k0 + kKc);
          mfma_chunk(buf);
          if (more) stage(buf ^ 1);
          __syncthreads();
          buf ^= 1;
        }
      } else {
        for (int k0 = 0; k0 < kdim; k0 += kKc) {
          stage(0);
          __syncthreads();
          if (k0 + kKc < kdim) fetch(k0 + kKc);
          mfma_chunk(0);
          __syncthreads();
        }
      }
    }
  } else {
    for (int k0 = 0; k0 < kdim; k0 += kKc) {
      if constexpr (!BT) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int kk = k0 + akq + u;
          float v = 0.f;
          if (arow && kk < kdim) {
            if constexpr (STRIDED) {
              v = abase[static_cast<int64_t>(kk) * g.d];
            } else {
              const int blk = kk / C, c = kk - blk * C;
              v = abase[static_cast<int64_t>(blk) * g.d * C + c];
            }
          }
          sA[0][ar][akq + u] = v;
          const int col = c0 + ar;
          sB[0][ar][akq + u] = (col < ncols && kk < kdim) ? g.w[static_cast<int64_t>(col) * g.k + kk] : 0.f;
        }
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int kk = k0 + akq + u;
          sA[0][ar][akq + u] = (arow && kk < kdim) ? abase[static_cast<int64_t>(kk) * g.d] : 0.f;
        }
        const int kk = k0 + wk;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int col = c0 + wc + u;
          sB[0][wc + u][wk ^ bsw(wc + u)] =
              (kk < kdim && col < ncols) ? g.w[static_cast<int64_t>(kk) * wld + col] : 0.f;
        }
      }
      __syncthreads();
      mfma_chunk(0);
      __syncthreads();
    }
  }
  // the lane's four output rows rho0 .. rho0 + 3: one division, then (n, m) stepped
  const int64_t rho0 = r0 + wave * 16 + 4 * (lane >> 4);
  int64_t n = rho0 / d;
  int m = static_cast<int>(rho0 - n * d);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if (v > 0 && ++m == d) {
      m = 0;
      ++n;
    }
    if (rho0 + v >= g.rows) continue;
    float* __restrict__ orow = FWD ? out + n * a.ywidth + g.yoff + m : out + n * a.xwidth + g.xoff + m * C;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int col = c0 + t * 16 + (lane & 15);
      if (col >= ncols) continue;
      const float val = a.alpha * acc[t][v];
      if (FWD) {
        orow[col * d] = val;
      } else {
        const int blk = col / C, c = col - blk * C;
        orow[blk * d * C + c] = val;
      }
    }
  }
}

// The maps that write y on the bf16 matrix cores, fp32 operands in three parts (split_bf16.hpp): 64 rows x TN
// columns per block (one 64 x 128 block reads each row once where the fp32 kernel's 64-column tiles read
// it twice), K in chunks of 32.  Both operands are split when a chunk is staged: a thread holds
// eight consecutive k of a row or column, one 16-byte LDS unit per part, in the operand order
// [part][octet of k][row or column]; the next chunk's loads are in flight during the current one's
// matrix instructions (two LDS buffers, one barrier per chunk).  Wave w computes rows 32 (w % 2) ..
// and columns (TN / 2) (w / 2) ..  The small part products have accumulators of their own.
// Bound by the staging between barriers at two blocks per CU.  2048 nodes, C = O = 128, counts (4, 6, 7, 6)
// (19.9 GFLOP over forward and both adjoints): 52 us, on fp32 MFMA 75 us; error against float64 1.6e-7, 5.0e-7
// there.  One LDS buffer with two barriers per chunk (three blocks per CU): 61 us.
constexpr int kSpRows = kTile + 2;       // units per octet row: staggers the staging writes' banks

template <int N>
struct SplitTile {
  bf16x8 v[3][kKc / 8][N];
};

template <int MODE, int TN>
__global__ void __launch_bounds__(256, 2)
degree_linear_split_kernel(const float* __restrict__ in, float* __restrict__ out, const LinearArgs a) {
  static_assert(MODE != kInputGrad, "degree_linear_input_grad_kernel");
  constexpr bool BT = MODE == kMulIrT;
  constexpr bool STRIDED = MODE != kForward;
  constexpr int NCT = TN / 64;           // 32-column tiles per wave
  constexpr int NBT = TN / 64;           // octets of B per thread
  const DegreeGeometry g = a.g[blockIdx.z];
  const int d = g.d;
  const int ncols = a.out_channels, kdim = g.k;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int c0 = blockIdx.y * TN;
  if (r0 >= g.rows || c0 >= ncols) return;
  __shared__ SplitTile<kSpRows> sA[2];
  __shared__ SplitTile<TN + 2> sB[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = a.channels;
  const int ar = tid >> 2, ao = tid & 3, akq = ao * 8;   // A: row ar, octet ao
  const int64_t arho = r0 + ar;
  const int64_t an = arho < g.rows ? arho / d : 0;   // rows past the end read row 0; not stored
  const int am = arho < g.rows ? static_cast<int>(arho - an * d) : 0;
  const float* __restrict__ abase = in + an * a.xwidth + g.xoff + (STRIDED ? am : static_cast<int64_t>(am) * C);
  float ra[8], rb[NBT][8];
  auto fetch = [&](int k0) {
    if constexpr (STRIDED) {
      const float* p = abase + (k0 + akq) * d;
#pragma unroll
      for (int u = 0; u < 8; ++u) ra[u] = p[u * d];
    } else {
      const int blk = k0 / C, c = k0 - blk * C + akq;
      const float* p = abase + blk * d * C + c;
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(p), hi = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
      for (int u = 0; u < 4; ++u) ra[u] = lo[u], ra[4 + u] = hi[u];
    }
#pragma unroll
    for (int q = 0; q < NBT; ++q) {
      if constexpr (!BT) {   // weight row of column 64 q + tid / 4, its octet tid % 4
        const int col = c0 + 64 * q + ar < ncols ? c0 + 64 * q + ar : ncols - 1;   // (not stored)
        const float* p = g.w + static_cast<int64_t>(col) * g.k + k0 + akq;
        const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(p), hi = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) rb[q][u] = lo[u], rb[q][4 + u] = hi[u];
      } else {               // column 64 q + tid % 64, octet tid / 64: eight weight rows
        const int col = c0 + 64 * q + (tid & 63) < ncols ? c0 + 64 * q + (tid & 63) : ncols - 1;
        const float* p = g.w + static_cast<int64_t>(k0 + 8 * (tid >> 6)) * ncols + col;
#pragma unroll
        for (int u = 0; u < 8; ++u) rb[q][u] = p[static_cast<int64_t>(u) * ncols];
      }
    }
  };
  auto stage = [&](int buf) {
    const Split8 sa = split8(ra);
#pragma unroll
    for (int q = 0; q < 3; ++q) sA[buf].v[q][ao][ar] = sa.p[q];
#pragma unroll
    for (int t = 0; t < NBT; ++t) {
      const Split8 sb = split8(rb[t]);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        if constexpr (!BT)
          sB[buf].v[q][ao][64 * t + ar] = sb.p[q];
        else
          sB[buf].v[q][tid >> 6][64 * t + (tid & 63)] = sb.p[q];
      }
    }
  };
  const int r = lane & 31, half = lane >> 5, row_t = (wave & 1) * 32, col_t = (wave >> 1) * (TN / 2);
  f32x16 hi[1][NCT], lo[1][NCT];
#pragma unroll
  for (int t = 0; t < NCT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) hi[0][t][i] = lo[0][t][i] = 0.f;
  if (kdim > 0) {   // uniform; a degree without path blocks writes its zero forward rows
    fetch(0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < kdim; k0 += kKc) {
      const bool more = k0 + kKc < kdim;
      if (more) fetch(k0 + kKc);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        Split8 av[1], bv[NCT];
#pragma unroll
        for (int q = 0; q < 3; ++q) av[0].p[q] = sA[buf].v[q][2 * k + half][row_t + r];
#pragma unroll
        for (int t = 0; t < NCT; ++t)
#pragma unroll
          for (int q = 0; q < 3; ++q) bv[t].p[q] = sB[buf].v[q][2 * k + half][col_t + 32 * t + r];
        mfma_split(av, bv, hi, lo);
      }
      if (more) stage(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }
#pragma unroll
  for (int t = 0; t < NCT; ++t) {
#pragma unroll
    for (int i = 0; i < 16; ++i) hi[0][t][i] += lo[0][t][i];
    const int col = c0 + col_t + 32 * t + r;
    const bool redo = any_nonfinite(hi[0][t]);   // see split_bf16.hpp: these results again in fp32
#pragma unroll
    for (int q = 0; q < 4; ++q) {   // four consecutive rows: one division, then (n, m) stepped
      const int64_t rho0 = r0 + row_t + mfma_row(4 * q, half);
      int64_t n = rho0 / d;
      int m = static_cast<int>(rho0 - n * d);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (v > 0 && ++m == d) {
          m = 0;
          ++n;
        }
        if (rho0 + v >= g.rows || col >= ncols) continue;
        float val = hi[0][t][4 * q + v] * kSplitUnscale;
        if (redo) {
          val = 0.f;
          for (int k = 0; k < kdim; ++k) {
            const int64_t xk = STRIDED ? static_cast<int64_t>(k) * d + m : (static_cast<int64_t>(k / C) * d + m) * C + k % C;
            const float xa = in[n * a.xwidth + g.xoff + xk];
            val = fmaf(xa, BT ? g.w[static_cast<int64_t>(k) * ncols + col] : g.w[static_cast<int64_t>(col) * g.k + k], val);
          }
        }
        val *= a.alpha;
        out[n * a.ywidth + g.yoff + static_cast<int64_t>(col) * d + m] = val;
      }
    }
  }
}

// Input adjoint on the bf16 matrix cores: gx rows = alpha gY W with a short K = O (16 KS) and many
// columns (counts C).  A wave keeps 32 gY rows split in registers (12 KS VGPRs) and walks the columns; W
// arrives in chunks of 64 columns, split into LDS once per block (one buffer, the next chunk's loads in
// flight), its columns in the order even, odd so that a lane owns two neighbouring ones and stores
// them together (256 contiguous bytes of two rows per instruction).  LinearSplit lists the launch's blocks:
// 128 rows of one degree times `chunks` column chunks.
// 2048 nodes, C = O = 128, counts (4, 6, 7, 6): 54 us, on fp32 MFMA 84 us (the six part products take 16 at the
// matrix cores' peak, the 104 MB of gx 13 at HBM's; the rest is the first loads and the last partly filled
// round of blocks); error against float64 1.6e-7, 2.0e-7 there.
struct LinearSplit {
  int64_t block0[ICTC_LINEAR_MAX_DEGREES + 1];   // first block of each degree
  int splits[ICTC_LINEAR_MAX_DEGREES];           // column splits of a degree
  int chunks, degrees;                           // column chunks per block
};

template <int KS>
__global__ void __launch_bounds__(256, 2)
degree_linear_input_grad_kernel(const float* __restrict__ gy, float* __restrict__ gx, const LinearArgs a,
                                const LinearSplit sp) {
  constexpr int K = 16 * KS, OCT = 2 * KS, PER = OCT / 4;   // octets of K; per thread and chunk
  int z = 0;
  const int64_t b = blockIdx.x;
  while (z + 1 < sp.degrees && b >= sp.block0[z + 1]) ++z;
  const DegreeGeometry g = a.g[z];
  const int64_t t = b - sp.block0[z];
  const int split = static_cast<int>(t % sp.splits[z]);
  const int d = g.d, C = a.channels;
  const int nchunks = (g.k + 63) / 64;
  const int ch0 = split * sp.chunks, ch1 = ch0 + sp.chunks < nchunks ? ch0 + sp.chunks : nchunks;
  __shared__ bf16x8 sB[3][OCT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, half = lane >> 5;
  const int64_t row0 = (t / sp.splits[z]) * 128 + wave * 32;
  float wv[PER][8];
  auto fetch = [&](int ch) {   // column tid % 64, octets tid / 64 + 4 q
    const int col = 64 * ch + (tid & 63) < g.k ? 64 * ch + (tid & 63) : g.k - 1;   // (past the end: not stored)
    const float* __restrict__ p = g.w + static_cast<int64_t>(8 * (tid >> 6)) * g.k + col;
#pragma unroll
    for (int q = 0; q < PER; ++q)
#pragma unroll
      for (int u = 0; u < 8; ++u) wv[q][u] = p[static_cast<int64_t>(32 * q + u) * g.k];
  };
  auto stage = [&]() {
    const int col = tid & 63, slot = 32 * (col & 1) + col / 2;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const Split8 s = split8(wv[q]);
#pragma unroll
      for (int p = 0; p < 3; ++p) sB[p][4 * q + (tid >> 6)][slot] = s.p[p];
    }
  };
  fetch(ch0);
  Split8 av[KS][1];
  {
    const int64_t rho = row0 + r < g.rows ? row0 + r : g.rows - 1;   // rows past the end: not stored
    const int64_t n = rho / d;
    const float* __restrict__ p = gy + n * a.ywidth + g.yoff + (rho - n * d) + 8 * half * d;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(16 * k + u) * d];
      av[k][0] = split8(v);
    }
  }
  // byte offsets of the lane's sixteen result rows from the node of the wave's first row
  const int64_t nbase = (row0 < g.rows ? row0 : 0) / d;
  const int mbase = static_cast<int>((row0 < g.rows ? row0 : 0) - nbase * d);
  float* __restrict__ obase = gx + nbase * a.xwidth + g.xoff;
  const rsrc_t ro = make_rsrc(obase, 0x7FFFFFF0u);
  uint32_t roff[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int q = mbase + mfma_row(i, half), dn = q / d;
    const bool in = row0 + mfma_row(i, half) < g.rows;
    roff[i] = in ? static_cast<uint32_t>((dn * a.xwidth + static_cast<int64_t>(q - dn * d) * C) * 4) : 0xFFFFFFF0u;
  }
  stage();
  __syncthreads();
  for (int ch = ch0; ch < ch1; ++ch) {
    const bool more = ch + 1 < ch1;
    if (more) fetch(ch + 1);
    f32x16 acc[1][2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[0][c][i] = 0.f;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      Split8 bv[2];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int p = 0; p < 3; ++p) bv[c].p[p] = sB[p][2 * k + half][32 * c + r];
      mfma_split(av[k], bv, acc, acc);
    }
    const int col = 64 * ch + 2 * r;     // the lane's columns col, col + 1 (counts C is even)
    const int blk = col / C;
    const uint32_t coff = static_cast<uint32_t>(blk * d * C + (col - blk * C)) * 4u;
    const bool redo = any_nonfinite(acc[0][0]) || any_nonfinite(acc[0][1]);   // see split_bf16.hpp: again in fp32
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      f32x2 v{acc[0][0][i] * kSplitUnscale, acc[0][1][i] * kSplitUnscale};
      if (redo) {
        v = f32x2{0.f, 0.f};
        const int64_t rho = row0 + mfma_row(i, half);
        if (rho < g.rows && col < g.k) {
          const int64_t n = rho / d;
          for (int k = 0; k < K; ++k) {
            const float y = gy[n * a.ywidth + g.yoff + static_cast<int64_t>(k) * d + (rho - n * d)];
            const float* __restrict__ w = g.w + static_cast<int64_t>(k) * g.k + col;
            v = f32x2{fmaf(y, w[0], v[0]), fmaf(y, w[1], v[1])};
          }
        }
      }
      v = f32x2{v[0] * a.alpha, v[1] * a.alpha};
      const uint32_t off = roff[i] == 0xFFFFFFF0u || col >= g.k ? 0xFFFFFFF0u : roff[i] + coff;
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), ro, off, 0, 0);
    }
    __syncthreads();
    if (more) {
      stage();
      __syncthreads();
    }
  }
}

int prepare(const ictc_degree_linear_desc* desc, const float* const* weights, float alpha, int64_t nodes,
            LinearArgs* a, int* live_degrees, int64_t* max_rows, int* max_cols, bool fwd) {
  if (desc == nullptr || weights == nullptr || nodes < 0) return ICTC_ERR_INVALID_ARGUMENT;
  if (desc->lmax < 0 || desc->lmax >= ICTC_LINEAR_MAX_DEGREES || desc->channels < 1 || desc->out_channels < 1)
    return ICTC_ERR_INVALID_ARGUMENT;
  int64_t xw = 0;
  for (int l = 0; l <= desc->lmax; ++l) {
    if (desc->counts[l] < 0) return ICTC_ERR_INVALID_ARGUMENT;
    xw += static_cast<int64_t>(desc->counts[l]) * (2 * l + 1) * desc->channels;
  }
  a->xwidth = xw;
  a->ywidth = static_cast<int64_t>(desc->out_channels) * (desc->lmax + 1) * (desc->lmax + 1);
  a->channels = desc->channels;
  a->out_channels = desc->out_channels;
  a->alpha = alpha;
  *live_degrees = desc->lmax + 1;
  *max_rows = 0;
  *max_cols = 0;
  int64_t xoff = 0;
  for (int l = 0; l <= desc->lmax; ++l) {
    DegreeGeometry& g = a->g[l];
    g.d = 2 * l + 1;
    g.rows = nodes * g.d;
    g.k = desc->counts[l] * desc->channels;
    g.xoff = xoff;
    g.yoff = static_cast<int64_t>(desc->out_channels) * l * l;
    g.w = weights[l];
    if (g.k > 0 && g.w == nullptr) return ICTC_ERR_INVALID_ARGUMENT;
    xoff += static_cast<int64_t>(g.k) * g.d;
    if (g.rows > *max_rows) *max_rows = g.rows;
    const int cols = fwd ? desc->out_channels : g.k;
    if (cols > *max_cols) *max_cols = cols;
  }
  return ICTC_OK;
}

// Blocks of an input-adjoint launch: the column chunks per block with the fewest rounds of resident
// blocks (two per CU), each costing its chunks and about two more for the block's own rows.
LinearSplit input_grad_split(const LinearArgs& a, int degrees) {
  LinearSplit best{};
  int64_t cost = INT64_MAX;
  for (int chunks = 1; chunks <= 64; ++chunks) {
    LinearSplit s{};
    s.chunks = chunks;
    s.degrees = degrees;
    int most = 0;
    for (int l = 0; l < degrees; ++l) {
      const int n = (a.g[l].k + 63) / 64;
      s.splits[l] = n == 0 ? 1 : (n + chunks - 1) / chunks;
      s.block0[l + 1] = s.block0[l] + (n == 0 ? 0 : (a.g[l].rows + 127) / 128 * s.splits[l]);
      most = n > most ? n : most;
    }
    const int64_t slots = 2 * static_cast<int64_t>(compute_units());
    const int64_t c = (s.block0[degrees] + slots - 1) / slots * ((chunks < most ? chunks : most) + 2);
    if (c < cost) cost = c, best = s;
    if (chunks >= most) break;
  }
  return best;
}

template <int MODE>
int launch(const ictc_degree_linear_desc* desc, const float* in, const float* const* weights, float alpha,
           float* out, int64_t nodes, hipStream_t stream) {
  LinearArgs a{};
  int degrees = 0, max_cols = 0;
  int64_t max_rows = 0;
  const int st = prepare(desc, weights, alpha, nodes, &a, &degrees, &max_rows, &max_cols, MODE != kInputGrad);
  if (st != ICTC_OK) return st;
  if (MODE == kMulIr || MODE == kMulIrT) {   // one channel block per degree: x mul_ir [N, C (L+1)^2]
    for (int l = 0; l <= desc->lmax; ++l)
      if (desc->counts[l] != 1) return ICTC_ERR_INVALID_ARGUMENT;
  }
  if (nodes == 0) return ICTC_OK;
  if (in == nullptr || out == nullptr) return ICTC_ERR_INVALID_ARGUMENT;
  const int64_t row_tiles = (max_rows + kTile - 1) / kTile;
  if (row_tiles > 0x7fffffff) return ICTC_ERR_UNSUPPORTED;
  // two LDS buffers for the long K of the forward (counts C), one for the short K of the others;
  // the input adjoint's vector path takes 128 columns per block (its B tile is read once per
  // 64 x 128 outputs instead of 64 x 64)
  const bool vec = desc->channels % 32 == 0 &&
                   ((MODE != kInputGrad && MODE != kMulIrT) || desc->out_channels % 32 == 0);
  constexpr int kTn = MODE == kInputGrad ? kTileIg : kTile;
  const int tn = vec ? kTn : kTile;
  const dim3 grid(static_cast<unsigned>(row_tiles), static_cast<unsigned>((max_cols + tn - 1) / tn),
                  static_cast<unsigned>(degrees));
  if (vec && MODE == kInputGrad && max_cols > 64 &&
      (desc->out_channels == 64 || desc->out_channels == 96 || desc->out_channels == 128) &&
      128 * a.xwidth * 4 < 0x40000000) {
    // The register-resident rows where its 128-row blocks give every CU one.  Counted in blocks of one
    // 64-column chunk, a single degree (d = 1: every load and store of the fp32 kernel is contiguous) has to
    // fill the chip a few times over, and up to 128 columns of more than 64 outputs whole rounds of one or two
    // blocks per CU: a CU's second block costs 6 us of 16.  us on either side of the lines, fp32 in brackets:
    // single degree, O = 128, one path block, 49,152 nodes 28.1 (27.2), 65,536 30.5 (34.1); four, 12,288 nodes
    // 29.2 (27.0), 16,384 30.0 (33.8); O = 64, four, 16,384 nodes 15.6 (14.8), 20,480 17.5 (19.0); several degrees,
    // O = 128, one path block: 256 blocks 15.8 (17.6, lmax 3), 260 21.0 (17.1, lmax 2), 320 20.9 (18.0, lmax 3),
    // 384 22.6 (24.1, lmax 2), 21.5 (18.3, lmax 3), 512 23.2 (29.8, lmax 3).
    const LinearSplit sp = input_grad_split(a, degrees);
    const int64_t cus = compute_units();
    int64_t chunked = 0;
    for (int l = 0; l < degrees; ++l) chunked += (a.g[l].rows + 127) / 128 * ((a.g[l].k + 63) / 64);
    const bool fills = degrees == 1 ? chunked > (desc->out_channels > 64 ? 3 : 2) * cus
                                    : max_cols > 128 || desc->out_channels == 64 || chunked <= cus || chunked >= 2 * cus;
    if (fills && sp.block0[degrees] >= compute_units() && sp.block0[degrees] <= 0x7fffffff) {
      const dim3 igrid(static_cast<unsigned>(sp.block0[degrees]));
      if (desc->out_channels == 64)
        hipLaunchKernelGGL(degree_linear_input_grad_kernel<4>, igrid, dim3(256), 0, stream, in, out, a, sp);
      else if (desc->out_channels == 96)
        hipLaunchKernelGGL(degree_linear_input_grad_kernel<6>, igrid, dim3(256), 0, stream, in, out, a, sp);
      else
        hipLaunchKernelGGL(degree_linear_input_grad_kernel<8>, igrid, dim3(256), 0, stream, in, out, a, sp);
      return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
    }
  }
  if constexpr (MODE != kInputGrad) {
    // Split-bf16 blocks (two per CU) where they give every CU one: fewer, larger blocks than the fp32
    // kernel's, which keeps the smaller calls.  A 64-column block stages as many rows as a 128-column one for
    // half the products, so that its K has to be long: C = O = 64, lmax 3, 4,096 nodes, one path block (K = 64)
    // 14.8 us (fp32 13.6), two (K = 128) 18.5 (18.6), four 27.0 (27.3), and at 2,048 nodes two 11.4 (15.0), four
    // 16.5 (24.4); C = O = 32, 4,096 nodes, one 10.2 (8.3), three (K = 96) 14.1 (13.2), and at 2,048 nodes three
    // 8.8 (11.3).  A single degree (d = 1: contiguous in the fp32 kernel too) starts at 5/4 of the CUs: 128 x
    // 128, 16,384 nodes 10.5 (9.2), 20,480 12.1 (12.2), 32,768 14.0 (16.5).
    const int stn = max_cols > 64 ? 128 : 64;
    int64_t blocks = 0, rows = 0, steps = 0;
    for (int l = 0; l < degrees; ++l) {
      blocks += ((a.g[l].rows + kTile - 1) / kTile) * ((a.out_channels + stn - 1) / stn);
      rows += a.g[l].k > 0 ? a.g[l].rows : 0;
      steps += a.g[l].rows * a.g[l].k;
    }
    const bool deep = stn == 128 || steps >= 96 * rows;
    if (vec && deep && 4 * blocks >= (degrees > 1 ? 4 : 5) * static_cast<int64_t>(compute_units())) {
      const dim3 sgrid(static_cast<unsigned>(row_tiles), static_cast<unsigned>((max_cols + stn - 1) / stn),
                       static_cast<unsigned>(degrees));
      if (stn == 128)
        hipLaunchKernelGGL((degree_linear_split_kernel<MODE, 128>), sgrid, dim3(256), 0, stream, in, out, a);
      else
        hipLaunchKernelGGL((degree_linear_split_kernel<MODE, 64>), sgrid, dim3(256), 0, stream, in, out, a);
      return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
    }
  }
  if (vec)
    hipLaunchKernelGGL((degree_linear_kernel<MODE, true, MODE == kForward ? 2 : 1, kTn>), grid, dim3(256), 0, stream,
                       in, out, a);
  else
    hipLaunchKernelGGL((degree_linear_kernel<MODE, false, 1, kTile>), grid, dim3(256), 0, stream, in, out, a);
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}

// Weight adjoint per degree (the dense product the layouts above otherwise need rearranged
// copies for):  gW_l[o, j] = alpha * sum_{rows rho = n d + m} gy[n, o, m] * x[rho, j], with the x
// rows of the forward (kWgIrMul: x[n, k, m, c], j = k C + c) or of the mul_ir map (kWgMulIr:
// x[n, c, m] at offset C l^2, j = c).  The rows of a degree are split into ranges (range_rows, a
// multiple of the 32-row chunk sized so that every block of the launch is resident at once: the
// LDS of three blocks fits a CU, and a second partial round of blocks would idle most CUs); a
// block of kWgWaves waves computes the 128 (o) x 64 (j) partial of one range (each wave 32 o x 32 j on
// the bf16 matrix cores, fp32 operands in three parts: split_bf16.hpp) over 32-row chunks: a thread's
// operand unit is eight rows of one column, split when the chunk is staged, the next chunk's loads in
// flight during the current chunk's matrix instructions (one LDS buffer, two barriers per chunk).  The
// partials go to the workspace; a second kernel sums the ranges in order and scales by alpha (fixed order:
// bit-identical run to run).  Rows past the end read zeros from the buffer range check (their offsets lie
// past the tensors).  2048 nodes, C = O = 128, counts (4, 6, 7, 6): 80 us with the sum, 101 us with fp32
// MFMA; error against float64 1.7e-7, 4.4e-7 there.
enum WgLayout { kWgIrMul = 0, kWgMulIr = 1 };
constexpr int kWgMinRows = 256;   // shortest range (8 chunks)
// 36,864 B of LDS and 80 VGPRs (six waves per SIMD), which spills 4 VGPRs in the ir_mul layout, 2 in mul_ir
// (20 and 12 bytes of scratch per lane)
constexpr int kWgBlocksPerCu = 3;
constexpr int kWgO = 128, kWgJ = 64;
constexpr int kWgWaves = 8;   // waves per block: 32 o x 32 j each

struct WgDegree {
  int64_t rows;     // N d
  int d, k;         // 2l + 1, output columns (counts[l] C)
  int64_t xoff, yoff;
  int ranges, otiles, jtiles;
  int64_t tile0;    // first block of the degree
  int64_t ws0;      // first workspace float of the degree: [ranges][O][k]
  float* gw;        // [O, k] or null (not asked for)
};

struct WgArgs {
  WgDegree g[ICTC_LINEAR_MAX_DEGREES];
  int degrees;
  int64_t tiles;
  int64_t xwidth, ywidth;
  int C, O;
  int range_rows;
  float alpha;
  uint32_t xbytes, ybytes;
};

template <int LAYOUT>
__global__ void __launch_bounds__(64 * kWgWaves, 6)
degree_linear_wgrad_kernel(const float* __restrict__ gy, const float* __restrict__ x, float* __restrict__ ws,
                           const WgArgs a) {
  // XCD-contiguous block order: the column tiles of one row range (which read the same gY rows)
  // run on one XCD and share its L2
  const int64_t b = xcd_block(blockIdx.x, gridDim.x);
  int z = 0;
  while (z + 1 < a.degrees && b >= a.g[z + 1].tile0) ++z;
  const WgDegree g = a.g[z];
  if (g.gw == nullptr) return;   // uniform: the degree's gradient is not asked for
  const int64_t t = b - g.tile0;
  const int ot = static_cast<int>(t % g.otiles);
  const int64_t rest = t / g.otiles;
  const int jt = static_cast<int>(rest % g.jtiles);
  const int range = static_cast<int>(rest / g.jtiles);
  const int o0 = ot * kWgO, j0 = jt * kWgJ;
  const int64_t r0 = static_cast<int64_t>(range) * a.range_rows;
  const int64_t r1 = r0 + a.range_rows < g.rows ? r0 + a.range_rows : g.rows;
  const int d = g.d, C = a.C, O = a.O;
  __shared__ SplitTile<kWgO> sA;
  __shared__ SplitTile<kWgJ> sB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const rsrc_t ry = make_rsrc(gy, a.ybytes), rx = make_rsrc(x, a.xbytes);
  // A units: column (o) tid % 128, rows 8 (tid / 128) ..; o past O (or past the tile) reads o = 0 of
  // its row: those accumulator rows are never stored.  B units, the first four waves: column (j)
  // tid % 64, rows 8 (tid / 64) ..; j past k reads column 0.
  const bool hasb = wave < 4;   // wave-uniform
  const int ao = tid & (kWgO - 1), aoct = tid / kWgO, bj = tid & (kWgJ - 1), boct = tid / kWgJ;
  const int aoc = o0 + ao < O ? o0 + ao : 0;
  const int bjc = j0 + bj < g.k ? j0 + bj : 0;
  uint32_t bcol;   // byte offset of column bjc inside a row's degree block (m = 0)
  if constexpr (LAYOUT == kWgIrMul) {
    const int blk = bjc / C, c = bjc - blk * C;
    bcol = static_cast<uint32_t>(blk * d * C + c) * 4u;
  } else {
    bcol = static_cast<uint32_t>(bjc * d) * 4u;
  }
  // Row rho = n d + m of a chunk starting at c0 = n0 d + m0: the row q of the chunk has
  // n = n0 + (m0 + q) / d, computed as floor((m0 + q + 0.5) / d) in float (exact: m0 + q < 47 and
  // the rounding error is far below 0.5 / d).  Offsets are 32-bit bytes (tensors below 2 GiB).
  const float inv_d = 1.f / static_cast<float>(d);
  const uint32_t yw4 = static_cast<uint32_t>(a.ywidth) * 4u, xw4 = static_cast<uint32_t>(a.xwidth) * 4u;
  const uint32_t yo4 = static_cast<uint32_t>(g.yoff) * 4u + static_cast<uint32_t>(aoc * d) * 4u;
  const uint32_t xo4 = static_cast<uint32_t>(g.xoff) * 4u + bcol;
  const uint32_t mstep = (LAYOUT == kWgIrMul ? static_cast<uint32_t>(C) : 1u) * 4u;
  float ra[8], rb[8];
  // eight rows of one column, from row c0 + first of the degree: offset n * width + base + m * step
  // (rows past r1 belong to the next range or lie past the end: an out-of-range offset reads 0)
  auto octet = [&](rsrc_t rs, int64_t c0, int first, uint32_t width, uint32_t base, uint32_t step, float (&v)[8]) {
    const int n0 = static_cast<int>(c0 / d), m0 = static_cast<int>(c0 - static_cast<int64_t>(n0) * d);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q = m0 + first + i;
      const int dn = static_cast<int>((static_cast<float>(q) + 0.5f) * inv_d), m = q - dn * d;
      const uint32_t off = static_cast<uint32_t>(n0 + dn) * width + base + static_cast<uint32_t>(m) * step;
      v[i] = buf_load<1>(rs, c0 + first + i < r1 ? off : 0xFFFFFFF0u).v[0];
    }
  };
  auto fetch = [&](int64_t c0) {
    octet(ry, c0, 8 * aoct, yw4, yo4, 4u, ra);
    if (hasb) octet(rx, c0, 8 * boct, xw4, xo4, mstep, rb);
  };
  const int r = lane & 31, half = lane >> 5, o_t = (wave & 3) * 32, j_t = (wave >> 2) * 32;
  const bool work = o0 + o_t < O && j0 + j_t < g.k;   // wave-uniform: any result to store
  f32x16 acc[1][1], lo[1][1];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][0][i] = lo[0][0][i] = 0.f;
  fetch(r0);
  for (int64_t c0 = r0; c0 < r1; c0 += 32) {
    const Split8 va = split8(ra);
#pragma unroll
    for (int q = 0; q < 3; ++q) sA.v[q][aoct][ao] = va.p[q];
    if (hasb) {
      const Split8 vb = split8(rb);
#pragma unroll
      for (int q = 0; q < 3; ++q) sB.v[q][boct][bj] = vb.p[q];
    }
    __syncthreads();
    if (c0 + 32 < r1) fetch(c0 + 32);
    if (work) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        Split8 av[1], bv[1];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          av[0].p[q] = sA.v[q][2 * k + half][o_t + r];
          bv[0].p[q] = sB.v[q][2 * k + half][j_t + r];
        }
        mfma_split(av, bv, acc, lo);
      }
    }
    __syncthreads();
  }
  float* __restrict__ part = ws + g.ws0 + static_cast<int64_t>(range) * O * g.k;
  const int j = j0 + j_t + r;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][0][i] += lo[0][0][i];
  const bool redo = any_nonfinite(acc[0][0]);   // see split_bf16.hpp: these results again in fp32
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int o = o0 + o_t + mfma_row(i, half);
    if (o >= O || j >= g.k) continue;
    float v = acc[0][0][i] * kSplitUnscale;
    if (redo) {
      v = 0.f;
      for (int64_t rho = r0; rho < r1; ++rho) {
        const int64_t n = rho / d, m = rho - n * d;
        const int64_t xj = LAYOUT == kWgIrMul ? (static_cast<int64_t>(j / C) * d + m) * C + j % C
                                              : static_cast<int64_t>(j) * d + m;
        v = fmaf(gy[n * a.ywidth + g.yoff + static_cast<int64_t>(o) * d + m], x[n * a.xwidth + g.xoff + xj], v);
      }
    }
    part[static_cast<int64_t>(o) * g.k + j] = v;
  }
}

// gW_l = alpha * the sum of the degree's range partials, in range order (one thread per entry).
__global__ void __launch_bounds__(256) degree_linear_wgrad_sum_kernel(const float* __restrict__ ws, const WgArgs a,
                                                                      int64_t entries) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < entries;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    int64_t base = 0;
    int z = 0;
    for (; z < a.degrees; ++z) {
      const int64_t n = static_cast<int64_t>(a.O) * a.g[z].k;
      if (i < base + n) break;
      base += n;
    }
    const WgDegree& g = a.g[z];
    if (g.gw == nullptr) continue;
    const int64_t e = i - base, stride = static_cast<int64_t>(a.O) * g.k;
    const float* p = ws + g.ws0 + e;
    float s = 0.f;
    int r = 0;
    for (; r + 4 <= g.ranges; r += 4) {   // four loads in flight, added in range order
      const float v0 = p[r * stride], v1 = p[(r + 1) * stride], v2 = p[(r + 2) * stride], v3 = p[(r + 3) * stride];
      s = (((s + v0) + v1) + v2) + v3;
    }
    for (; r < g.ranges; ++r) s += p[r * stride];
    g.gw[e] = a.alpha * s;
  }
}

// Workspace floats of one weight-adjoint call, and the launch geometry (0 for an empty call).
int wgrad_prepare(const ictc_degree_linear_desc* desc, int layout, float alpha, int64_t nodes, float* const* grad_w,
                  WgArgs* a, int64_t* ws_floats, int64_t* entries) {
  if (desc == nullptr || nodes < 0 || (layout != kWgIrMul && layout != kWgMulIr)) return ICTC_ERR_INVALID_ARGUMENT;
  if (desc->lmax < 0 || desc->lmax >= ICTC_LINEAR_MAX_DEGREES || desc->channels < 1 || desc->out_channels < 1)
    return ICTC_ERR_INVALID_ARGUMENT;
  *a = WgArgs{};
  a->degrees = desc->lmax + 1;
  a->C = desc->channels;
  a->O = desc->out_channels;
  a->alpha = alpha;
  int64_t xw = 0;
  for (int l = 0; l <= desc->lmax; ++l) {
    if (desc->counts[l] < 0) return ICTC_ERR_INVALID_ARGUMENT;
    if (layout == kWgMulIr && desc->counts[l] != 1) return ICTC_ERR_INVALID_ARGUMENT;
    xw += static_cast<int64_t>(desc->counts[l]) * (2 * l + 1) * desc->channels;
  }
  a->xwidth = xw;
  a->ywidth = static_cast<int64_t>(desc->out_channels) * (desc->lmax + 1) * (desc->lmax + 1);
  const int64_t xb = nodes * a->xwidth * 4, yb = nodes * a->ywidth * 4;
  if (xb >= 0x7FFFFFF0 || yb >= 0x7FFFFFF0) return ICTC_ERR_UNSUPPORTED;   // 32-bit buffer offsets
  a->xbytes = static_cast<uint32_t>(xb);
  a->ybytes = static_cast<uint32_t>(yb);
  int64_t xoff = 0, work = 0, columns = 0;
  for (int l = 0; l <= desc->lmax; ++l) {
    WgDegree& g = a->g[l];
    g.d = 2 * l + 1;
    g.rows = nodes * g.d;
    g.k = desc->counts[l] * desc->channels;
    g.xoff = layout == kWgIrMul ? xoff : static_cast<int64_t>(desc->channels) * l * l;
    g.yoff = static_cast<int64_t>(desc->out_channels) * l * l;
    g.gw = g.k > 0 ? grad_w[l] : nullptr;
    xoff += static_cast<int64_t>(g.k) * g.d;
    g.otiles = (desc->out_channels + kWgO - 1) / kWgO;
    g.jtiles = (g.k + kWgJ - 1) / kWgJ;
    if (g.gw) {
      work += g.rows * g.otiles * g.jtiles;
      columns += static_cast<int64_t>(g.otiles) * g.jtiles;
    }
  }
  // ranges: blocks = sum ceil(rows / R) tiles <= work / R + columns <= the resident capacity
  const int64_t room = static_cast<int64_t>(kWgBlocksPerCu) * compute_units() - columns;
  int64_t rr = room > 0 ? (work + room - 1) / room : work;
  rr = (rr + 31) / 32 * 32;
  a->range_rows = static_cast<int>(rr < kWgMinRows ? kWgMinRows : (rr > (1 << 30) ? (1 << 30) : rr));
  int64_t tiles = 0, ws = 0, ent = 0;
  for (int l = 0; l <= desc->lmax; ++l) {
    WgDegree& g = a->g[l];
    g.ranges = g.gw ? static_cast<int>((g.rows + a->range_rows - 1) / a->range_rows) : 0;
    g.tile0 = tiles;
    g.ws0 = ws;
    tiles += static_cast<int64_t>(g.ranges) * g.otiles * g.jtiles;
    ws += static_cast<int64_t>(g.ranges) * desc->out_channels * g.k;
    ent += static_cast<int64_t>(desc->out_channels) * g.k;
  }
  a->tiles = tiles;
  *ws_floats = ws;
  *entries = ent;
  return ICTC_OK;
}

}  // namespace
}  // namespace ictc

extern "C" {

int ictc_hip_degree_linear_forward(const ictc_degree_linear_desc* desc, const float* x, const float* const* weights,
                                   float alpha, float* y, int64_t nodes, hipStream_t stream) {
  return ictc::launch<ictc::kForward>(desc, x, weights, alpha, y, nodes, stream);
}

int ictc_hip_degree_linear_input_grad(const ictc_degree_linear_desc* desc, const float* grad_y,
                                      const float* const* weights, float alpha, float* grad_x, int64_t nodes,
                                      hipStream_t stream) {
  return ictc::launch<ictc::kInputGrad>(desc, grad_y, weights, alpha, grad_x, nodes, stream);
}

int ictc_hip_degree_linear_mul_ir(const ictc_degree_linear_desc* desc, const float* x, const float* const* weights,
                                  float alpha, float* y, int64_t nodes, hipStream_t stream) {
  return ictc::launch<ictc::kMulIr>(desc, x, weights, alpha, y, nodes, stream);
}

int ictc_hip_degree_linear_mul_ir_transposed(const ictc_degree_linear_desc* desc, const float* x,
                                             const float* const* weights, float alpha, float* y, int64_t nodes,
                                             hipStream_t stream) {
  return ictc::launch<ictc::kMulIrT>(desc, x, weights, alpha, y, nodes, stream);
}

int64_t ictc_hip_degree_linear_weight_grad_workspace(const ictc_degree_linear_desc* desc, int x_layout,
                                                     int64_t nodes) {
  float* none[ICTC_LINEAR_MAX_DEGREES];
  float dummy = 0.f;
  for (int l = 0; l < ICTC_LINEAR_MAX_DEGREES; ++l) none[l] = &dummy;   // every degree asked for
  ictc::WgArgs a;
  int64_t ws = 0, entries = 0;
  const int st = ictc::wgrad_prepare(desc, x_layout, 1.f, nodes, none, &a, &ws, &entries);
  return st == ICTC_OK ? ws : -static_cast<int64_t>(st);
}

int ictc_hip_degree_linear_weight_grad(const ictc_degree_linear_desc* desc, int x_layout, const float* grad_y,
                                       const float* x, float alpha, float* workspace, int64_t workspace_floats,
                                       float* const* grad_weights, int64_t nodes, hipStream_t stream) {
  if (grad_weights == nullptr) return ICTC_ERR_INVALID_ARGUMENT;
  ictc::WgArgs a;
  int64_t ws = 0, entries = 0;
  const int st = ictc::wgrad_prepare(desc, x_layout, alpha, nodes, grad_weights, &a, &ws, &entries);
  if (st != ICTC_OK) return st;
  if (entries == 0) return ICTC_OK;
  // no rows: no ranges, and the sum kernel writes zero gradients
  if (nodes > 0 && (grad_y == nullptr || x == nullptr || workspace == nullptr || workspace_floats < ws))
    return ICTC_ERR_INVALID_ARGUMENT;
  if (a.tiles > 0x7fffffff) return ICTC_ERR_UNSUPPORTED;
  if (a.tiles > 0) {
    if (x_layout == ictc::kWgIrMul)
      hipLaunchKernelGGL(ictc::degree_linear_wgrad_kernel<ictc::kWgIrMul>, dim3(static_cast<unsigned>(a.tiles)),
                         dim3(64 * ictc::kWgWaves), 0, stream, grad_y, x, workspace, a);
    else
      hipLaunchKernelGGL(ictc::degree_linear_wgrad_kernel<ictc::kWgMulIr>, dim3(static_cast<unsigned>(a.tiles)),
                         dim3(64 * ictc::kWgWaves), 0, stream, grad_y, x, workspace, a);
    if (hipGetLastError() != hipSuccess) return ICTC_ERR_LAUNCH;
  }
  const int64_t blocks = (entries + 255) / 256;
  hipLaunchKernelGGL(ictc::degree_linear_wgrad_sum_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)),
                     dim3(256), 0, stream, workspace, a, entries);
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}

}  // extern "C"
