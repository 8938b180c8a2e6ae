// extern "C" entry points of the symmetric-contraction family; per-configuration
// instantiations are compiled in generated/sc_inst_*.hip.
#include "sc_kernels.hpp"

namespace ictc {
#define ICTC_SC(L, T, K, KTOT)                                                                     \
  extern template int launch_sc<L, T, K>(int, const float*, const float*, const int64_t*, const float*,   \
                                         const float*, float*, int, int64_t, int, hipStream_t);           \
  extern template int launch_sc_weight_grad<L, T, K>(const float*, const float*, const int64_t*, const int32_t*, \
                                                     const float*, float*, int, int64_t, int, int64_t, int,      \
                                                     hipStream_t);
#include "generated/sc_instances.def"
#undef ICTC_SC

using ScWeightGrad = int (*)(const float*, const float*, const int64_t*, const int32_t*, const float*, float*, int,
                             int64_t, int, int64_t, int, hipStream_t);
using ScLaunch = int (*)(int, const float*, const float*, const int64_t*, const float*, const float*, float*,
                         int, int64_t, int, hipStream_t);
struct ScEntry {
  ScLaunch fn;
  ScWeightGrad weight_grad;
  int ktot;
};
#define ICTC_SC(L, T, K, KTOT) [L * 16 + T * 4 + K] = {&launch_sc<L, T, K>, &launch_sc_weight_grad<L, T, K>, KTOT},
const ScEntry kSc[64] = {
#include "generated/sc_instances.def"
};
#undef ICTC_SC

inline const ScEntry* sc_entry(int lmax, int target, int corr) {
  if (lmax < 0 || lmax > 3 || target < 0 || target > lmax || corr < 1 || corr > 3) return nullptr;
  const ScEntry* e = &kSc[lmax * 16 + target * 4 + corr];
  return e->fn ? e : nullptr;
}

// modes: 0 forward, 1 VJP, 2 weight features, 3 JVP, 4 Hessian-vector, 5 weight-feature JVP
inline int sc_call(int mode, int lmax, int target, int corr, int channels, const float* x, const float* t,
                   const int64_t* species, const float* w, int num_species, const float* u, float* out,
                   int64_t nodes, hipStream_t stream) {
  const ScEntry* e = sc_entry(lmax, target, corr);
  if (e == nullptr) return ICTC_ERR_UNSUPPORTED;
  if (channels < 1 || nodes < 0 || num_species < 1) return ICTC_ERR_INVALID_ARGUMENT;
  if (nodes == 0) return ICTC_OK;
  const bool needs_w = mode != 2 && mode != 5, needs_u = mode != 0 && mode != 3, needs_t = mode >= 3;
  if (!x || !species || !out || (needs_w && !w) || (needs_u && !u) || (needs_t && !t))
    return ICTC_ERR_INVALID_ARGUMENT;
  return e->fn(mode, x, t, species, w, u, out, channels, nodes, num_species, stream);
}

// Nodes ordered by species (stable) and each species' first position: block s counts the nodes of lower
// species, then places its own in node order.  Every block reads all species indices (four per
// thread and step, L2 after the first block); an index outside [0, S) counts as species 0, as in the
// contraction kernels.
constexpr int kOrderThreads = 1024;
constexpr int kOrderWaves = kOrderThreads / kWave;

__global__ void __launch_bounds__(kOrderThreads)
sc_species_order_kernel(const int64_t* __restrict__ species, int64_t nodes, int num_species,
                        int32_t* __restrict__ order, int32_t* __restrict__ start) {
  __shared__ int part[kOrderWaves];
  const int s = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  auto at = [&](int64_t i) -> int {
    const int64_t v = species[i];
    return v < 0 || v >= num_species ? 0 : static_cast<int>(v);
  };
  // sum over the block, the same on every thread
  auto block_sum = [&](int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    if (lane == 0) part[wave] = v;
    __syncthreads();
    int total = 0;
    for (int w = 0; w < kOrderWaves; ++w) total += part[w];
    __syncthreads();
    return total;
  };
  int lower = 0;
  for (int64_t i = tid; i < nodes; i += kOrderThreads) lower += at(i) < s;
  int base = block_sum(lower);
  if (tid == 0) start[s] = base;
  if (tid == 0 && s == num_species - 1) start[num_species] = static_cast<int32_t>(nodes);
  for (int64_t i0 = 0; i0 < nodes; i0 += 4 * kOrderThreads) {
    bool mine[4];
    int count = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t i = i0 + 4 * tid + q;
      mine[q] = i < nodes && at(i) == s;
      count += mine[q];
    }
    int before = count;   // inclusive scan over the wave
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int v = __shfl_up(before, off, kWave);
      if (lane >= off) before += v;
    }
    if (lane == kWave - 1) part[wave] = before;
    __syncthreads();
    int total = 0, first = base + before - count;
    for (int w = 0; w < kOrderWaves; ++w) {
      if (w < wave) first += part[w];
      total += part[w];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (mine[q]) order[first++] = static_cast<int32_t>(i0 + 4 * tid + q);
    base += total;
  }
}

// out[s, :] = sum of the partial slots of species s (r + s for the ranges r that hold its nodes), in order.
__global__ void __launch_bounds__(256)
sc_weight_sum_kernel(const float* __restrict__ ws, const int32_t* __restrict__ start, int per_range, int64_t width,
                     float* __restrict__ out) {
  const int s = blockIdx.y;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (j >= width) return;
  const int first = start[s], last = start[s + 1] - 1;
  float v = 0.f;
  if (last >= first) {
    const int r1 = last / per_range;
    int r = first / per_range;
    const float* __restrict__ p = ws + (static_cast<int64_t>(r) + s) * width + j;
    for (; r + 3 <= r1; r += 4, p += 4 * width) {   // four loads in flight, added in order
      const float a = p[0], b = p[width], c = p[2 * width], d = p[3 * width];
      v = (((v + a) + b) + c) + d;
    }
    for (; r <= r1; ++r, p += width) v += p[0];
  }
  out[s * width + j] = v;
}

// Workspace of a weight-gradient call, in floats: the partial slots, the node order, the species starts.
struct ScWgSpace {
  int64_t ranges, per_range, slots, floats;
};

ScWgSpace sc_wg_space(const ScEntry& e, int channels, int num_species, int64_t nodes) {
  ScWgSpace w;
  const int64_t r = sc_wg_ranges(e.ktot, channels, nodes);
  w.per_range = nodes > r ? (nodes + r - 1) / r : 1;
  w.ranges = (nodes + w.per_range - 1) / w.per_range;   // every launched range holds nodes
  w.slots = w.ranges + num_species;
  w.floats = w.slots * e.ktot * channels + nodes + num_species + 1;
  return w;
}

}  // namespace ictc

extern "C" {

int ictc_hip_sc_weight_columns(int lmax, int target_lmax, int correlation) {
  const ictc::ScEntry* e = ictc::sc_entry(lmax, target_lmax, correlation);
  return e ? e->ktot : -1;
}

int ictc_hip_sc_forward(int lmax, int target_lmax, int correlation, int channels, const float* node_features,
                        const int64_t* species, const float* weights, int num_elements, float* out,
                        int64_t nodes, hipStream_t stream) {
  return ictc::sc_call(0, lmax, target_lmax, correlation, channels, node_features, nullptr, species, weights,
                       num_elements, nullptr, out, nodes, stream);
}

int ictc_hip_sc_backward(int lmax, int target_lmax, int correlation, int channels, const float* node_features,
                         const int64_t* species, const float* weights, int num_elements, const float* grad_out,
                         float* grad_features, int64_t nodes, hipStream_t stream) {
  return ictc::sc_call(1, lmax, target_lmax, correlation, channels, node_features, nullptr, species, weights,
                       num_elements, grad_out, grad_features, nodes, stream);
}

int ictc_hip_sc_weight_features(int lmax, int target_lmax, int correlation, int channels,
                                const float* node_features, const int64_t* species, int num_elements,
                                const float* grad_out, float* features_out, int64_t nodes,
                                hipStream_t stream) {
  return ictc::sc_call(2, lmax, target_lmax, correlation, channels, node_features, nullptr, species, nullptr,
                       num_elements, grad_out, features_out, nodes, stream);
}

int ictc_hip_sc_jvp(int lmax, int target_lmax, int correlation, int channels, const float* node_features,
                    const int64_t* species, const float* weights, int num_elements, const float* tangent,
                    float* out, int64_t nodes, hipStream_t stream) {
  return ictc::sc_call(3, lmax, target_lmax, correlation, channels, node_features, tangent, species, weights,
                       num_elements, nullptr, out, nodes, stream);
}

int ictc_hip_sc_hvp(int lmax, int target_lmax, int correlation, int channels, const float* node_features,
                    const int64_t* species, const float* weights, int num_elements, const float* grad_out,
                    const float* tangent, float* grad_features, int64_t nodes, hipStream_t stream) {
  return ictc::sc_call(4, lmax, target_lmax, correlation, channels, node_features, tangent, species, weights,
                       num_elements, grad_out, grad_features, nodes, stream);
}

int ictc_hip_sc_weight_features_jvp(int lmax, int target_lmax, int correlation, int channels,
                                    const float* node_features, const int64_t* species, int num_elements,
                                    const float* grad_out, const float* tangent, float* features_out,
                                    int64_t nodes, hipStream_t stream) {
  return ictc::sc_call(5, lmax, target_lmax, correlation, channels, node_features, tangent, species, nullptr,
                       num_elements, grad_out, features_out, nodes, stream);
}

int64_t ictc_hip_sc_weight_grad_workspace(int lmax, int target_lmax, int correlation, int channels, int num_elements,
                                          int64_t nodes) {
  const ictc::ScEntry* e = ictc::sc_entry(lmax, target_lmax, correlation);
  if (e == nullptr || channels < 1 || num_elements < 1 || num_elements > 65535 || nodes < 0 || nodes > 0x7fffffff)
    return -ICTC_ERR_INVALID_ARGUMENT;
  if (e->ktot > ictc::kScWgColumns) return 0;
  return ictc::sc_wg_space(*e, channels, num_elements, nodes).floats;
}

int ictc_hip_sc_weight_grad(int lmax, int target_lmax, int correlation, int channels, const float* node_features,
                            const int64_t* species, int num_elements, const float* grad_out, const float* tangent,
                            float* workspace, int64_t workspace_floats, float* grad_weights, int64_t nodes,
                            hipStream_t stream) {
  using namespace ictc;
  const int64_t need = ictc_hip_sc_weight_grad_workspace(lmax, target_lmax, correlation, channels, num_elements, nodes);
  if (need < 0) return ICTC_ERR_INVALID_ARGUMENT;
  if (need == 0) return ICTC_ERR_UNSUPPORTED;
  if (!grad_weights || !workspace || workspace_floats < need) return ICTC_ERR_INVALID_ARGUMENT;
  if (nodes > 0 && (!node_features || !species || !grad_out)) return ICTC_ERR_INVALID_ARGUMENT;
  const ScEntry& e = *sc_entry(lmax, target_lmax, correlation);
  const int64_t width = static_cast<int64_t>(e.ktot) * channels;
  const ScWgSpace w = sc_wg_space(e, channels, num_elements, nodes);
  int32_t* order = reinterpret_cast<int32_t*>(workspace + w.slots * width);
  int32_t* start = order + nodes;
  hipLaunchKernelGGL(sc_species_order_kernel, dim3(static_cast<unsigned>(num_elements)), dim3(kOrderThreads), 0, stream,
                     species, nodes, num_elements, order, start);
  if (hipGetLastError() != hipSuccess) return ICTC_ERR_LAUNCH;
  if (nodes > 0) {   // (no nodes: empty species ranges, zero sums)
    const int st = e.weight_grad(node_features, tangent, species, order, grad_out, workspace, channels, nodes,
                                 num_elements, w.ranges, static_cast<int>(w.per_range), stream);
    if (st != ICTC_OK) return st;
  }
  const dim3 grid(static_cast<unsigned>((width + 255) / 256), static_cast<unsigned>(num_elements));
  hipLaunchKernelGGL(sc_weight_sum_kernel, grid, dim3(256), 0, stream, workspace, start,
                     static_cast<int>(w.per_range), width, grad_weights);
  return hipGetLastError() == hipSuccess ? ICTC_OK : ICTC_ERR_LAUNCH;
}

}  // extern "C"
