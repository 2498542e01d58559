// weighted.hip -- weighted PageRank, its adjoint solve and the gradient assembly (no counterpart in the reference).
//
// Transition probabilities P[u,v] = w_uv / W_u with FP32 edge weights w and FP64 out-weight sums W_u.
//   forward  (pull over the in-CSR):  r_v   <- (1-a) s_v + a * sum_{u in in(v)}  w_uv * (r_u / W_u)
//   adjoint  (pull over the out-CSR): lam_u <- g_u + (a / W_u) * sum_{v in out(u)} w_uv * lam_v
// i.e. (I - a P^T) r = (1-a) s and its transpose (I - a P) lam = g, both by the same Jacobi pull with the convergence
// control of the rank update (fused L-inf, device-side stop). The solves run on the degree-ordered layout (its in-CSR
// forward, its out-CSR for the adjoint), with the weights carried to layout slots through layout_edge_map_kernel, so
// that the most-gathered values share cache lines as in the rank update. The gradient of L(r) follows without storing
// per-edge terms: dL/ds = (1-a) lam and dL/dw_uv = (a r_u / W_u) (lam_v - (lam_u - g_u)/a), where (lam_u - g_u)/a =
// sum_v P[u,v] lam_v is recomputed from the adjoint fixed point.
#include "prh_device.hpp"
#include "prh_internal.hpp"

namespace prh {
namespace {

template <bool ADJOINT>
__device__ __forceinline__ double wfinish(const WeightedArgs &A, uint32_t i, double sum) {
  double a;
  if constexpr (ADJOINT) {
    a = fma(A.P / A.W[i], sum, A.term[i]);
    A.z_new[i] = a;
  } else {
    a = fma(A.P, sum, (1 - A.P) * A.term[i]);
    A.z_new[i] = a / A.W[i];
  }
  A.x_new[i] = a;
  return fabs(a - A.x_old[i]);
}

// Sum of w z over edges i, i + STEP, ... < n of the row whose edges start at b, U of them in flight: a batch costs two
// round trips, and two at a time left a wave's row of 4096 edges a chain of 64.
template <int STEP, int U>
__device__ __forceinline__ double wgather(const WeightedArgs &A, uint32_t b, uint32_t i, uint32_t n) {
  const uint32_t *idx = A.idx + b;
  const float *w = A.w + b;
  double s0 = 0.0, s1 = 0.0;
  for (; i < n; i += U * STEP) {
    uint32_t u[U];
    float f[U];
    double x[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const bool in = i + k * STEP < n;
      u[k] = in ? idx[i + k * STEP] : 0u;
      f[k] = in ? w[i + k * STEP] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) x[k] = i + k * STEP < n ? A.z[u[k]] : 0.0;
#pragma unroll
    for (int k = 0; k < U; k += 2) {
      s0 += double(f[k]) * x[k];
      if (k + 1 < U) s1 += double(f[k + 1]) * x[k + 1];
    }
  }
  return s0 + s1;
}

// Rows order[rb .. re) of one band, W lanes per row, 64/W rows per wave per round.
template <bool ADJOINT, int W>
__device__ __forceinline__ void band_rows(const WeightedArgs &A, uint32_t rb, uint32_t re, double &emax) {
  constexpr int G = kWave / W;
  const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const int g = lane / W, j = lane % W;
  for (uint32_t i0 = rb + w * G; i0 < re; i0 += kWavesPerBlock * G) {  // wave-uniform
    const uint32_t i = i0 + g;
    double s = 0.0;
    uint32_t v = 0;
    if (i < re) {
      v = A.sched.order[i];
      const uint32_t b = A.off[v];
      s = wgather<W, 2>(A, b, j, A.off[v + 1] - b);
    }
    s = group_sum<W>(s);
    if (i < re && j == 0) emax = fmax(emax, wfinish<ADJOINT>(A, v, s));
  }
}

// One Jacobi step. Blocks [0, n_chunks) sum one chunk of a heavy row each (its partial); the next nb_high blocks
// take the rows of degree in (64, kWeightedChunk], a wave per row; the rest the low-row bands. Fused L-inf for the
// rows finished here.
template <bool ADJOINT>
__global__ __launch_bounds__(kBlock) void weighted_step_kernel(WeightedArgs A, uint32_t nb_high, LoopCtl ctl) {
  if (!iteration_begin(ctl)) return;
  __shared__ double lds[kWavesPerBlock];
  const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (blockIdx.x < A.n_chunks) {  // block-uniform
    const uint32_t cb = A.chunk_beg[blockIdx.x];
    const double s = group_sum<kWave>(wgather<kBlock, 8>(A, cb, threadIdx.x, A.chunk_end[blockIdx.x] - cb));
    if (lane == 0) lds[w] = s;
    __syncthreads();
    if (threadIdx.x == 0) A.partial[blockIdx.x] = (lds[0] + lds[1]) + (lds[2] + lds[3]);
    report_begun(ctl);
    return;
  }
  const uint32_t b = blockIdx.x - A.n_chunks;
  double emax = 0.0;
  if (b < nb_high) {
    const uint32_t *order = A.sched.order + A.sched.n_low;
    const uint32_t n = A.sched.n_high;
    for (uint32_t i = b * kWavesPerBlock + w; i < n; i += nb_high * kWavesPerBlock) {
      const uint32_t v = order[i];
      const uint32_t rb = A.off[v];
      const double s = group_sum<kWave>(wgather<kWave, 8>(A, rb, lane, A.off[v + 1] - rb));
      if (lane == 0) emax = fmax(emax, wfinish<ADJOINT>(A, v, s));
    }
  } else {
    const uint32_t lb = b - nb_high;
    int k = 0;
    while (k + 1 < A.n_bands && lb >= A.band[k + 1].block_begin) ++k;
    const RankSection &S = A.band[k];
    const uint32_t rb = S.begin + (lb - S.block_begin) * S.per_block;
    const uint32_t re = min(S.end, rb + S.per_block);
    switch (S.width) {
      case 32: band_rows<ADJOINT, 32>(A, rb, re, emax); break;
      case 16: band_rows<ADJOINT, 16>(A, rb, re, emax); break;
      case 8: band_rows<ADJOINT, 8>(A, rb, re, emax); break;
      case 4: band_rows<ADJOINT, 4>(A, rb, re, emax); break;
      case 2: band_rows<ADJOINT, 2>(A, rb, re, emax); break;
      default: band_rows<ADJOINT, 1>(A, rb, re, emax); break;
    }
  }
  report_change(ctl, emax);
  report_begun(ctl);
}

// Heavy rows, after the step of the same iteration: a wave per row adds its chunk sums in chunk order.
template <bool ADJOINT>
__global__ __launch_bounds__(kBlock) void weighted_heavy_kernel(WeightedArgs A, LoopCtl ctl) {
  if (!iteration_begin(ctl)) return;
  const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const uint32_t *order = A.sched.order + A.sched.n_low + A.sched.n_high;
  double emax = 0.0;
  for (uint32_t h = blockIdx.x * kWavesPerBlock + w; h < A.sched.n_huge; h += gridDim.x * kWavesPerBlock) {
    double s = 0.0;
    for (uint32_t k = A.heavy_first[h] + lane; k < A.heavy_first[h + 1]; k += kWave) s += A.partial[k];
    s = group_sum<kWave>(s);
    if (lane == 0) emax = fmax(emax, wfinish<ADJOINT>(A, order[h], s));
  }
  report_change(ctl, emax);
}

// Sum of w[i], w[i + STEP], ... below n, eight loads in flight.
template <int STEP>
__device__ __forceinline__ double weight_sum(const float *w, uint32_t i, uint32_t n) {
  double s0 = 0.0, s1 = 0.0;
  for (; i < n; i += 8 * STEP) {
    float f[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] = i + k * STEP < n ? w[i + k * STEP] : 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      s0 += double(f[k]);
      s1 += double(f[k + 1]);
    }
  }
  return s0 + s1;
}

// W_u = sum of u's out-weights (FP64): a lane, a wave or a workgroup per row by its class in `order` (the rows
// partitioned by out-degree: counts[0] up to kSumLane, counts[1] up to kSumWave, counts[2] heavier; device words). The
// first nb_hub workgroups take the heaviest rows, the next nb_wave the middle ones. With a wave for every row and one
// load in flight the hubs set the time: 1M vertices, 17M edges 897 -> 58 us, and 16 us for the partition.
__global__ __launch_bounds__(kBlock) void out_weight_sum_kernel(const uint32_t *out_off, const float *w,
                                                                const uint32_t *order, const uint32_t *counts,
                                                                uint32_t nb_hub, uint32_t nb_wave, double *W) {
  __shared__ double part[kWavesPerBlock];
  const uint32_t t = threadIdx.x, wv = t / kWave, lane = t & (kWave - 1);
  const uint32_t n_lane = counts[0], n_wave = counts[1], n_hub = counts[2];
  if (blockIdx.x < nb_hub) {
    for (uint32_t i = blockIdx.x; i < n_hub; i += nb_hub) {  // block-uniform
      const uint32_t u = order[n_lane + n_wave + i], b = out_off[u];
      const double s = group_sum<kWave>(weight_sum<kBlock>(w + b, t, out_off[u + 1] - b));
      if (lane == 0) part[wv] = s;
      __syncthreads();
      if (t == 0) W[u] = (part[0] + part[1]) + (part[2] + part[3]);
      __syncthreads();
    }
  } else if (blockIdx.x < nb_hub + nb_wave) {
    for (uint32_t i = (blockIdx.x - nb_hub) * kWavesPerBlock + wv; i < n_wave; i += nb_wave * kWavesPerBlock) {
      const uint32_t u = order[n_lane + i], b = out_off[u];
      const double s = group_sum<kWave>(weight_sum<kWave>(w + b, lane, out_off[u + 1] - b));
      if (lane == 0) W[u] = s;
    }
  } else {
    const uint32_t nb = gridDim.x - nb_hub - nb_wave;
    for (uint32_t i = (blockIdx.x - nb_hub - nb_wave) * kBlock + t; i < n_lane; i += nb * kBlock) {
      const uint32_t u = order[i], b = out_off[u];
      W[u] = weight_sum<1>(w + b, 0, out_off[u + 1] - b);
    }
  }
}

// For a CSR of the degree-ordered layout (rows and ids in new numbering, perm: new -> old): eid[k] = the raw
// out-CSR slot of the same edge as slot k, by binary search in the source's ascending out-row. transpose: rows are
// destinations (the layout in-CSR), else sources (its out-CSR).
__global__ __launch_bounds__(kBlock) void layout_edge_map_kernel(const uint32_t *l_off, const uint32_t *l_idx,
                                                                 const uint32_t *perm, const uint32_t *out_off,
                                                                 const uint32_t *out_dst, uint32_t N, int transpose,
                                                                 uint32_t *eid, int *missing) {
  const int wv = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  bool bad = false;
  for (uint32_t i = blockIdx.x * kWavesPerBlock + wv; i < N; i += gridDim.x * kWavesPerBlock) {
    const uint32_t a = perm[i];
    for (uint32_t k = l_off[i] + lane; k < l_off[i + 1]; k += kWave) {
      const uint32_t b = perm[l_idx[k]];
      const uint32_t u = transpose ? b : a, v = transpose ? a : b;
      uint32_t lo = out_off[u], hi = out_off[u + 1];
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (out_dst[mid] < v) lo = mid + 1;
        else hi = mid;
      }
      const bool found = lo < out_off[u + 1] && out_dst[lo] == v;
      bad |= !found;
      eid[k] = found ? lo : 0u;
    }
  }
  if (bad) atomicOr(missing, 1);
}

__global__ __launch_bounds__(kBlock) void permute_weights_kernel(const float *w_out, const uint32_t *in_eid, size_t M,
                                                                 float *w_in) {
  for (size_t k = size_t(blockIdx.x) * kBlock + threadIdx.x; k < M; k += size_t(gridDim.x) * kBlock)
    w_in[k] = w_out[in_eid[k]];
}

__global__ __launch_bounds__(kBlock) void permute_u32_kernel(const uint32_t *src, const uint32_t *idx, size_t M,
                                                             uint32_t *dst) {
  for (size_t k = size_t(blockIdx.x) * kBlock + threadIdx.x; k < M; k += size_t(gridDim.x) * kBlock)
    dst[k] = src[idx[k]];
}

// x = z = start (adjoint: lam0 = g) or x = s, z = s / W (forward: r0 = s).
__global__ __launch_bounds__(kBlock) void weighted_init_kernel(const double *start, const double *W, uint32_t N,
                                                               int adjoint, double *x, double *z) {
  for (uint32_t v = blockIdx.x * kBlock + threadIdx.x; v < N; v += gridDim.x * kBlock) {
    const double s = start[v];
    x[v] = s;
    z[v] = adjoint ? s : s / W[v];
  }
}

// Per source u: dL/ds_u, and the factors of its edges' gradients dL/dw_uv = fu (lam_v - su).
__global__ __launch_bounds__(kBlock) void weighted_factors_kernel(const double *W, const double *r, const double *lam,
                                                                  const double *g, double P, uint32_t N, double *fu,
                                                                  double *su, double *grad_s) {
  for (uint32_t u = blockIdx.x * kBlock + threadIdx.x; u < N; u += gridDim.x * kBlock) {
    const double lu = lam[u];
    su[u] = (lu - g[u]) / P;
    fu[u] = P * r[u] / W[u];
    grad_s[u] = (1 - P) * lu;
  }
}

constexpr uint32_t kGradEdges = 4096;  // edges per workgroup of the gradient

// dL/dw in the caller's edge order, so that the gradients are written once and in sequence, kGradEdges edges a
// workgroup however the rows fall (every row has an edge). A wave finds the tile's first row (64 offsets a round); the
// rows that start in the tile leave their number at their first edge, and a running maximum turns that into every
// edge's row. (A wave per row of the layout, and the result scattered to the caller's order: 507 + 120 us on 1M
// vertices, 17M edges, bound by the hubs' rows; a workgroup per 256 rows 1758 us, bound by the 256 that hold the hubs;
// this: 123 us, and 15 us for the factors.)
__global__ __launch_bounds__(kBlock) void weighted_grad_kernel(const uint32_t *out_off, const uint32_t *out_dst,
                                                               const double *lam, const double *fu, const double *su,
                                                               uint32_t N, uint64_t M, double *grad_w) {
  constexpr uint32_t E = kGradEdges / kBlock;  // edges per thread
  __shared__ uint16_t row[kGradEdges];
  __shared__ uint32_t first, top[kWavesPerBlock];
  const uint32_t t = threadIdx.x, wv = t / kWave, lane = t & (kWave - 1);
  const uint64_t e0 = uint64_t(blockIdx.x) * kGradEdges;
  const uint32_t n = uint32_t(min(uint64_t(kGradEdges), M - e0));
  if (wv == 0) {  // the last row with off[row] <= e0
    uint64_t lo = 0, hi = N;
    while (hi - lo > 1) {
      const uint64_t step = (hi - lo + kWave - 1) / kWave, at = lo + lane * step;
      const uint32_t k = __popcll(__ballot(at < hi && out_off[at] <= e0));  // at least 1: lane 0
      hi = min(hi, lo + k * step);
      lo += (k - 1) * step;
    }
    if (lane == 0) first = uint32_t(lo);
  }
#pragma unroll
  for (uint32_t k = 0; k < E; ++k) row[k * kBlock + t] = 0;
  __syncthreads();
  const uint32_t r0 = first;
  for (uint32_t i = 1 + t; i <= kGradEdges && r0 + i < N; i += kBlock) {
    const uint64_t b = out_off[r0 + i] - e0;  // row r0 + i > r0 starts after e0
    if (b >= n) break;
    row[b] = uint16_t(i);
  }
  __syncthreads();
  // Running maximum: thread t over its E edges, then over the threads before it.
  uint32_t m[E], best = 0;
#pragma unroll
  for (uint32_t k = 0; k < E; ++k) m[k] = best = max(best, uint32_t(row[t * E + k]));
  uint32_t up = best;  // inclusive over the wave
#pragma unroll
  for (int d = 1; d < kWave; d *= 2) {
    const uint32_t o = __shfl_up(up, d);
    if (lane >= uint32_t(d)) up = max(up, o);
  }
  if (lane == kWave - 1) top[wv] = up;
  uint32_t before = __shfl_up(up, 1);
  if (lane == 0) before = 0;
  __syncthreads();
  for (uint32_t k = 0; k < wv; ++k) before = max(before, top[k]);
#pragma unroll
  for (uint32_t k = 0; k < E; ++k) row[t * E + k] = uint16_t(max(before, m[k]));
  __syncthreads();
  for (uint32_t i = t; i < n; i += 8 * kBlock) {
    uint32_t v[8];
    double x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = i + k * kBlock < n ? out_dst[e0 + i + k * kBlock] : 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = i + k * kBlock < n ? lam[v[k]] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (i + k * kBlock >= n) break;
      const uint32_t u = r0 + row[i + k * kBlock];
      grad_w[e0 + i + k * kBlock] = fu[u] * (x[k] - su[u]);
    }
  }
}

inline uint32_t blocks(size_t n, size_t per, uint32_t cap) {
  const size_t g = (n + per - 1) / per;
  return uint32_t(g < 1 ? 1 : (g > cap ? cap : g));
}

// key[i] = 64 - degree of row order[i] (low rows only: degree <= 64), for the degree sort of the low rows.
__global__ __launch_bounds__(kBlock) void degree_keys_kernel(const uint32_t *off, const uint32_t *order, uint32_t n,
                                                             uint32_t *key) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const uint32_t v = order[i];
    key[i] = 64u - (off[v + 1] - off[v]);
  }
}

template <bool ADJOINT>
hipError_t launch_step(const WeightedArgs &A, const LoopCtl &ctl, hipStream_t s) {
  const uint32_t nb_high = A.sched.n_high ? blocks(A.sched.n_high, kWavesPerBlock, 16384) : 0;
  uint32_t nb_low = 0;
  for (int k = 0; k < A.n_bands; ++k)
    nb_low = max(nb_low, A.band[k].block_begin +
                             (A.band[k].end - A.band[k].begin + A.band[k].per_block - 1) / A.band[k].per_block);
  const uint32_t grid = A.n_chunks + nb_high + nb_low;
  if (grid) weighted_step_kernel<ADJOINT><<<grid, kBlock, 0, s>>>(A, nb_high, ctl);
  if (A.sched.n_huge)
    weighted_heavy_kernel<ADJOINT><<<blocks(A.sched.n_huge, kWavesPerBlock, 4096), kBlock, 0, s>>>(A, ctl);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_weighted_step(bool adjoint, const WeightedArgs &A, const LoopCtl &ctl, hipStream_t s) {
  return adjoint ? launch_step<true>(A, ctl, s) : launch_step<false>(A, ctl, s);
}

hipError_t launch_degree_keys(const uint32_t *off, const uint32_t *order, uint32_t n, uint32_t *key, hipStream_t s) {
  if (!n) return hipSuccess;
  degree_keys_kernel<<<blocks(n, kBlock, 8192), kBlock, 0, s>>>(off, order, n, key);
  return hipGetLastError();
}

hipError_t launch_out_weight_sum(const uint32_t *out_off, const float *w, uint32_t N, const uint32_t *order,
                                 const uint32_t *counts, double *W, hipStream_t s) {
  if (!N) return hipSuccess;
  const uint32_t nb_hub = 256, nb_wave = blocks(N, 16 * kWavesPerBlock, 2048), nb_lane = blocks(N, kBlock, 8192);
  out_weight_sum_kernel<<<nb_hub + nb_wave + nb_lane, kBlock, 0, s>>>(out_off, w, order, counts, nb_hub, nb_wave, W);
  return hipGetLastError();
}

hipError_t launch_layout_edge_map(const uint32_t *l_off, const uint32_t *l_idx, const uint32_t *perm,
                                  const uint32_t *out_off, const uint32_t *out_dst, uint32_t N, bool transpose,
                                  uint32_t *eid, int *missing, hipStream_t s) {
  if (!N) return hipSuccess;
  layout_edge_map_kernel<<<blocks(N, kWavesPerBlock, 16384), kBlock, 0, s>>>(l_off, l_idx, perm, out_off, out_dst, N,
                                                                              transpose ? 1 : 0, eid, missing);
  return hipGetLastError();
}

hipError_t launch_permute_weights(const float *w_out, const uint32_t *in_eid, size_t M, float *w_in, hipStream_t s) {
  if (!M) return hipSuccess;
  permute_weights_kernel<<<blocks(M, kBlock, 16384), kBlock, 0, s>>>(w_out, in_eid, M, w_in);
  return hipGetLastError();
}

hipError_t launch_permute_u32(const uint32_t *src, const uint32_t *idx, size_t M, uint32_t *dst, hipStream_t s) {
  if (!M) return hipSuccess;
  permute_u32_kernel<<<blocks(M, kBlock, 16384), kBlock, 0, s>>>(src, idx, M, dst);
  return hipGetLastError();
}

hipError_t launch_weighted_init(const double *start, const double *W, uint32_t N, bool adjoint, double *x, double *z,
                                hipStream_t s) {
  if (!N) return hipSuccess;
  weighted_init_kernel<<<blocks(N, kBlock, 8192), kBlock, 0, s>>>(start, W, N, adjoint ? 1 : 0, x, z);
  return hipGetLastError();
}

hipError_t launch_weighted_grad(const uint32_t *out_off, const uint32_t *out_dst, const double *W, const double *r,
                                const double *lam, const double *g, double P, uint32_t N, uint64_t M, double *fu,
                                double *su, double *grad_w, double *grad_s, hipStream_t s) {
  if (!N) return hipSuccess;
  weighted_factors_kernel<<<blocks(N, kBlock, 8192), kBlock, 0, s>>>(W, r, lam, g, P, N, fu, su, grad_s);
  if (M)
    weighted_grad_kernel<<<uint32_t((M + kGradEdges - 1) / kGradEdges), kBlock, 0, s>>>(out_off, out_dst, lam, fu, su, N,
                                                                                       M, grad_w);
  return hipGetLastError();
}

}  // namespace prh
