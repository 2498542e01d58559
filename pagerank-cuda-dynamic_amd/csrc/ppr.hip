// ppr.hip -- batched personalized PageRank: up to 64 teleport columns solved together.
//
// Column j: r_j <- (1-P) s_j + P * sum_{u in in(v)} r_j[u]/deg[u], from r_j = s_j, stopping at the first iteration
// whose L-inf change of column j is below the tolerance (the rule of pagerankLoopCuU, pagerankCuda.hxx:680-690,
// applied per column).
//
// Layout. The columns are cut into tiles of KT (all of them when there are at most kPprTile), and a tile keeps its
// contributions r/deg as rows of KT FP64 values, [tile][V][KT] in the graph's degree-ordered layout. One iteration of
// one tile gathers from one tile's array only. What bounds the gathers is where their lines come from: the 64-column
// rows of a million-vertex graph are 537 MB, more than the Infinity Cache, and an L2 holds 8K of them; a 32-column tile's
// are 268 MB and 16K. With few columns the rows are short, and a wave takes many edges at once instead of leaving most
// of its lanes idle. Measured against 512-byte rows for any number of columns, one lane each, in the caller's order and
// with ranks beside the contributions (per iteration): 64 columns, 1M vertices, 17M edges 2003 -> 850 us (10.3 TB/s of
// gathered rows); five columns, 100K vertices 315 -> 21 us; one column, 1M vertices 1.8 ms -> 0.1 ms.
//
// Only contributions are kept. The change of a column at v is |c_new - c_old| * deg, and the ranks are written once, by
// a last pass (FINAL) that repeats each column's last iteration from the contributions it read, into the caller's
// order: 8 bytes less written and 8 less held per vertex, column and iteration than keeping ranks beside them.
// Converged columns are masked: nothing of theirs is written, and a tile whose columns have all converged is left out.
//
// A wave reads KT columns of 64 / (KT / 2) edges at a time, two columns a lane. Rows by in-degree:
//   up to kPprGroup edges   one row per group of KT / 2 lanes, four edges in flight;
//   up to the chunk size    one row per wave, eight steps in flight, the lane groups' sums added across the wave;
//   heavier                 cut into chunks, one wave each, whose sums a second kernel adds in chunk order.
// A row whose only in-neighbour is itself (or none) and that is no seed stays 0 in every column; it is skipped (half the
// vertices of an RMAT graph). Every sum is taken in a fixed order, so results repeat bit for bit. The iteration index
// lives on the device (PprState::iter) and each replay of a captured run of iterations advances it once.
#include <algorithm>

#include "prh_device.hpp"
#include "prh_internal.hpp"

namespace prh {
namespace {

typedef double d2 __attribute__((ext_vector_type(2)));

template <int KT>
struct Shape {
  static constexpr int kVec = KT >= 2 ? 2 : 1;       // columns per lane
  static constexpr int kLanes = KT / kVec;           // lanes per edge
  static constexpr int kEdges = kWave / kLanes;      // edges per wave and step
};

template <int VEC>
struct Vals {
  double x[VEC];
};

// What a lane knows of its columns: their numbers, which are running, and where their contributions are read.
template <int KT>
struct Cols {
  static constexpr int V = Shape<KT>::kVec;
  int l;                 // iteration index
  uint32_t j;            // first column of the lane
  bool on[V];            // running (FINAL: a column of the caller's)
  int n[V];              // FINAL: iterations of the column
  const double *src[V];  // this lane's column in row 0 of the tile's contributions to read
  double *dst;           // and to write (first column)
};

template <int KT, bool FINAL>
__device__ __forceinline__ Cols<KT> columns(const PprArgs &A, int step, uint32_t tile, bool record) {
  constexpr int V = Shape<KT>::kVec;
  Cols<KT> q;
  const uint32_t c = (threadIdx.x & (kWave - 1)) % Shape<KT>::kLanes;
  const size_t base = size_t(tile) * A.N * KT + V * c;
  q.j = tile * KT + V * c;
  q.l = FINAL ? 0 : A.state->iter + step;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int j = int(q.j) + i;
    q.n[i] = 0;
    if constexpr (FINAL) {
      q.on[i] = j < A.k;
      const int d = q.on[i] ? A.state->done[j] : 0;
      q.n[i] = d ? d : A.max_iter;
      q.src[i] = A.contrib[(q.n[i] + 1) & 1] + base + i;  // what the column's last iteration read
    } else {
      bool a = j < A.k && q.l < A.max_iter && A.state->done[j] == 0;
      if (a && q.l > 0 && __longlong_as_double((long long)A.err[size_t(q.l - 1) * kPprCols + j]) < A.tol) {
        a = false;
        if (record) A.state->done[j] = q.l;
      }
      q.on[i] = a;
      q.src[i] = A.contrib[q.l & 1] + base + i;
    }
  }
  q.dst = A.contrib[(q.l + 1) & 1] + base;
  return q;
}

template <int KT>
__device__ __forceinline__ bool any_on(const Cols<KT> &q) {
  bool a = q.on[0];
  if constexpr (Shape<KT>::kVec == 2) a |= q.on[1];
  return __ballot(a) != 0;
}

// The lane's columns of row u. In the last pass the two columns may come from different buffers.
template <int KT, bool FINAL>
__device__ __forceinline__ Vals<Shape<KT>::kVec> load_row(const Cols<KT> &q, uint32_t u) {
  Vals<Shape<KT>::kVec> r;
  if constexpr (KT == 1) {
    r.x[0] = q.src[0][u];
  } else if constexpr (FINAL) {
    r.x[0] = q.src[0][size_t(u) * KT];
    r.x[1] = q.src[1][size_t(u) * KT];
  } else {
    const d2 t = *reinterpret_cast<const d2 *>(q.src[0] + size_t(u) * KT);
    r.x[0] = t.x;
    r.x[1] = t.y;
  }
  return r;
}

// Sum of the lane's columns over edges i, i + STEP, ... < n of the row whose sources start at src, U rows in flight.
template <int KT, bool FINAL, int STEP, int U>
__device__ __forceinline__ Vals<Shape<KT>::kVec> sum_rows(const Cols<KT> &q, const uint32_t *src, uint32_t i,
                                                          uint32_t n) {
  constexpr int V = Shape<KT>::kVec;
  Vals<V> s{};
  for (; i < n; i += U * STEP) {
    uint32_t u[U];
    Vals<V> x[U];
#pragma unroll
    for (int k = 0; k < U; ++k) u[k] = i + k * STEP < n ? src[i + k * STEP] : 0u;
#pragma unroll
    for (int k = 0; k < U; ++k) x[k] = i + k * STEP < n ? load_row<KT, FINAL>(q, u[k]) : Vals<V>{};
#pragma unroll
    for (int k = 0; k < U; ++k)
#pragma unroll
      for (int c = 0; c < V; ++c) s.x[c] += x[k].x[c];
  }
  return s;
}

// Adds the lane groups' sums across the wave (every lane ends with the total of its columns).
template <int KT>
__device__ __forceinline__ void add_groups(Vals<Shape<KT>::kVec> &s) {
#pragma unroll
  for (int d = Shape<KT>::kLanes; d < kWave; d *= 2)
#pragma unroll
    for (int i = 0; i < Shape<KT>::kVec; ++i) s.x[i] += __shfl_xor(s.x[i], d);
}

// Row v from its in-sum: the next contribution and the change (into emax), or in the last pass the rank.
template <int KT, bool FINAL>
__device__ __forceinline__ void finish_row(const PprArgs &A, const Cols<KT> &q, uint32_t v, int32_t row,
                                           const Vals<Shape<KT>::kVec> &cv, double *out,
                                           Vals<Shape<KT>::kVec> &emax) {
  constexpr int V = Shape<KT>::kVec;
  Vals<V> s{}, a;
  if (row >= 0)
#pragma unroll
    for (int i = 0; i < V; ++i) s.x[i] = A.seed_mass[size_t(row) * A.cols + q.j + i];
#pragma unroll
  for (int i = 0; i < V; ++i) a.x[i] = fma(A.P, cv.x[i], (1 - A.P) * s.x[i]);
  if constexpr (FINAL) {
    double *o = out + size_t(A.perm[v]) * A.k + q.j;
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (q.on[i]) o[i] = q.n[i] ? a.x[i] : s.x[i];
  } else {
    const Vals<V> old = load_row<KT, FINAL>(q, v);
    const double d = max(A.deg[v], 1u);  // a dead end's contribution is never gathered: its rank stands there
#pragma unroll
    for (int i = 0; i < V; ++i) {
      a.x[i] = a.x[i] / d;
      emax.x[i] = fmax(emax.x[i], fabs(a.x[i] - old.x[i]) * d);
    }
    double *p = q.dst + size_t(v) * KT;
    if constexpr (V == 1) {
      if (q.on[0]) p[0] = a.x[0];
    } else if (q.on[0] && q.on[1]) {
      *reinterpret_cast<d2 *>(p) = d2{a.x[0], a.x[1]};
    } else {
      if (q.on[0]) p[0] = a.x[0];
      if (q.on[1]) p[1] = a.x[1];
    }
  }
}

// Says which of the lane's columns changed by at least the tolerance (as report_change does for one column).
template <int KT>
__device__ __forceinline__ void report_columns(const PprArgs &A, const Cols<KT> &q,
                                               const Vals<Shape<KT>::kVec> &emax) {
#pragma unroll
  for (int i = 0; i < Shape<KT>::kVec; ++i)
    if (q.on[i] && emax.x[i] >= A.tol) A.err[size_t(q.l) * kPprCols + q.j + i] = kChanged;
}

// One iteration's sums, tile after tile: heavy rows' chunks (partial sums), wave rows and group rows (finished here).
// Eight waves per SIMD (64 VGPRs, a few spilled) pay where lines come from memory: 64 columns at 1M vertices 114.9 ->
// 112.0 ms per solve; narrow tiles, which the L2s serve, lose (five columns at 100K 2.62 -> 2.73 ms).
template <int KT, bool FINAL>
__global__ __launch_bounds__(kBlock, KT >= 16 ? 8 : 1) void ppr_gather_kernel(PprArgs A, int step, uint32_t nb_chunk, uint32_t nb_high,
                                                            uint32_t nb_low, double *out) {
  using S = Shape<KT>;
  const uint32_t nb = nb_chunk + nb_high + nb_low;
  const uint32_t tile = blockIdx.x / nb;
  uint32_t b = blockIdx.x - tile * nb;
  const Cols<KT> q = columns<KT, FINAL>(A, step, tile, b == 0 && threadIdx.x < kWave);
  if (!any_on(q)) return;
  const uint32_t w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1), slot = lane / S::kLanes;
  Vals<S::kVec> emax{};
  if (b < nb_chunk) {
    for (uint32_t i = b * kWavesPerBlock + w; i < A.n_chunks; i += nb_chunk * kWavesPerBlock) {
      const uint32_t b0 = A.chunk_beg[i];
      Vals<S::kVec> s = sum_rows<KT, FINAL, S::kEdges, 8>(q, A.src + b0, slot, A.chunk_end[i] - b0);
      add_groups<KT>(s);
      if (slot == 0) {
        double *p = A.partial + size_t(i) * A.cols + q.j;
#pragma unroll
        for (int k = 0; k < S::kVec; ++k) p[k] = s.x[k];
      }
    }
    if (!FINAL && blockIdx.x == 0 && threadIdx.x == 0) tell_host(A.host, q.l + 1);
    return;
  }
  b -= nb_chunk;
  if (b < nb_high) {
    for (uint32_t i = b * kWavesPerBlock + w; i < A.n_high; i += nb_high * kWavesPerBlock) {
      const uint32_t v = A.order[A.n_low + i];
      const uint32_t e = A.off[v], end = A.off[v + 1];
      const int32_t row = A.seed_row[v];
      Vals<S::kVec> s = sum_rows<KT, FINAL, S::kEdges, 8>(q, A.src + e, slot, end - e);
      add_groups<KT>(s);
      if (slot == 0) finish_row<KT, FINAL>(A, q, v, row, s, out, emax);
    }
  } else {
    b -= nb_high;
    constexpr uint32_t kRows = kWavesPerBlock * S::kEdges;  // rows per workgroup and round
    for (uint32_t i = b * kRows + w * S::kEdges + slot; i < A.n_low; i += nb_low * kRows) {
      const uint32_t v = A.order[i];
      const uint32_t e = A.off[v], end = A.off[v + 1];
      const int32_t row = A.seed_row[v];
      // Rows fed by nothing but themselves, no seed of any column: 0 in both buffers from the start.
      if (!FINAL && row < 0 && end - e <= 1 && (end == e || A.src[e] == v)) continue;
      const Vals<S::kVec> s = sum_rows<KT, FINAL, 1, 4>(q, A.src + e, 0, end - e);
      finish_row<KT, FINAL>(A, q, v, row, s, out, emax);
    }
  }
  if constexpr (!FINAL) {
    report_columns<KT>(A, q, emax);
    if (blockIdx.x == 0 && threadIdx.x == 0) tell_host(A.host, q.l + 1);
  }
}

// Heavy rows: add the chunk partials (lane group g takes chunks g, g + groups, ...) and finish.
template <int KT, bool FINAL>
__global__ __launch_bounds__(kBlock) void ppr_combine_kernel(PprArgs A, int step, uint32_t nb, double *out) {
  using S = Shape<KT>;
  const uint32_t tile = blockIdx.x / nb, b = blockIdx.x - tile * nb;
  const Cols<KT> q = columns<KT, FINAL>(A, step, tile, false);
  if (!any_on(q)) return;
  const uint32_t w = threadIdx.x / kWave, slot = (threadIdx.x & (kWave - 1)) / S::kLanes;
  Vals<S::kVec> emax{};
  for (uint32_t h = b * kWavesPerBlock + w; h < A.n_heavy; h += nb * kWavesPerBlock) {
    const uint32_t v = A.order[A.n_low + A.n_high + h];
    Vals<S::kVec> s{};
    for (uint32_t i = A.heavy_first[h] + slot; i < A.heavy_first[h + 1]; i += S::kEdges)
#pragma unroll
      for (int k = 0; k < S::kVec; ++k) s.x[k] += A.partial[size_t(i) * A.cols + q.j + k];
    add_groups<KT>(s);
    if (slot == 0) finish_row<KT, FINAL>(A, q, v, A.seed_row[v], s, out, emax);
  }
  if constexpr (!FINAL) report_columns<KT>(A, q, emax);
}

// After a run of `steps` iterations: the columns whose last one was below the tolerance are done; the next run's index.
// Tells the host how far it is, and when no column is left.
__global__ __launch_bounds__(kWave) void ppr_advance_kernel(PprArgs A, int steps) {
  const int j = threadIdx.x, l = A.state->iter + steps - 1;
  int d = j < A.k ? A.state->done[j] : 1;
  if (d == 0 && l < A.max_iter && __longlong_as_double((long long)A.err[size_t(l) * kPprCols + j]) < A.tol)
    A.state->done[j] = d = l + 1;
  const bool all = __ballot(d == 0) == 0;
  if (j == 0) {
    A.state->iter = l + 1;
    if (all) tell_host(A.host + 1, 1);
    else tell_host(A.host, l + 1);
  }
}

__global__ __launch_bounds__(kBlock) void ppr_reset_kernel(PprArgs A, int32_t *seed_row, double *mass, size_t rows) {
  const size_t t = size_t(blockIdx.x) * kBlock + threadIdx.x, st = size_t(gridDim.x) * kBlock;
  for (size_t x = t; x < size_t(A.max_iter) * kPprCols; x += st) A.err[x] = 0ull;
  for (size_t x = t; x < A.N; x += st) seed_row[x] = -1;
  for (size_t x = t; x < rows * A.cols; x += st) mass[x] = 0.0;
  if (t < kPprCols) A.state->done[t] = 0;
  if (t == 0) A.state->iter = A.state->rows = 0;
}

// How many lanes of the wave the calling lane answers for: valid lanes with the same key leave it to the first of them, who
// gets their number, the others 0. Every lane must call it.
__device__ __forceinline__ uint32_t answers_for(uint32_t key, bool valid) {
  uint32_t n = 0;
  for (unsigned long long todo = __ballot(valid); todo;) {
    const int leader = __ffsll(todo) - 1;
    const uint32_t its = __shfl(key, leader);
    const unsigned long long same = __ballot(key == its) & todo;
    if (lane_id() == leader) n = __popcll(same);
    todo &= ~same;
  }
  return n;
}

// The columns' concatenated seed sets turned into layout rows; the first entry to claim a row takes the next row of the
// mass table for it. (One atomic on one word per entry took 12 ms for a million entries of one vertex.)
__global__ __launch_bounds__(kBlock) void ppr_claim_kernel(uint32_t *seeds, uint32_t n, const uint32_t *inv,
                                                           int32_t *seed_row, PprState *state) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  for (size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x; i - lane < n; i += size_t(gridDim.x) * kBlock) {
    uint32_t v = 0;
    if (i < n) seeds[i] = v = inv[seeds[i]];
    if (answers_for(v, i < n && seed_row[v] == -1) && atomicCAS(&seed_row[v], -1, -2) == -1)
      seed_row[v] = atomicAdd(&state->rows, 1);
  }
}

// mass[row of v][j] = occurrences of v in seed set j, column j = blockIdx.x. Whole numbers, so the order of the additions
// does not matter. Equal seeds of a wave make one addition, and several workgroups share a column. Per call, a workgroup per
// column that adds every share by itself -> this: a million repeats of one vertex 26.1 -> 1.2 ms (64 vertices), of 64
// vertices 5.1 -> 1.6, a million seeds of 8,192 vertices 4.1 -> 1.5; one seed 1.01 and 1.00.
__global__ __launch_bounds__(kBlock) void ppr_count_kernel(const uint32_t *seeds, const uint32_t *first,
                                                           const int32_t *seed_row, int cols, double *mass) {
  const uint32_t j = blockIdx.x, n = first[j + 1] - first[j], lane = threadIdx.x & (kWave - 1);
  seeds += first[j];
  for (size_t i = blockIdx.y * kBlock + threadIdx.x; i - lane < n; i += gridDim.y * kBlock) {
    const uint32_t row = i < n ? uint32_t(seed_row[seeds[i]]) : 0u;
    if (const uint32_t k = answers_for(row, i < n)) atomicAdd(&mass[size_t(row) * cols + j], double(k));
  }
}

// The counts of the mass table turned into shares s_j[v] = count / |seed set j|, and the contributions s/deg of the start
// ranks r = s (zero outside the seeds and for unused columns). Rows that the iterations may skip get their zeros in both
// buffers.
__global__ __launch_bounds__(kBlock) void ppr_init_kernel(PprArgs A, const uint32_t *first, double *mass) {
  const size_t n = size_t(A.N) * A.cols;
  for (size_t x = size_t(blockIdx.x) * kBlock + threadIdx.x; x < n; x += size_t(gridDim.x) * kBlock) {
    const size_t t = x / A.tile;
    const uint32_t c = uint32_t(x - t * A.tile), tile = uint32_t(t / A.N), v = uint32_t(t - size_t(tile) * A.N);
    const uint32_t j = tile * A.tile + c;
    const int32_t row = A.seed_row[v];
    double s = 0.0;
    if (row >= 0 && j < uint32_t(A.k)) {
      double *m = mass + size_t(row) * A.cols + j;  // no other thread's: v's row, column j
      *m = s = *m / double(first[j + 1] - first[j]);
    }
    A.contrib[0][x] = s / max(A.deg[v], 1u);
    if (A.off[v + 1] - A.off[v] <= 1) A.contrib[1][x] = 0.0;
  }
}

inline uint32_t grid_for(size_t n, size_t per, uint32_t cap) {
  const size_t g = (n + per - 1) / per;
  return uint32_t(g < 1 ? 1 : (g > cap ? cap : g));
}

template <int KT, bool FINAL>
hipError_t launch_pass(const PprArgs &A, int step, double *out, hipStream_t s) {
  const uint32_t tiles = uint32_t(A.cols / KT);
  const uint32_t nb_chunk = A.n_chunks ? grid_for(A.n_chunks, kWavesPerBlock, 8192) : 0;
  const uint32_t nb_high = A.n_high ? grid_for(A.n_high, kWavesPerBlock, 16384) : 0;
  const uint32_t nb_low = A.n_low ? grid_for(A.n_low, kWavesPerBlock * Shape<KT>::kEdges, 16384) : 0;
  const uint32_t nb = nb_chunk + nb_high + nb_low;
  if (nb) ppr_gather_kernel<KT, FINAL><<<nb * tiles, kBlock, 0, s>>>(A, step, nb_chunk, nb_high, nb_low, out);
  if (A.n_heavy) {
    const uint32_t hb = grid_for(A.n_heavy, kWavesPerBlock, 4096);
    ppr_combine_kernel<KT, FINAL><<<hb * tiles, kBlock, 0, s>>>(A, step, hb, out);
  }
  return hipGetLastError();
}

template <bool FINAL>
hipError_t launch_tiles(const PprArgs &A, int step, double *out, hipStream_t s) {
  switch (A.tile) {
    case 1: return launch_pass<1, FINAL>(A, step, out, s);
    case 2: return launch_pass<2, FINAL>(A, step, out, s);
    case 4: return launch_pass<4, FINAL>(A, step, out, s);
    case 8: return launch_pass<8, FINAL>(A, step, out, s);
    case 16: return launch_pass<16, FINAL>(A, step, out, s);
    case 32: return launch_pass<32, FINAL>(A, step, out, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_ppr_setup(const PprArgs &A, uint32_t *seeds, uint32_t n_seeds, const uint32_t *first,
                            const uint32_t *inv, int32_t *seed_row, double *mass, hipStream_t s) {
  const size_t rows = std::min(n_seeds, A.N);  // of the mass table
  const size_t most = std::max<size_t>(std::max<size_t>(A.N, size_t(A.max_iter) * kPprCols), rows * A.cols);
  ppr_reset_kernel<<<grid_for(most, kBlock, 4096), kBlock, 0, s>>>(A, seed_row, mass, rows);
  ppr_claim_kernel<<<grid_for(n_seeds, kBlock, 4096), kBlock, 0, s>>>(seeds, n_seeds, inv, seed_row, A.state);
  ppr_count_kernel<<<dim3(A.k, grid_for(n_seeds, 8 * kBlock, 256)), kBlock, 0, s>>>(seeds, first, seed_row, A.cols, mass);
  ppr_init_kernel<<<grid_for(size_t(A.N) * A.cols, kBlock, 16384), kBlock, 0, s>>>(A, first, mass);
  return hipGetLastError();
}

hipError_t launch_ppr_iteration(const PprArgs &A, int step, hipStream_t s) {
  return launch_tiles<false>(A, step, nullptr, s);
}

hipError_t launch_ppr_advance(const PprArgs &A, int steps, hipStream_t s) {
  ppr_advance_kernel<<<1, kWave, 0, s>>>(A, steps);
  return hipGetLastError();
}

hipError_t launch_ppr_ranks(const PprArgs &A, double *out, hipStream_t s) { return launch_tiles<true>(A, 0, out, s); }

}  // namespace prh
