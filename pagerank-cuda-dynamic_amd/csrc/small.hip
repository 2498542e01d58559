// small.hip -- the iterations of a small graph's solve in one workgroup (every unweighted variant, row plan).
//
// On a graph of a few thousand vertices a launch per iteration is all latency: the entry test, the row's operands, its
// source ids, the gathers and the reduction follow one another through L2, and the next launch waits for the last.
// Here one workgroup of sixteen waves keeps the whole problem in LDS (contributions twice, ranks, out-degrees, flags and
// source ids) and runs the iterations one after another with two barriers in each.
//
// One CU then does all the work, and the id lists are laid out for few instructions and few LDS reads.
// Rows in order of in-degree take W lanes each, so many that a lane has about kSmallEdges / 2 to kSmallEdges edges; 64 / W
// rows make an item, which a wave runs in rounds of four edges a lane, as many as its first and longest row needs. A
// lane's four ids of a round are one 8-byte word (at 8 times the vertex, the offset of its contribution), 64 lanes' words
// follow one another, and a list that ends early goes on with a vertex whose contribution is 0: a round is one wide load,
// four gathers and four additions, without a test. The rest of a vertex's update (its divisions above all) runs with
// a vertex in every lane afterwards. What is left is a chain of LDS round trips and barriers: 1.75 us an iteration on
// RMAT-10 (12K edges), where a launch an iteration takes 3.8.
//
// Whole solves through the C entry, a launch an iteration -> this: 100 vertices 475 -> 197 us, 1,024 454 -> 253, 2,200 445
// -> 330 (16 edges each); DF at 1,500 vertices, where an iteration is two launches, 873 -> 432; DF-P 417 -> 271. So it is
// taken wherever the problem fits (about 2,500 vertices of 16 edges, 3,300 of few). 8 edges a lane instead of 16: 277 us
// at 1,024 vertices, 32: 266; gathers of two and four rounds in flight together: 262 and 271.
//
// The update and flag rules are those of update.hpp; the frontier's extension is the pull form. Sums are taken in a fixed
// order, so results repeat bit for bit.
#include <type_traits>

#include "prh_device.hpp"
#include "prh_internal.hpp"
#include "update.hpp"

namespace prh {
namespace {

constexpr int kSmallWaves = kSmallBlock / kWave;

// The problem in LDS.
struct SmallState {
  uint64_t *ids;   // four ids a word: round q of item i at [(first(i) + q) * 64 + lane]
  uint8_t *lds;    // two lists of contributions, old and new in turn (doubles, addressed in bytes); that of vertex N is 0
  double *r;       // ranks
  uint32_t *item;  // first(i) | rounds << 16
  uint16_t *deg;   // out-degrees
  uint8_t *vaff, *naff;
};

// (A list is a distance from `lds`: a choice between two pointers would make its loads generic, not LDS ones.)
__device__ __forceinline__ double &at(const SmallState &S, uint32_t list, uint32_t byte) {
  return *reinterpret_cast<double *>(S.lds + (list + byte));
}

// Calls f(W, item, lane's row, whether it is one) for this wave's items of every band.
template <int W, class F>
__device__ __forceinline__ void each_item_of(const SmallArgs &A, int k, const F &f) {
  constexpr uint32_t G = kWave / W;
  const uint32_t w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  const uint32_t b = A.item[k], e = A.item[k + 1];
  for (uint32_t i = b + (w - b) % kSmallWaves; i < e; i += kSmallWaves) {  // wave-uniform
    const uint32_t v = A.band[k] + (i - b) * G + lane / W;
    f(std::integral_constant<int, W>{}, i, v, v < A.band[k + 1]);
  }
}
template <class F>
__device__ __forceinline__ void each_item(const SmallArgs &A, const F &f) {
  each_item_of<64>(A, 0, f);
  each_item_of<32>(A, 1, f);
  each_item_of<16>(A, 2, f);
  each_item_of<8>(A, 3, f);
  each_item_of<4>(A, 4, f);
  each_item_of<2>(A, 5, f);
  each_item_of<1>(A, 6, f);
}

// Row v's new rank, contribution and flags, from the sum in cn; returns the change of its rank.
template <int VARIANT>
__device__ __forceinline__ double small_finish(const SmallArgs &A, const SmallState &S, uint32_t c, uint32_t cn,
                                               uint32_t v) {
  using T = Traits<VARIANT>;
  const double cv = at(S, cn, 8 * v), crv = at(S, c, 8 * v), rv = S.r[v];
  if (T::dynamic && !S.vaff[v]) {
    at(S, cn, 8 * v) = crv;
    if constexpr (T::frontier) S.naff[v] = 0;
    return 0.0;
  }
  const uint32_t d = S.deg[v];
  double av;
  if constexpr (T::prune) av = fma(A.P, cv - crv, A.C0) * (1.0 / (1.0 - A.P / d));
  else av = fma(A.P, cv, A.C0);
  S.r[v] = av;
  at(S, cn, 8 * v) = av / d;
  const double ev = fabs(av - rv);
  if constexpr (T::frontier) {
    const double rel = ev / fmax(rv, av);
    if (T::prune && rel <= A.C) S.vaff[v] = 0;
    S.naff[v] = rel > A.D ? 1 : 0;
  }
  return ev;
}

template <int VARIANT>
__global__ __launch_bounds__(kSmallBlock) void small_solve_kernel(SmallArgs A) {
  using T = Traits<VARIANT>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kSmallLds];
  __shared__ uint32_t wave_rounds[kSmallWaves];
  const uint32_t N = A.N, t = threadIdx.x, w = t / kWave, lane = t & (kWave - 1);
  SmallState S;
  S.lds = lds;
  const uint32_t list = 8 * (N + 1);  // bytes
  S.r = reinterpret_cast<double *>(lds + 2 * list);
  S.ids = reinterpret_cast<uint64_t *>(S.r + N);
  S.item = reinterpret_cast<uint32_t *>(S.ids + size_t(A.rounds) * kWave);
  S.deg = reinterpret_cast<uint16_t *>(S.item + A.item[7]);
  S.vaff = reinterpret_cast<uint8_t *>(S.deg + N);
  S.naff = S.vaff + N;
  for (uint32_t v = t; v < N; v += kSmallBlock) {
    const uint32_t d = A.deg[v];
    const double r = A.rank[A.first & 1][v];
    S.deg[v] = uint16_t(d);
    S.r[v] = r;
    at(S, 0, 8 * v) = r / d;
    if constexpr (T::dynamic) {
      S.vaff[v] = A.vaff[v];
      S.naff[v] = 0;
    }
  }
  if (t == 0) {
    at(S, 0, 8 * N) = 0.0;
    at(S, list, 8 * N) = 0.0;
    S.naff[N] = 0;
  }
  // The items' rounds and where their ids start: a thread an item, prefix sums by waves.
  uint32_t rounds = 0;
  if (t < A.item[7]) {
    int k = 0;
    while (t >= A.item[k + 1]) ++k;
    const uint32_t v = A.band[k] + (t - A.item[k]) * (1u << k);
    rounds = small_rounds(A.off[v + 1] - A.off[v], k);
  }
  uint32_t sum = rounds;
  for (int o = 1; o < kWave; o *= 2) {
    const uint32_t x = __shfl_up(sum, o);
    if (lane >= uint32_t(o)) sum += x;
  }
  if (lane == kWave - 1) wave_rounds[w] = sum;
  __syncthreads();
  uint32_t first = sum - rounds;
  for (uint32_t i = 0; i < w; ++i) first += wave_rounds[i];
  if (t < A.item[7]) S.item[t] = first | rounds << 16;
  __syncthreads();
  each_item(A, [&](auto width, uint32_t i, uint32_t v, bool row) {
    constexpr int W = decltype(width)::value;
    const uint32_t it = S.item[i], rounds = it >> 16;
    uint64_t *ids = S.ids + (it & 0xFFFF) * kWave + lane;
    const uint32_t end = row ? A.off[v + 1] : 0;
    uint32_t e = row ? A.off[v] + lane % W : 0;
    for (uint32_t q = 0; q < rounds; ++q) {
      uint64_t x = 0;
      for (int k = 0; k < 4; ++k, e += W) x |= uint64_t(8 * (e < end ? A.src[e] : N)) << (16 * k);
      ids[q * kWave] = x;
    }
  });
  __syncthreads();
  bool stop = false;
  int l = A.first;
  while (l < A.last && !stop) {  // uniform
    const uint32_t c = (l - A.first) & 1 ? list : 0, cn = list - c;
    each_item(A, [&](auto width, uint32_t i, uint32_t v, bool row) {
      constexpr int W = decltype(width)::value;
      if (T::dynamic) {
        row = row && S.vaff[v];
        if (__ballot(row) == 0) return;
      }
      const uint32_t it = __builtin_amdgcn_readfirstlane(S.item[i]), rounds = it >> 16;
      const uint64_t *ids = S.ids + (it & 0xFFFF) * kWave + lane;
      double s0 = 0.0, s1 = 0.0;
      for (uint32_t q = 0; q < rounds; ++q) {
        const uint64_t x = ids[q * kWave];
        const uint32_t lo = uint32_t(x), hi = uint32_t(x >> 32);
        s0 += at(S, c, lo & 0xFFFF) + at(S, c, lo >> 16);
        s1 += at(S, c, hi & 0xFFFF) + at(S, c, hi >> 16);
      }
      const double cv = group_sum<W>(s0 + s1);
      if (row && lane % W == 0) at(S, cn, 8 * v) = cv;
    });
    __syncthreads();
    double emax = 0.0;
    for (uint32_t v = t; v < N; v += kSmallBlock) emax = fmax(emax, small_finish<VARIANT>(A, S, c, cn, v));
    ++l;
    stop = __syncthreads_or(emax >= A.tol) == 0;  // no change reached the tolerance (as report_change has it)
    if constexpr (T::frontier) {
      if (!stop) {  // rows not affected become so if an in-neighbour is in the frontier
        each_item(A, [&](auto, uint32_t i, uint32_t v, bool row) {
          row = row && !S.vaff[v];
          if (__ballot(row) == 0) return;
          const uint32_t it = __builtin_amdgcn_readfirstlane(S.item[i]), rounds = it >> 16;
          const uint64_t *ids = S.ids + (it & 0xFFFF) * kWave + lane;
          uint32_t hit = 0;
          for (uint32_t q = 0; q < rounds; ++q) {
            const uint64_t x = ids[q * kWave];
            const uint32_t lo = uint32_t(x), hi = uint32_t(x >> 32);
            hit |= S.naff[(lo & 0xFFFF) >> 3] | S.naff[lo >> 19] | S.naff[(hi & 0xFFFF) >> 3] | S.naff[hi >> 19];
          }
          if (row && hit) S.vaff[v] = 1;
        });
        __syncthreads();
      }
    }
  }
  for (uint32_t v = t; v < N; v += kSmallBlock) {
    A.rank[l & 1][v] = S.r[v];
    if constexpr (T::dynamic) A.vaff[v] = S.vaff[v];
  }
  if (t == 0) tell_host(A.host + (stop ? 1 : 0), l);
}

}  // namespace

hipError_t launch_small_solve(int variant, const SmallArgs &A, hipStream_t s) {
  switch (variant) {
    case kPlain: small_solve_kernel<kPlain><<<1, kSmallBlock, 0, s>>>(A); break;
    case kTraversal: small_solve_kernel<kTraversal><<<1, kSmallBlock, 0, s>>>(A); break;
    case kFrontier: small_solve_kernel<kFrontier><<<1, kSmallBlock, 0, s>>>(A); break;
    case kPrune: small_solve_kernel<kPrune><<<1, kSmallBlock, 0, s>>>(A); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace prh
