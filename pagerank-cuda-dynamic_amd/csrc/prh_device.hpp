// prh_device.hpp -- device-side building blocks for the gfx950 (CDNA4, wave64) PageRank kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "prh_internal.hpp"

namespace prh {

// ---------------------------------------------------------------------------------------------------------
// Cross-lane moves. DPP (data-parallel primitives) moves within a 16-lane row are free operand modifiers on
// VALU moves; ds_swizzle crosses the two rows of a 32-lane half; readlane crosses the halves. A 64-bit value
// moves as its two 32-bit halves. All lanes of the wave must be active when these are called.
// ---------------------------------------------------------------------------------------------------------
enum : int {
  kDppQuadSwap1 = 0xB1,       // quad_perm [1,0,3,2]: lane i <- lane i^1
  kDppQuadSwap2 = 0x4E,       // quad_perm [2,3,0,1]: lane i <- lane i^2
  kDppRowHalfMirror = 0x141,  // lane i <- lane 7-i within each 8-lane half-row
  kDppRowMirror = 0x140,      // lane i <- lane 15-i within each 16-lane row
};

template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// ds_swizzle in bit-mask mode with xor 16 (offset = and 0x1F | xor 0x10 << 10): lane i <- lane i^16 within 32.
__device__ __forceinline__ double swizzle_xor16(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_ds_swizzle(int(b), 0x401F);
  const int hi = __builtin_amdgcn_ds_swizzle(int(b >> 32), 0x401F);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double read_lane(double x, int lane) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane(int(b), lane);
  const int hi = __builtin_amdgcn_readlane(int(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Sum over aligned groups of W lanes (W = 1, 2, 4, ..., 64). Each step pairs lanes symmetrically, so every lane
// of a group ends with the same value (for W = 64 the result is wave-uniform).
template <int W>
__device__ __forceinline__ double group_sum(double x) {
  if constexpr (W >= 2) x += dpp_move<kDppQuadSwap1>(x);
  if constexpr (W >= 4) x += dpp_move<kDppQuadSwap2>(x);
  if constexpr (W >= 8) x += dpp_move<kDppRowHalfMirror>(x);
  if constexpr (W >= 16) x += dpp_move<kDppRowMirror>(x);
  if constexpr (W >= 32) x += swizzle_xor16(x);
  if constexpr (W >= 64) x = read_lane(x, 0) + read_lane(x, 32);
  return x;
}

__device__ __forceinline__ int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)); }

// Number of set bits of a 64-bit wave mask below this lane.
__device__ __forceinline__ unsigned lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi(unsigned(mask >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(mask), 0));
}

// ---------------------------------------------------------------------------------------------------------
// Iteration control on the device. err[l] tells whether iteration l's L-inf change
// reached the tolerance (see report_change); *done records the first
// iteration index l at which err[l-1] < tolerance was seen, after which every kernel of later iterations exits
// at once. This keeps "stop at the first iteration whose change is below tolerance" without a host round trip.
// ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ int iter_index(const LoopCtl &c) { return c.l >= 0 ? c.l : c.done[1] - 1 - c.l; }

// The loop only asks whether an iteration's largest change is below the tolerance, so nothing needs that maximum: a
// wave that saw a change of at least tol says so with a plain store of one value, the same from every wave (infinity,
// which no tolerance exceeds); a slot left 0 means every change was below tol (with tol = 0 the loop never stops, as
// 0 < 0 is false). A maximum kept by one atomic per workgroup made the workgroups of a launch
// queue on one address: RMAT-16, 500 of them, 29.0 -> 26.6 us per iteration without it (and 18.5 -> 11.3 us once the
// row plan uses 1,000). NaN changes count as no change, as with a maximum.
constexpr unsigned long long kChanged = 0x7FF0000000000000ull;  // +infinity

// `e`: the lane's largest change. Every lane of the wave must call it.
__device__ __forceinline__ void report_change(const LoopCtl &c, double e) {
  if (__ballot(e >= c.tol) != 0 && lane_id() == 0) c.err[iter_index(c)] = kChanged;
}

// A word of host memory (pinned): the store is visible to the host while the launches that follow run.
__device__ __forceinline__ void tell_host(int *p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Entry test for the first kernel of iteration l; all threads of a block agree.
// done and err[l-1] were last written by earlier launches, whose completion made them visible: plain loads suffice. A
// volatile read here would be a system-scope load at the start of every wave.
// The test needs two loads; a workgroup's item can be loaded with them instead of after the test. `broken`, never true, is
// a condition on the item: it keeps the compiler from moving the item's load behind the test. (The kernels that pass none
// wait for done before they load err[l-1].) (An empty asm statement in its
// place made the later uniform loads vector loads: RMAT-20, blocked, 3.60 -> 4.17 ms per solve.) Blocked plan, per solve,
// test first -> together, and accumulate's first batch before its sums are cleared: RMAT-20 3.59 -> 3.46 ms, RMAT-24
// 40.6 -> 40.4, weighted forward and backward on RMAT-20 9.79 -> 9.48.
struct LoopState {
  int done, l;
  double e;
};
__device__ __forceinline__ LoopState loop_state(const LoopCtl &c, bool broken = false) {
  const int done = *c.done, l = iter_index(c);
  return {done | int(broken), l, l > 0 ? __longlong_as_double((long long)c.err[l - 1]) : c.tol};
}

__device__ __forceinline__ bool iteration_begin(const LoopCtl &c, const LoopState &s) {
  if (s.done || s.l >= c.max_iter) return false;
  if (s.e < c.tol) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *(volatile int *)c.done = s.l;
      if (c.host) tell_host(c.host + 1, s.l);
    }
    return false;
  }
  return true;
}
__device__ __forceinline__ bool iteration_begin(const LoopCtl &c) { return iteration_begin(c, loop_state(c)); }

// The first kernel of an iteration tells the host that it has run, at its end: a store before the kernel's loads would
// keep the compiler from making the uniform ones scalar (RMAT-20, blocked: 3.79 -> 4.41 ms per solve).
__device__ __forceinline__ void report_begun(const LoopCtl &c) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && c.host) tell_host(c.host, iter_index(c) + 1);
}

// Entry test for kernels that follow the rank update within iteration l (frontier extension).
__device__ __forceinline__ bool iteration_continues(const LoopCtl &c) {
  const int done = *c.done, l = iter_index(c);
  if (done || l >= c.max_iter) return false;
  return __longlong_as_double((long long)c.err[l]) >= c.tol;
}

}  // namespace prh
