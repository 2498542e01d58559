// solve.hip -- the solver driver: restates pagerankInvokeCuda + pagerankLoopCuU (pagerankCuda.hxx:675-692,
// :713-849) for one HIP stream. Per repeat, partition (and initial ranks) = initialization time, affected marking =
// marking time, iterations = computation time, each measured with HIP events. Iterations run without a host
// round trip per iteration: convergence is detected on the device (LoopCtl), the device tells the host in pinned memory
// how far it is, and the host keeps a few iterations enqueued ahead of it until the device says it has stopped, so the
// iteration count and final ranks equal those of the per-iteration check.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "capi_internal.hpp"

namespace prhc {


int stage_batch(prh_context *c, const prh_graph *g, const uint32_t *du, const uint32_t *dv, size_t nd,
                const uint32_t *iu, size_t ni, bool host, DevBatch &b) {
  b.ND = nd;
  b.NI = ni;
  if (nd + ni == 0) return PRH_SUCCESS;
  if ((nd && (!du || !dv)) || (ni && !iu)) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "null batch array");
  PRH_CHECK(ensure(c, c->batch, 2 * nd + ni));
  uint32_t *d = c->batch.p;
  const hipMemcpyKind kind = host ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
  if (nd) {
    PRH_HIP(c, hipMemcpyAsync(d, du, nd * 4, kind, c->stream));
    PRH_HIP(c, hipMemcpyAsync(d + nd, dv, nd * 4, kind, c->stream));
  }
  if (ni) PRH_HIP(c, hipMemcpyAsync(d + 2 * nd, iu, ni * 4, kind, c->stream));
  const uint32_t N = g->N;
  PRH_CHECK(ensure(c, c->flags, 4));
  PRH_HIP(c, prh::launch_fill_i32(c->flags.p, 0, 1, c->stream));
  PRH_HIP(c, prh::launch_validate_ids(d, 2 * nd + ni, N, c->flags.p, 1, c->stream));
  PRH_HIP(c, hipMemcpyAsync(c->pinned, c->flags.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  PRH_HIP(c, hipStreamSynchronize(c->stream));
  if (*reinterpret_cast<int *>(c->pinned)) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "batch vertex id >= N (%u)", N);
  PRH_HIP(c, prh::launch_map_ids(d, 2 * nd + ni, g->inv, c->stream));
  b.delu = d;
  b.delv = d + nd;
  b.insu = d + 2 * nd;
  return PRH_SUCCESS;
}

// Marking phase of the dynamic methods (pagerankCuda.hxx:821 with the fm lambdas :926-928, :955-957, :984-986),
// on the layout's out-CSR with layout ids.
// xo: the out-degree schedule and chunk table (out_schedule), needed by the traversal levels only.
int mark_affected(prh_context *c, const prh_graph *g, int method, const DevBatch &b, const prh::ExtendArgs &xo) {
  const uint32_t N = g->N;
  hipStream_t s = c->stream;
  PRH_HIP(c, prh::launch_fill_u8(c->vaff.p, 0, N, s));
  PRH_HIP(c, prh::launch_fill_u8(c->naff.p, 0, N, s));
  if (b.ND + b.NI == 0) return PRH_SUCCESS;
  PRH_HIP(c, prh::launch_mark_partial(c->naff.p, c->vaff.p, b.delu, b.delv, b.ND, b.insu, b.NI, s));
  // The flagged vertices are the batch's sources: extend from the batch list.
  const size_t nb = b.ND + b.NI + 1;
  PRH_CHECK(ensure(c, c->ext_chunks, 2 * nb));
  size_t tmp_bytes = 0;
  PRH_HIP(c, prh::launch_extend_batch(c->vaff.p, c->naff.p, b.delu, b.ND, b.insu, b.NI, g->l_out_off, g->l_out_dst,
                                      c->ext_chunks.p, c->ext_chunks.p + nb, nullptr, tmp_bytes, s));
  PRH_CHECK(ensure(c, c->ext_tmp, std::max<size_t>(tmp_bytes, 16)));
  PRH_HIP(c, prh::launch_extend_batch(c->vaff.p, c->naff.p, b.delu, b.ND, b.insu, b.NI, g->l_out_off, g->l_out_dst,
                                      c->ext_chunks.p, c->ext_chunks.p + nb, c->ext_tmp.p, tmp_bytes, s));
  if (method != PRH_DYNAMIC_TRAVERSAL) return PRH_SUCCESS;
  // Traversal closure: breadth-first levels from every marked vertex until no vertex is newly marked.
  PRH_CHECK(ensure(c, c->flags, 4));
  uint8_t *front = c->naff.p, *fresh = c->buff.p;
  PRH_HIP(c, hipMemcpyAsync(front, c->vaff.p, N, hipMemcpyDeviceToDevice, s));
  for (;;) {
    PRH_HIP(c, prh::launch_fill_u8(fresh, 0, N, s));
    PRH_HIP(c, prh::launch_fill_i32(c->flags.p + 1, 0, 1, s));
    prh::ExtendArgs T = xo;
    T.vaff = c->vaff.p;
    T.naff = front;
    T.off = g->l_out_off;
    T.dst = g->l_out_dst;
    T.fresh = fresh;
    T.changed = c->flags.p + 1;
    T.direction = nullptr;
    PRH_HIP(c, prh::launch_extend(T, s));
    PRH_HIP(c, hipMemcpyAsync(c->pinned, c->flags.p + 1, sizeof(int), hipMemcpyDeviceToHost, s));
    PRH_HIP(c, hipStreamSynchronize(s));
    if (*reinterpret_cast<int *>(c->pinned) == 0) break;
    std::swap(front, fresh);
  }
  return PRH_SUCCESS;
}

void reset_progress(prh_context *c) {
  __atomic_store_n(c->progress, 0, __ATOMIC_RELAXED);
  __atomic_store_n(c->progress + 1, 0, __ATOMIC_RELEASE);
}

// Polls for a few microseconds (iterations of small graphs last no longer), then offers its core to other threads between
// polls, and from a millisecond on sleeps between them: iterations that long leave the host time, as some are enqueued
// ahead. Polling throughout -> this, blocked solves of 1M vertices: four threads on one core 246 -> 292 a second, on two
// cores 323 -> 334; one thread 246 and 246 (64K vertices 1438 and 1432). Batched PPR, runs of 29 ms: the calling thread is
// busy for 13 of 116 ms.
int wait_progress(prh_context *c, int begun) {
  using clock = std::chrono::steady_clock;
  using std::chrono::microseconds;
  const auto waiting = [&]() {
    return !loop_stopped(c) && __atomic_load_n(c->progress, __ATOMIC_ACQUIRE) < begun;
  };
  for (int i = 0; i < 256; ++i)
    if (!waiting()) return PRH_SUCCESS;
  const clock::time_point begin = clock::now();
  clock::time_point query = begin + microseconds(100000);
  while (waiting()) {
    const clock::time_point now = clock::now();
    if (now - begin > microseconds(1000)) std::this_thread::sleep_for(microseconds(50));
    else if (now - begin > microseconds(20)) std::this_thread::yield();
    // Long iterations, or launches that failed: ask the stream now and then (a query adds a marker to it).
    if (now < query) continue;
    query = now + microseconds(100000);
    const hipError_t e = hipStreamQuery(c->stream);
    if (e == hipSuccess) break;
    if (e != hipErrorNotReady) return fail(c, PRH_ERROR_DEVICE, "iterations: %s", hipGetErrorString(e));
  }
  return PRH_SUCCESS;
}

int end_loop(prh_context *c, int max_iter, int *n) {
  if (!loop_stopped(c)) PRH_HIP(c, hipStreamSynchronize(c->stream));
  const int k = loop_stopped(c);
  *n = k ? k : max_iter;
  return PRH_SUCCESS;
}

int ensure_workspace(prh_context *c, uint32_t N, bool dynamic, int L) {
  for (int i = 0; i < 2; ++i) {
    PRH_CHECK(ensure(c, c->rank[i], N));
    PRH_CHECK(ensure(c, c->contrib[i], N));
  }
  if (dynamic) {
    PRH_CHECK(ensure(c, c->sched_out, N));
    PRH_CHECK(ensure(c, c->vaff, N));
    PRH_CHECK(ensure(c, c->naff, (size_t(N) + 3) / 4 * 4));  // whole 32-bit words (the batch extension's claims)
    PRH_CHECK(ensure(c, c->buff, N));
  }
  PRH_CHECK(ensure(c, c->loop, size_t(L) + 1));
  PRH_CHECK(ensure(c, c->flags, 4));
  return PRH_SUCCESS;
}

// Start ranks in layout order: rank[0][i] = q[perm[i]] (q staged through contrib[1], which the initialisation
// overwrites).
static int load_initial_ranks(prh_context *c, const prh_graph *g, const double *q, bool host) {
  const double *src = q;
  if (host) {
    PRH_HIP(c, hipMemcpyAsync(c->contrib[1].p, q, size_t(g->N) * 8, hipMemcpyHostToDevice, c->stream));
    src = c->contrib[1].p;
  }
  PRH_HIP(c, prh::launch_gather_f64(src, g->perm, g->N, c->rank[0].p, c->stream));
  return PRH_SUCCESS;
}

// Edges up to which a row plan's frontier extension (direction chosen by the library) is part of the next iteration's
// update, whose unaffected rows look at their in-neighbours' flags (RankArgs::prev), instead of a launch of its own for
// which the update sums what either direction would cost. Per solve, launch of its own -> inside: RMAT, 16 edges a vertex,
// DF: 5,000 vertices 794 -> 523 us, 64K 1019 -> 729; 20 edges: 200K 1720 -> 1262, 1M 5.74 -> 5.17 ms; DF-P at 1M with 1e-3
// of the edges changed 4.25 -> 4.24. Grids, where ten changed edges leave nearly all rows unaffected to the end: 1.2M edges
// 562 -> 324 us, 11.2M 1154 -> 937. Both sides meet at about 20M edges (40M, DF-P: 8.3 -> 8.7 ms).
constexpr uint64_t kExtendInside = uint64_t(1) << 24;

// Whether a frontier solve that pushes its extension (direction 0) reads the in-CSR past the Infinity Cache (256 MB): where
// an iteration's other arrays (the out-CSR and its schedule, ranks and contributions, degrees, flags) fit there without the
// in-CSR but not with it. Per DF solve through the cache -> past it, 1e-2 of the edges changed: 4M vertices, 16M edges
// 25.1 -> 22.2 ms, RMAT-21 23.8 -> 22.4; where all of it fits (RMAT-20) 10.5 -> 11.8, where not even the rest does
// (RMAT-22) 48.6 -> 49.5. The pull and the solves without a frontier gain nothing from it (RMAT-21: 14.6 -> 16.7, pulled).
static bool stream_in_csr(const prh_graph *g) {
  const uint64_t cache = uint64_t(256) << 20, N = g->N, csr = 4 * (g->M + N), rest = csr + 42 * N;
  return rest <= cache && csr + rest > cache;
}

// The bands and items of a small graph's solve; false if the graph does not fit. (That the ids' 16-bit byte offsets hold
// every vertex follows from the size of LDS. The out-degrees are kept in 16 bits too; M bounds them only where the graph
// came with its out-CSR, whose rows they are checked against.)
static bool small_plan(const prh_graph *g, prh::SmallArgs &A) {
  if (g->layout != 0 || g->updated || g->M > 65535 || g->max_outdeg > 65535 ||
      prh::small_lds(g->N, 0, g->M / 256) > prh::kSmallLds)
    return false;
  A.N = g->N;
  A.band[0] = A.item[0] = A.rounds = 0;
  for (int k = 0; k < 7; ++k) {
    A.band[k + 1] = k == 6 ? g->N : std::max(A.band[k], layout_rows_above(g, prh::kSmallEdges * (32u >> k)));
    for (uint32_t v = A.band[k]; v < A.band[k + 1]; v += 1u << k) A.rounds += prh::small_rounds(g->sorted_deg[v], k);
    A.item[k + 1] = A.item[k] + (A.band[k + 1] - A.band[k] + (1u << k) - 1) / (1u << k);
  }
  return prh::small_lds(g->N, A.item[7], A.rounds) <= prh::kSmallLds && A.item[7] <= prh::kSmallBlock;
}

int solve_impl(prh_context *c, const prh_graph *g, int method, const prh_options *o, const uint32_t *du,
               const uint32_t *dv, size_t nd, const uint32_t *iu, size_t ni, const double *q, double *ranks,
               prh_stats *st, bool host, bool account_prep) {
  if (!c) return PRH_ERROR_INVALID_ARGUMENT;
  if (!g || !o || !valid_method(method)) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "null graph/options or bad method");
  if (g->ctx != c) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "graph belongs to another context");
  if (o->repeat < 1 || o->max_iterations < 0 || !(o->tolerance >= 0) || !(o->damping > 0 && o->damping < 1))
    return fail(c, PRH_ERROR_INVALID_ARGUMENT, "bad options (repeat >= 1, max_iterations >= 0, tolerance >= 0, 0 < damping < 1)");
  if (method != PRH_STATIC && !q) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "initial ranks required for this method");
  if (method == PRH_PRUNE_DYNAMIC_FRONTIER && g->dead_ends)
    return fail(c, PRH_ERROR_INVALID_GRAPH,
                "DF-P's closed-form update divides by the out-degree: %u vertices have none (dead ends)", g->dead_ends);
  const uint32_t N = g->N;
  prh_stats stats{};
  if (N == 0) {  // the reference returns an empty result for an empty graph (pagerankCuda.hxx:869)
    if (st) *st = stats;
    return PRH_SUCCESS;
  }
  if (!ranks) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "null ranks");
  const bool dynamic = method >= PRH_DYNAMIC_TRAVERSAL;
  const bool frontier = method >= PRH_DYNAMIC_FRONTIER;
  if (dynamic && !g->l_out_off) return fail(c, PRH_ERROR_UNSUPPORTED, "dynamic method needs the graph's out-CSR");
  const int L = o->max_iterations;
  const int variant = method == PRH_PRUNE_DYNAMIC_FRONTIER ? prh::kPrune
                      : method == PRH_DYNAMIC_FRONTIER    ? prh::kFrontier
                      : method == PRH_DYNAMIC_TRAVERSAL   ? prh::kTraversal
                                                          : prh::kPlain;
  hipStream_t s = c->stream;
  PRH_HIP(c, hipSetDevice(c->device));
  PRH_CHECK(ensure_workspace(c, N, dynamic, L));
  prh_graph *gm = const_cast<prh_graph *>(g);
  if (c->tuning.layout != g->layout && !g->updated) PRH_CHECK(relayout(c, gm, c->tuning.layout));
  const bool binned = c->tuning.blocking > 0;
  const bool window = !binned && c->tuning.window != 0 && g->layout == 1;
  const bool sliced = !binned && !window && variant == prh::kPlain && c->tuning.source_slices > 0 && g->layout == 0;
  // A row plan's small graph runs its iterations in one workgroup. (Timed launches are one per iteration.)
  prh::SmallArgs sm{};
  const bool small = !binned && !window && !sliced && !c->ktiming && small_plan(g, sm);
  if (!binned) PRH_CHECK(ensure_in_csr(c, gm));  // the other plans read the in-CSR in every iteration
  if (binned) PRH_CHECK(build_binned_plan(c, gm));
  else if (window) PRH_CHECK(build_window_plan(c, gm));
  else if (sliced) PRH_CHECK(build_sliced_plan(c, gm));
  else PRH_CHECK(build_rank_plan(c, gm));
  // One-time preparation of this graph not yet reported by a solve: its layout (built at upload) and the plan this
  // solve runs (built on first use), plus the extension schedule below.
  float prep = 0.0f;
  if (account_prep)
    prep = gm->layout_prep.take() + gm->update_prep.take() +
           (binned   ? gm->bin.prep.take()
            : window ? gm->win_prep.take()
            : sliced ? gm->sliced_prep.take()
                     : gm->plan_prep.take());
  DevBatch b;
  if (dynamic) PRH_CHECK(stage_batch(c, g, du, dv, nd, iu, ni, host, b));
  if (q && !host) {  // device initial ranks: reject NaN/Inf (the reference would propagate them)
    PRH_HIP(c, prh::launch_fill_i32(c->flags.p, 0, 1, s));
    PRH_HIP(c, prh::launch_check_finite(q, N, c->flags.p, 1, s));
    PRH_HIP(c, hipMemcpyAsync(c->pinned, c->flags.p, sizeof(int), hipMemcpyDeviceToHost, s));
    PRH_HIP(c, hipStreamSynchronize(s));
    if (*reinterpret_cast<int *>(c->pinned)) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "initial ranks not finite");
  }
  if (q && host)
    for (uint32_t v = 0; v < N; ++v)
      if (!std::isfinite(q[v])) return fail(c, PRH_ERROR_INVALID_ARGUMENT, "initial ranks not finite (vertex %u)", v);
  if (c->ktiming && c->kev.size() < size_t(2) * L) {
    size_t old = c->kev.size();
    c->kev.resize(size_t(2) * L);
    for (size_t i = old; i < c->kev.size(); ++i) PRH_HIP(c, hipEventCreate(&c->kev[i]));
  }
  double ti = 0, tm = 0, tc = 0;
  int iterations = 0;
  unsigned long long *err = c->loop.p;
  int *done = reinterpret_cast<int *>(c->loop.p + L);
  const int ahead = iterations_ahead(c, g->M);
  const prh::RankPlan &plan = g->plan;
  // Extension direction (frontier variants): 0 push only, 1 chosen per iteration from the rank launch's costs,
  // 2 pull only. The pull form splits rows at in-degree 64 (a wave each) and 4 (8 lanes each).
  const int dir_mode = frontier ? c->tuning.extension_direction : 0;
  const bool inside = dir_mode == 1 && !binned && !window && g->M <= kExtendInside;
  const bool stream = frontier && dir_mode == 0 && stream_in_csr(g);
  const bool dir_auto = dir_mode == 1 && !binned && !small && !inside;
  if (dir_auto) PRH_CHECK(ensure(c, c->ext_stats, 2 * prh::kCostSums));  // the sums of two iterations in turn
  const prh::PullArgs pull{c->vaff.p, c->naff.p, g->l_in_off, g->l_in_src, layout_rows_above(g, 64),
                           layout_rows_above(g, 4), N};
  for (int rep = 0; rep < o->repeat; ++rep) {
    if (q) PRH_CHECK(load_initial_ranks(c, g, q, host));  // untimed, as the reference's q copy (pagerankCuda.hxx:810)
    PRH_HIP(c, hipEventRecord(c->ev[0], s));
    // Initialisation. The degree classes the reference partitions here (pagerankCuda.hxx:811-814) are the row
    // ranges of the layout, fixed when the graph was prepared; the extension kernels' out-degree split is per solve.
    // The out-degree schedule serves the traversal levels and the row plan's frontier extension; the initial
    // extension runs from the batch list and the blocked plan extends inside its update.
    prh::ExtendArgs xo{};
    if (dynamic && (method == PRH_DYNAMIC_TRAVERSAL || (frontier && !binned && !small && !inside))) {
      PRH_CHECK(out_schedule(c, gm, xo));
      if (account_prep) prep += gm->out_prep.take();
    }
    // The blocked and banded plans compute contributions from the ranks where they read them and keep none.
    const bool keeps = !binned && !window;
    PRH_HIP(c, prh::launch_init_ranks(c->rank[0].p, c->rank[1].p, keeps ? c->contrib[0].p : nullptr,
                                      keeps ? c->contrib[1].p : nullptr, g->l_outdeg, N,
                                      q != nullptr, s));
    PRH_HIP(c, hipEventRecord(c->ev[1], s));
    if (dynamic) PRH_CHECK(mark_affected(c, g, method, b, xo));
    PRH_HIP(c, hipEventRecord(c->ev[2], s));
    // Iterations.
    if (!small) PRH_HIP(c, prh::launch_fill_u64(err, 0ull, size_t(L) + 1, s));
    if (dir_auto)
      PRH_HIP(c, prh::launch_fill_u64(reinterpret_cast<unsigned long long *>(c->ext_stats.p), 0ull,
                                      2 * prh::kCostSums, s));
    const double P = o->damping;
    const double C0 = (1 - P) / N;
    auto costs = [&](int l) { return dir_auto ? c->ext_stats.p + prh::kCostSums * (l & 1) : nullptr; };
    reset_progress(c);
    if (small) {
      sm.rank[0] = c->rank[0].p;
      sm.rank[1] = c->rank[1].p;
      sm.off = g->l_in_off;
      sm.src = g->l_in_src;
      sm.deg = g->l_outdeg;
      sm.vaff = c->vaff.p;
      sm.C0 = C0;
      sm.P = P;
      sm.D = o->frontier_tolerance;
      sm.C = o->prune_tolerance;
      sm.tol = o->tolerance;
      sm.host = c->progress;
    }
    for (int l = 0; small && l < L && !loop_stopped(c); l = sm.last) {
      sm.first = l;
      sm.last = L - l > prh::kSmallIterations ? l + prh::kSmallIterations : L;
      PRH_HIP(c, prh::launch_small_solve(variant, sm, s));
      PRH_CHECK(wait_progress(c, sm.last));
    }
    for (int l = 0; !small && l < L; ++l) {
      PRH_CHECK(wait_progress(c, l - ahead + 1));
      if (loop_stopped(c)) break;
      const prh::LoopCtl ctl{err, done, l, L, o->tolerance, c->progress};
      prh::RankArgs A{c->rank[(l + 1) & 1].p, c->rank[l & 1].p, c->contrib[(l + 1) & 1].p, c->contrib[l & 1].p,
                      c->naff.p, c->vaff.p, g->l_in_off, g->l_in_src, g->l_outdeg, C0, P, o->frontier_tolerance,
                      o->prune_tolerance, costs(l)};
      A.stream = stream;
      if (inside) {  // the flags of two iterations in turn (the second buffer is the traversal levels')
        uint8_t *const flags[2] = {c->naff.p, c->buff.p};
        A.naff = flags[l & 1];
        A.prev = l ? flags[(l - 1) & 1] : nullptr;
      }
      if (c->ktiming) PRH_HIP(c, hipEventRecord(c->kev[2 * l], s));
      hipEvent_t mark = c->ktiming ? c->kev[2 * l + 1] : nullptr;
      if (binned)
        PRH_HIP(c, prh::launch_binned_update(variant, A, g->bin.plan, ctl, frontier && l > 0, s, mark));
      else if (window) {
        PRH_HIP(c, prh::launch_window_update(variant, A, g->win, ctl, s));
        if (mark) PRH_HIP(c, hipEventRecord(mark, s));
      } else if (sliced) PRH_HIP(c, prh::launch_sliced_update(A, g->sliced, ctl, s, mark));
      else PRH_HIP(c, prh::launch_rank_update(variant, A, plan, ctl, s, mark));
      if (frontier && !binned && !inside) {  // else the extension is inside the next iteration's update
        prh::ExtendArgs E = xo;
        E.vaff = c->vaff.p;
        E.naff = c->naff.p;
        E.off = g->l_out_off;
        E.dst = g->l_out_dst;
        E.fresh = nullptr;
        E.changed = nullptr;
        E.direction = nullptr;
        PRH_HIP(c, prh::launch_extend_either(E, pull, costs(l), costs(l + 1), dir_mode, ctl, s));
      }
    }
    PRH_HIP(c, hipEventRecord(c->ev[3], s));
    int n = 0;
    PRH_CHECK(end_loop(c, L, &n));
    // Final ranks are in the buffer written by the last iteration (pagerankCuda.hxx:688, :826); back to the caller's
    // vertex order (scatter through perm), as the reference scatters to span (:827). The device has told how many
    // iterations it took, so these launches go out before the host waits for anything.
    if (rep + 1 == o->repeat) {
      const double *res = c->rank[n & 1].p;
      double *to = host ? c->contrib[(n + 1) & 1].p : ranks;
      PRH_HIP(c, prh::launch_scatter_f64(res, g->perm, N, to, s));
      if (host) PRH_CHECK(copy_to_host(c, ranks, to, size_t(N) * 8));
      else PRH_HIP(c, hipStreamSynchronize(s));
    } else {
      PRH_HIP(c, hipEventSynchronize(c->ev[3]));
    }
    float t01 = 0, t12 = 0, t23 = 0;
    PRH_HIP(c, hipEventElapsedTime(&t01, c->ev[0], c->ev[1]));
    PRH_HIP(c, hipEventElapsedTime(&t12, c->ev[1], c->ev[2]));
    PRH_HIP(c, hipEventElapsedTime(&t23, c->ev[2], c->ev[3]));
    ti += t01;
    tm += t12;
    tc += t23;
    iterations = n;
    if (c->ktiming) {
      for (int l = 0; l < n; ++l) {
        float ms = 0;
        PRH_HIP(c, hipEventElapsedTime(&ms, c->kev[2 * l], c->kev[2 * l + 1]));
        c->k_ms += ms;
        ++c->k_launches;
      }
    }
  }
  stats.iterations = iterations;
  stats.initialization_time = float(ti / o->repeat) + prep;
  stats.marking_time = float(tm / o->repeat);
  stats.computation_time = float(tc / o->repeat);
  stats.time = float((ti + tm + tc) / o->repeat) + prep;
  stats.preparation_time = prep;
  if (st) *st = stats;
  return PRH_SUCCESS;
}

}  // namespace prhc
