// Walks that build the alias table of the current vertex on the fly (replaces OnlineWalkKernel /
// OnlineWalkShMem / OnlineWalkGMem of src/online_walk.cu:82-166,245-327 and online_walk_gmem.cu).
//
// Static bias (DeepWalk, PPR): the table of a vertex does not depend on the walker, so each
// step builds, once, the tables of the distinct vertices the live walkers stand on that were
// not built earlier in the call, through the kernels of the offline build, and then advances
// every walker by one draw.  The draws, and so the paths, are those of the offline walk.
//
// node2vec: the weights of a step depend on the walker's previous vertex
// (src/api/bias_node2vec.cu:15-27), so each (walker, step) builds its own table.
#include "sky_build_fused.h"
#include "sky_graph.h"
#include "sky_step_draw.h"

namespace sky {

__global__ __launch_bounds__(256) void walk_init_kernel(const uint32_t* __restrict__ seeds, uint32_t N, uint32_t len,
                                                        uint32_t V, uint32_t* __restrict__ paths,
                                                        uint32_t* __restrict__ lengths, CallDevice* __restrict__ call,
                                                        uint32_t* __restrict__ bitmap, uint32_t words,
                                                        uint32_t* __restrict__ counts, uint32_t ncounts) {
  call_stamp(call);
  const uint32_t i0 = blockIdx.x * 256u + threadIdx.x, step = gridDim.x * 256u;
  for (uint32_t i = i0; i < words; i += step) bitmap[i] = 0;
  for (uint32_t i = i0; i < ncounts; i += step) counts[i] = 0;
  for (uint32_t i = i0; i < N; i += step) {
    const uint32_t v = seeds[i];
    paths[(size_t)i * (len + 1)] = v;
    // "still walking"; a walker that stops at step s stores s < len.  A start vertex that does not exist
    // is recorded and never left.
    lengths[i] = v < V ? len : 0u;
  }
}
constexpr uint32_t WALK_INIT_BLOCKS = 2048;

// The draw of step s - 1 (the rows it needs have just been built) and, for the walkers that go on, the stop and dead-end
// tests of step s: the vertices whose table is still missing are appended to the segments of the degree
// classes, or, without segments (list not null), to a plain list.  counts[s * FRONTIER_WORDS ...] are the rows appended
// per class (or, in word 0, to the list), and in the last word the walkers that will draw.
constexpr uint32_t LIVE_WORD = FRONTIER_WORDS - 1;
static_assert((int)LIVE_WORD >= (int)CLS_COUNT, "no class counts in the word of the live walkers");
__global__ __launch_bounds__(256) void walk_advance_kernel(const uint32_t* __restrict__ xadj,
                                                           const uint32_t* __restrict__ adjncy,
                                                           const AliasEntry* __restrict__ table, int8_t* __restrict__ valid,
                                                           uint32_t N, uint32_t len, uint32_t s, float stop_prob, uint64_t seed,
                                                           uint32_t* __restrict__ paths, uint32_t* __restrict__ lengths,
                                                           uint32_t* bitmap, FrontierLists f, uint32_t* __restrict__ list,
                                                           uint32_t* __restrict__ all_counts, uint32_t* __restrict__ report) {
  __shared__ uint32_t s_cnt[CLS_COUNT], s_base[CLS_COUNT];
  __shared__ uint32_t s_n[256 / 64 + 1];
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  uint32_t* const counts = all_counts + (size_t)s * FRONTIER_WORDS;
  // how many walkers drew in the step before, for the host
  if (report && s && blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_store(report + s - 1, all_counts[(size_t)(s - 1) * FRONTIER_WORDS + LIVE_WORD], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  bool draws = false, fresh = false;
  uint32_t v = 0;
  if (i < N && lengths[i] == len) {
    uint32_t* path = paths + (size_t)i * (len + 1);
    bool walking = true;
    v = path[s ? s - 1 : 0];
    if (s) {
      const u32x4 r = philox(seed, i, s - 1, 0, DOM_WALK);
      const uint32_t off = xadj[v], deg = xadj[v + 1] - off;
      const uint32_t col = __umulhi(r.x, deg);
      const AliasEntry e = table[off + col];
      const uint32_t cand = u24(r.y) < e.prob ? col : e.alias;
      if (cand == SKY_INVALID) {
        lengths[i] = s - 1;
        walking = false;
      } else {
        v = adjncy[off + cand];
        path[s] = v;
      }
    }
    if (walking && s < len) {
      const u32x4 r = philox(seed, i, s, 0, DOM_WALK);
      if ((stop_prob > 0.0f && u24(r.z) < stop_prob) || xadj[v + 1] == xadj[v]) {
        lengths[i] = s;
      } else {
        draws = true;
        const uint32_t bit = 1u << (v & 31);
        if (!(bitmap[v >> 5] & bit)) fresh = !(atomicOr(&bitmap[v >> 5], bit) & bit);
      }
    }
  }
  if (s == len) return;
  if (!__syncthreads_or(draws)) return;
  const unsigned long long md = __ballot(draws);
  if (md && (threadIdx.x & 63) == (uint32_t)__ffsll((long long)md) - 1) atomicAdd(&counts[LIVE_WORD], (uint32_t)__popcll(md));
  if (list) append_list(fresh, v, list, counts, s_n);
  else append_rows(fresh, v, xadj, valid, f, counts, s_cnt, s_base);
}

int walk_online_node2vec(sky_graph* g, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                         float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                         double* seconds);

// Option online_full_build: -1: decide by the estimate below; 0: always build lazily, step by step; 1: always build
// every row first.

// Estimated milliseconds of the two ways to serve a static-bias online walk.  A lazy round costs a
// host round trip and a handful of small launches (about 1/8 ms measured), and the rounds together
// build at most min(N * len, V) rows; the full build runs at about 1.3e8 edges per millisecond.
static bool online_prefers_full_build(const sky_graph* g, uint32_t N, uint32_t len) {
  const long long mode = option(g, OPT_ONLINE_FULL_BUILD);
  if (mode >= 0) return mode != 0;
  const double all_ms = (double)g->E / 1.3e8;
  const double visited = std::min(1.0, (double)N * len / std::max(1u, g->V));
  return 0.4 + all_ms < 0.125 * len + visited * all_ms;
}

int walk_online(sky_graph* g, int bias_kind, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                double* seconds) {
  if (bias_kind == SKY_BIAS_NODE2VEC_REJECT)
    return walk_node2vec_reject(g, p, q, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds);
  if (bias_kind == SKY_BIAS_NODE2VEC)
    return walk_online_node2vec(g, p, q, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds);
  // Tables that already exist are used as they are.  Otherwise one build of every row, then the
  // offline kernel, is taken when it is expected to cost less than len rounds of lazy builds, each
  // of which waits for the host; the paths are the same either way.
  double build_sec = 0;
  if (!g->has_tables && N && len && online_prefers_full_build(g, N, len)) SKY_TRY(build_all_tables(g, &build_sec));
  if (g->has_tables) {
    SKY_TRY(walk_offline(g, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds));
    if (seconds) *seconds += build_sec;
    return SKY_OK;
  }
  hipStream_t st = g->stream;
  CallDevice* call = nullptr;
  uint32_t *bitmap = nullptr, *list = nullptr, *counts = nullptr;
  const uint32_t words = (g->V + 31) / 32;
  // Normally no step waits for the device: the rows of a step's list stay there (build_frontier), and whether any
  // walker still walks comes back through pinned host words that the host reads as they arrive, some steps behind
  // what it has enqueued; the steps enqueued past the last walker's end find nothing to do.
  const bool dev_sized = fused_possible(g) && option(g, OPT_ONLINE_DEVICE_SIZED) != 0;
  FrontierLists front;
  SKY_TRY(ensure_table_storage(g));
  const uint32_t upper = std::min(N, g->V);
  if (dev_sized) {
    SKY_TRY(frontier_lists(g, upper, &front));
    if (g->live_report_cap < len) {
      if (g->live_report) SKY_HIP(hipHostFree(g->live_report));
      g->live_report = nullptr;
      g->live_report_cap = 0;
      SKY_HIP(hipHostMalloc((void**)&g->live_report, (size_t)len * 4, hipHostMallocCoherent));
      g->live_report_cap = len;
    }
    for (uint32_t s = 0; s < len; ++s) g->live_report[s] = 0xFFFFFFFFu;  // "not reported yet"
    ++g->frontier_epoch;
  } else {
    SKY_TRY(prepare_build_scratch(g, upper));
    SKY_TRY(pool_get(g, sky_graph::POOL_LIST, (size_t)upper * 4, (void**)&list));
  }
  const uint64_t ncounts = ((uint64_t)len + 1) * FRONTIER_WORDS;
  if (ncounts > 0xFFFFFFFFull) return fail(SKY_ERR_LIMIT, "walk: too many steps");
  SKY_TRY(pool_get(g, sky_graph::POOL_BITMAP, (size_t)words * 4, (void**)&bitmap));
  SKY_TRY(pool_get(g, sky_graph::POOL_FRONT, (size_t)ncounts * 4, (void**)&counts));
  SKY_TRY(call_begin(g, &call));
  if (N) {
    const uint32_t blocks = (uint32_t)(((uint64_t)N + 255) / 256);
    hipLaunchKernelGGL(walk_init_kernel, dim3(std::min(std::max(blocks, (words + 255) / 256), WALK_INIT_BLOCKS)), dim3(256), 0, st,
                       seeds, N, len, g->V, paths, lengths, call, bitmap, words, counts, (uint32_t)ncounts);
    for (uint32_t s = 0; s <= len; ++s) {
      hipLaunchKernelGGL(walk_advance_kernel, dim3(blocks), dim3(256), 0, st, g->xadj, g->adjncy, g->table, g->valid, N, len, s,
                         stop_prob, seed, paths, lengths, bitmap, front, list, counts, dev_sized ? g->live_report : nullptr);
      if (s == len) break;
      if (dev_sized) {
        bool ended = false;
        for (uint32_t k = 0; k < s && !ended; ++k) ended = *(volatile uint32_t*)&g->live_report[k] == 0;
        if (ended) break;  // a step that has run found no walker left
        SKY_TRY(build_frontier(g, front, counts + (size_t)s * FRONTIER_WORDS, bitmap, g->frontier_epoch));
      } else {
        uint32_t cnt[FRONTIER_WORDS] = {0};
        SKY_HIP(hipMemcpyAsync(cnt, counts + (size_t)s * FRONTIER_WORDS, sizeof(cnt), hipMemcpyDeviceToHost, st));
        SKY_HIP(hipStreamSynchronize(st));
        if (cnt[LIVE_WORD] == 0) break;  // every walker has stopped
        SKY_TRY(build_rows(g, list, cnt[0], nullptr));
      }
    }
  }
  return call_end(g, sampled, seconds, lengths, N);
}

// ---------------------------------------------------------------- node2vec
// One workgroup per (walker, step) evaluates the one entry of the step's second-order table that the draw
// reads (step_draw_slot of sky_step_draw.h).
struct N2vRow {
  const float* w;
  const uint32_t* nbr;
  const uint32_t* prow;
  uint32_t pdeg, prev;
  bool has_prev;
  float p, q;
  // weight of the edge in slot k after the second-order factor (src/api/bias_node2vec.cu:15-27)
  __device__ __forceinline__ float operator()(uint32_t k) const {
    float x = w[k];
    if (has_prev) {
      const uint32_t t = nbr[k];
      if (t == prev) x = __fdiv_rn(x, p);
      else if (!row_contains(prow, pdeg, t)) x = __fdiv_rn(x, q);
    }
    return clamp_weight(x);
  }
};

__global__ __launch_bounds__(N2V_T) void n2v_step_kernel(const uint32_t* __restrict__ xadj,
                                                         const uint32_t* __restrict__ adjncy,
                                                         const float* __restrict__ wgt, uint32_t len, uint32_t s,
                                                         float p, float q, float stop_prob, uint64_t seed,
                                                         uint32_t* __restrict__ paths,
                                                         uint32_t* __restrict__ lengths) {
  const uint32_t i = blockIdx.x;
  const int tid = threadIdx.x;
  if (lengths[i] != len) return;  // stopped at an earlier step
  const u32x4 r = philox(seed, i, s, 0, DOM_WALK);
  uint32_t* path = paths + (size_t)i * (len + 1);
  const uint32_t v = path[s];
  const uint32_t off = xadj[v], d = xadj[v + 1] - off;
  if ((stop_prob > 0.0f && u24(r.z) < stop_prob) || d == 0) {
    if (tid == 0) lengths[i] = s;
    return;
  }
  N2vRow row;
  row.w = wgt + off;
  row.nbr = adjncy + off;
  row.has_prev = s > 0;
  row.prev = s > 0 ? path[s - 1] : 0;
  row.prow = adjncy + xadj[row.prev];
  row.pdeg = xadj[row.prev + 1] - xadj[row.prev];
  row.p = p;
  row.q = q;
  const uint32_t cand = step_draw_slot(row, d, r);
  if (tid == 0) {
    if (cand == NONE_SLOT) lengths[i] = s;
    else path[s + 1] = row.nbr[cand];
  }
}

int walk_online_node2vec(sky_graph* g, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                         float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                         double* seconds) {
  hipStream_t st = g->stream;
  CallDevice* call = nullptr;
  SKY_TRY(call_begin(g, &call));
  if (N) {
    hipLaunchKernelGGL(walk_init_kernel, dim3(std::min((uint32_t)(((uint64_t)N + 255) / 256), WALK_INIT_BLOCKS)), dim3(256), 0, st,
                       seeds, N, len, g->V, paths, lengths, call, (uint32_t*)nullptr, 0u, (uint32_t*)nullptr, 0u);
    for (uint32_t s = 0; s < len; ++s)
      hipLaunchKernelGGL(n2v_step_kernel, dim3(N), dim3(N2V_T), 0, st, g->xadj, g->adjncy, g->adjwgt, len, s, p, q, stop_prob,
                         seed, paths, lengths);
  }
  return call_end(g, sampled, seconds, lengths, N);
}

}  // namespace sky
