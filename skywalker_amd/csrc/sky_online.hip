// Walks on a graph without tables (replaces OnlineWalkKernel /
// OnlineWalkShMem / OnlineWalkGMem of src/online_walk.cu:82-166,245-327 and online_walk_gmem.cu).
//
// Static bias (DeepWalk, PPR): the rows that the walk is expected to draw from often get their tables, by the kernels of
// the offline build; from any other row the one entry that the draw reads is evaluated from the weights.  One
// kernel then takes every walker through its whole walk.  The draws, and so the paths, are those of the offline walk.
//
// node2vec: the weights of a step depend on the walker's previous vertex
// (src/api/bias_node2vec.cu:15-27), so each (walker, step) has a table of its own, of which one entry is evaluated.
#include <algorithm>
#include <cmath>

#include "sky_build_fused.h"
#include "sky_graph.h"
#include "sky_step_draw.h"

namespace sky {

int walk_online_node2vec(sky_graph* g, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                         float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                         double* seconds);

// ---------------------------------------------------------------- static bias
// A walker per workgroup of T threads, for the whole walk.  Rows of table_from entries and more have tables; from the
// others the draw is evaluated directly.
// A step is a chain: bounds, weights, draw, neighbour.  Most rows met are short (half of all cycles went to rows below 64 entries, 9,000 to 12,000
// a draw by the forms for long rows), so up to 64 entries have a slot a lane (draw_wave) and their neighbours loaded beside the weights,
// and up to 256 (512 where a walker is a wavefront) four (eight) slots a lane: 20,000 walkers x 4 on the scale-16 graph 79.1 -> 68.7 us, 9,000 x 10 on the scale-20 graph 124 -> 112.5,
// 10,000 x 8 on the scale-22 graph 187.9 -> 180.3, most of it the build of the long rows.
// Six wavefronts to a SIMD, 80 registers, is what 64 and 128 threads come to without spills (5,000 x 10 on the scale-18 graph by 128 threads
// 92.5 us before, 83.3 with the short rows apart, 78.7 with 80 registers for 87); 256 threads would spill and gain nothing.
template <int T>
__global__ __launch_bounds__(T, T <= 128 ? 6 : 1) void walk_direct_kernel(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
                                                        const float* __restrict__ wgt, const AliasEntry* __restrict__ table,
                                                        uint32_t table_from, const uint32_t* __restrict__ seeds, uint32_t first,
                                                        uint32_t V, uint32_t len, float stop_prob, uint64_t seed,
                                                        uint32_t* __restrict__ paths, uint32_t* __restrict__ lengths,
                                                        CallDevice* __restrict__ call, const CallDevice* __restrict__ words) {
  __shared__ DrawLds<T> lds;
  call_stamp(call);
  const uint32_t i = first + blockIdx.x;
  uint32_t* const path = paths + (size_t)i * (len + 1);
  const bool refused = words && words->refused;  // beside the start vertex
  uint32_t v = seeds[i], s = 0;
  if (refused) return;  // another plan is on its way
  if (threadIdx.x == 0) path[0] = v;
  for (; s < len && v < V; ++s) {
    const u32x4 r = philox(seed, i, s, 0, DOM_WALK);
    if (stop_prob > 0.0f && u24(r.z) < stop_prob) break;
    const uint32_t off = xadj[v], d = xadj[v + 1] - off;
    if (d == 0) break;
    uint32_t cand;
    if (d >= table_from) {
      const uint32_t col = __umulhi(r.x, d);
      const AliasEntry e = table[off + col];
      cand = u24(r.y) < e.prob ? col : e.alias;
      static_assert(NONE_SLOT == SKY_INVALID, "a row without weight ends the walk either way");
    } else if (d <= 64) {
      const uint32_t next = adjncy[off + min(threadIdx.x & 63, d - 1)];
      PlainRow row{wgt + off, d};
      cand = draw_wave<1>(row, d, r.x, u24(r.y));
      if (cand == NONE_SLOT) break;
      v = (uint32_t)__builtin_amdgcn_readlane((int)next, (int)cand);
      if (threadIdx.x == 0) path[s + 1] = v;
      continue;
    } else {
      PlainRow row{wgt + off, d};
      cand = draw_slot<T>(row, d, r, lds);
    }
    if (cand == NONE_SLOT) break;
    v = adjncy[off + cand];
    if (threadIdx.x == 0) path[s + 1] = v;
  }
  if (threadIdx.x == 0) lengths[i] = s;
}

// Threads of a walker: the walk ends with the walker that meets the longest rows without a table, so the longer these may be the more
// threads, and the more walkers the fewer, down to what fills the GPU.  (64 / 128 / 256 / 512 / 1024 threads, us.  Longest row of
// 300,000: 207 walkers x 3 233 / 137 / 86 / 69 / 69; 5,000 x 2 1137 / 604 / 328 / 226; 7,000 x 2 1410 / 774 / 413 / 303 / 307.  Of 50,000
// to 65,000: 352 x 8 269 / 158 / 102 / 84 / 89; 8,500 x 1 91 / 61 / 46 / 66; 20,000 x 2 233 / 190 / 195 / 288.  Of 25,000: 1,000 x 6
// 155 / 135 / 122 / 133 / 180; 3,000 x 10 471 / 348 / 274 / 333.  Of 5,000 to 8,000: 100 x 10 80 / 65 / 57 / 59 / 73; 1,000 x 12 135 / 119 / 119 / 142;
// 3,800 x 8 172 / 156 / 168 / 211; 7,000 x 10 237 / 221 / 252 / 371.  These are of draws before rows of up to 512 entries had draw_wave.  With it, over 36
// walks drawn from graphs of 1 M to 235 M entries, the number taken is 1.5 % slower than the best of the five in the mean and 13 % at most:
// 9,738 x 8, scale 23, 174 / 153 / 167, and 11 x 8 on the scale-22 graph with 18 edges a vertex 34 by 512 threads and 39 by 1024.)
static uint32_t walker_threads(uint32_t N, uint32_t longest) {
  if (longest > 65533) return N <= 256 ? 1024 : N <= 8192 ? 512 : 256;
  if (longest > 16384) return N <= 512 ? 512 : N <= 16384 ? 256 : 128;
  return N <= 1024 ? 256 : N <= 8192 ? 128 : 64;
}

// How to serve a static-bias walk on a graph without tables.  Every row drawn from costs either its table (BUILD_PS an entry, once, and
// BUILD_US the launches of a build) or two sweeps over its weights (DRAW_PS an entry, each time).  A start vertex is any vertex, or as
// online_plan finds; a later step leads to a row with a probability that grows with its length, so a row of d entries is drawn from N * (len - 1) * d / E
// times, and its table pays from some length on.  But a walk also lasts as long as the walker that meets the longest row without
// a table, ROW_NS an entry with 512 threads, inversely more with fewer and down to ROW_LEAST_NS with more.  What every choice would
// take is added up, from no tables over those of the longest class alone to those of every class from 33 entries on, and the least is taken.
// The figures were fitted, before rows of up to 512 entries were drawn from by draw_wave, to 36 walks on graphs of 1 M to 260 M entries with ten
// choices each: what was taken was 2 % slower than the best of the ten in the mean, 25 % at most.  With draw_wave, over 36 other walks with
// eleven choices each: 4 % in the mean, 19 % at most (343 x 13 on the scale-18 graph with 32 edges a vertex, 103 us without tables, 87 with those of
// rows from 382 entries on), so they are left as they are.  (Tables where N * len * d / E * 2.5 ps exceeds 8 ps, as before, and now, us: 5,000 walkers x 2 on the
// scale-24 graph 1301 / 169, 4,000 x 2 on the scale-22 graph with 40 edges a vertex 640 / 186, 500 x 8 with 30 288 / 192, 8,500 x 1 on the
// scale-23 graph 180 / 46, 20,000 x 12 there 415 / 375.)
constexpr double BUILD_PS = 7.5, DRAW_PS = 2.4, BUILD_US = 31.0, ROW_NS = 0.39, ROW_LEAST_NS = 0.25, STEP_US = 2.4;

struct OnlinePlan {
  bool full;            // every row, then the offline walk
  uint32_t table_from;  // else: the rows of at least so many entries
  double us;
  bool enqueued = false;  // of no tables: the walk goes out at once, and is refused if the rows of its start vertices are long
};
// starts: walkers whose first row is of each class.  `only`: null, or the plan that is to be rated.
static OnlinePlan plan_for(const sky_graph* g, uint32_t N, uint32_t len, double go, const double (&starts)[CLS_COUNT],
                           const OnlinePlan* only = nullptr) {
  OnlinePlan o{false, 0xFFFFFFFFu, 1e30, false};
  const double E = std::max(1u, g->E);
  const double edges = N * (go < 1.0 ? go * go * (1.0 - std::pow(go, len - 1.0)) / (1.0 - go) : len - 1.0);  // steps along an edge
  struct Rows {
    uint32_t from;
    double entries, read, chain;  // of all rows; of those drawn from, with repeats; of the one walker's that meets the most
  } rows[CLS_COUNT + 1];
  int n = 0;
  for (int c = CLS_G2; c < CLS_COUNT; ++c) {
    const double entries = (double)g->bin_edges[c], count = g->bin_counts[c];
    if (entries == 0 || count == 0) continue;
    const double mean = entries / count, times = edges * entries / E + starts[c];
    const double most = std::min(1.5 * mean, (double)g->max_degree);
    rows[n++] = Rows{class_min_degree(c), entries, times * mean, most * (std::min(1.0, times) + times / std::max(1u, N))};
  }
  std::sort(rows, rows + n, [](const Rows& a, const Rows& b) { return a.from < b.from; });
  const double to_max = edges * g->max_degree / E;
  double built = 0;
  for (int k = n; k >= 0; --k) {  // tables of rows[k] .. rows[n - 1]
    if (k < n) built += rows[k].entries;
    if (k < n && rows[k].from < 33) break;  // the shorter classes are not built apart from the rest
    const uint32_t from = k < n ? rows[k].from : 0xFFFFFFFFu;
    if (only && (only->full || only->table_from != from)) continue;
    double read = 0, chain = k < n ? 0.0 : g->max_degree * (std::min(1.0, to_max) + to_max / std::max(1u, N));
    for (int i = 0; i < k; ++i) {
      read += rows[i].read;
      chain = std::max(chain, rows[i].chain);
    }
    const double row_ns = std::max(ROW_LEAST_NS, ROW_NS * 512 / walker_threads(N, std::min(from - 1, g->max_degree)));
    const double us = (k < n ? BUILD_US + built * BUILD_PS * 1e-6 : 0.0) + read * DRAW_PS * 1e-6 + chain * row_ns * 1e-3 + STEP_US * len;
    if (us < o.us) {
      o.us = us;
      o.table_from = from;
    }
  }
  const double full_us = BUILD_US + E * BUILD_PS * 1e-6 + 1.2 * len;
  if (only ? only->full : option(g, OPT_ONLINE_FULL_BUILD) < 0 && full_us < o.us) {
    o.full = true;
    o.us = full_us;
  }
  return o;
}

// Classes of the rows of start vertices, all of them or 1,024 spread over them, 16 bits each; and, in the place of a class that is none,
// whether a walk without tables is refused: these rows hold more than `budget` entries, or one of them more than `longest`.
constexpr uint32_t STARTS_T = 512, STARTS_SEEN = 1024, STARTS_REFUSED = 22;
static_assert(3 * CALL_ANSWERS >= CLS_COUNT && 16 * 3 <= CALL_VALUE_BITS && class_min_degree(STARTS_REFUSED) == 0, "three classes a word");
__global__ __launch_bounds__(STARTS_T) void walk_starts_kernel(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ seeds,
                                                               uint32_t N, uint32_t V, unsigned long long budget, uint32_t longest,
                                                               CallDevice* __restrict__ words, CallHost* __restrict__ host,
                                                               unsigned long long number, CallDevice* __restrict__ call) {
  __shared__ uint32_t s_n[3 * CALL_ANSWERS];
  __shared__ unsigned long long s_entries;
  call_stamp(call);
  if (threadIdx.x < 3 * CALL_ANSWERS) s_n[threadIdx.x] = 0;
  if (threadIdx.x == 0) s_entries = 0;
  __syncthreads();
  const uint32_t seen = min(N, STARTS_SEEN);
  uint32_t v[STARTS_SEEN / STARTS_T];
#pragma unroll
  for (int u = 0; u < (int)(STARTS_SEEN / STARTS_T); ++u) {
    const uint32_t i = u * STARTS_T + threadIdx.x;
    v[u] = i < seen ? seeds[(uint64_t)i * N / seen] : V;
  }
  unsigned long long entries = 0;
#pragma unroll
  for (int u = 0; u < (int)(STARTS_SEEN / STARTS_T); ++u)
    if (v[u] < V) {
      const uint32_t d = xadj[v[u] + 1] - xadj[v[u]];
      atomicAdd(&s_n[degree_class(d)], 1u);
      entries += d > longest ? budget + 1 : d;
    }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) entries += shfl_xor_u64(entries, m);
  if ((threadIdx.x & 63) == 0) atomicAdd(&s_entries, entries);
  __syncthreads();
  const uint32_t t = threadIdx.x;
  const bool refused = s_entries > budget;
  if (t == 0) words->refused = refused;
  if (t < CALL_ANSWERS) {
    unsigned long long x = 0;
    for (uint32_t k = 0; k < 3; ++k) x |= (unsigned long long)(3 * t + k == STARTS_REFUSED ? (uint32_t)refused : s_n[3 * t + k]) << 16 * k;
    call_answer(host, number, (int)t, x);
  }
}

// The plan by what walk_starts_kernel has seen; *o as it is if it has been enqueued and is not refused.
static int plan_for_starts(sky_graph* g, uint32_t N, uint32_t len, double go, OnlinePlan* o) {
  unsigned long long counts[CALL_ANSWERS];
  SKY_TRY(call_answered(g, &g->call, counts, CALL_ANSWERS));
  auto of = [&](uint32_t c) { return (uint32_t)(counts[c / 3] >> 16 * (c % 3)) & 0xFFFFu; };
  if (o->enqueued && !of(STARTS_REFUSED)) return SKY_OK;
  double starts[CLS_COUNT];
  for (uint32_t c = 0; c < CLS_COUNT; ++c) starts[c] = c == STARTS_REFUSED ? 0.0 : N * go * of(c) / std::min(N, STARTS_SEEN);
  *o = plan_for(g, N, len, go, starts);
  return SKY_OK;
}

// Start vertices are the caller's.  Where the plan for any vertices is within ASK_US of the best for ends of edges they are not looked
// at, unless it is one without tables and they might all be the vertex with the longest row.  Else 1,024 of their rows are: for a plan without
// tables while the walk is on its way, 4 us later, unless it is refused; for another before the build, which waits 10 us for it.  (As planned
// for any vertices / as seen, us: 40,000 walkers x 1 on the scale-20 graph, any vertices 86 / 90, ends of edges 253 / 127, the longest row
// 2477 / 76; 8,500 x 1 there 32 / 37, 88 / 91, 606 / 61, on the scale-22 graph with 32 edges a vertex 33 / 37, 270 / 211, 2427 / 94;
// 5,000 x 2, scale 20, 89 / 95, 135 / 98, 454 / 83.)
constexpr double ASK_US = 15.0;
static int online_plan(sky_graph* g, const uint32_t* seeds, uint32_t N, uint32_t len, double go, OnlinePlan* o, CallDevice** first) {
  const long long mode = option(g, OPT_ONLINE_FULL_BUILD);
  *o = OnlinePlan{mode > 0, 0xFFFFFFFFu, 0.0, false};
  if (mode > 0 || option(g, OPT_ONLINE_DIRECT) > 0) return SKY_OK;
  SKY_TRY(ensure_plan(g, first));
  const double E = std::max(1u, g->E), V = std::max(1u, g->V);
  double any[CLS_COUNT], ends[CLS_COUNT], longest[CLS_COUNT] = {0.0};
  longest[degree_class(g->max_degree)] = N * go;
  for (int c = 0; c < CLS_COUNT; ++c) {
    any[c] = N * go * g->bin_counts[c] / V;
    ends[c] = N * go * g->bin_edges[c] / E;
  }
  *o = plan_for(g, N, len, go, any);
  const OnlinePlan other = plan_for(g, N, len, go, ends);
  auto loss = [&](const double (&starts)[CLS_COUNT], const OnlinePlan& best) { return plan_for(g, N, len, go, starts, o).us - best.us; };
  const bool none = !o->full && o->table_from == 0xFFFFFFFFu, other_none = !other.full && other.table_from == 0xFFFFFFFFu;
  if (o->full || (loss(ends, other) < ASK_US &&
                  !(none && !other_none && loss(longest, plan_for(g, N, len, go, longest)) > 4 * ASK_US)))
    return SKY_OK;
  // Without tables the start rows may take 10 us more than those of any vertices, and the longest 15, or as long as one that is met later.
  const double seen = std::min(N, STARTS_SEEN), row_ns = std::max(ROW_LEAST_NS, ROW_NS * 512 / walker_threads(N, g->max_degree));
  const double budget = 1.5 * seen * E / V + 10e6 / DRAW_PS * seen / N;
  const double most = std::max(15e3 / row_ns, g->max_degree * std::min(1.0, (len - 1.0) * N * g->max_degree / E));
  hipLaunchKernelGGL(walk_starts_kernel, dim3(1), dim3(STARTS_T), 0, g->stream, g->xadj, seeds, N, g->V, (unsigned long long)budget,
                     (uint32_t)std::min(most, 4294967295.0), g->call.dev, g->call.host, call_ask(&g->call), *first);
  SKY_HIP(hipGetLastError());
  *first = nullptr;
  o->enqueued = none;
  return none ? SKY_OK : plan_for_starts(g, N, len, go, o);
}

int walk_online(sky_graph* g, int bias_kind, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                double* seconds) {
  if (bias_kind == SKY_BIAS_NODE2VEC_REJECT)
    return walk_node2vec_reject(g, p, q, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds);
  if (bias_kind == SKY_BIAS_NODE2VEC)
    return walk_online_node2vec(g, p, q, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds);
  // Tables that already exist are used as they are.  Otherwise the rows that the walk will draw from often get theirs, all
  // of them when that is most of what it meets; the paths are the same either way.
  double plan_sec = 0, build_sec = 0;
  OnlinePlan how{false, 0xFFFFFFFFu, 0.0, false};
  CallDevice* call = nullptr;
  auto walk = [&] {
    const uint32_t T = walker_threads(N, std::min(how.table_from - 1, g->max_degree));
    const uint32_t most = 0xFFFFFFFFu / T;  // walkers of one launch: below 2^32 threads
    for (uint32_t f = 0; f < N; f += std::min(most, N - f)) {
      auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(std::min(most, N - f)), dim3(T), 0, g->stream, g->xadj, g->adjncy, g->adjwgt, g->table,
                           how.table_from, seeds, f, g->V, len, stop_prob, seed, paths, lengths, call, how.enqueued ? g->call.dev : nullptr);
      };
      if (T == 1024) go(walk_direct_kernel<1024>);
      else if (T == 512) go(walk_direct_kernel<512>);
      else if (T == 256) go(walk_direct_kernel<256>);
      else if (T == 128) go(walk_direct_kernel<128>);
      else go(walk_direct_kernel<64>);
      call = nullptr;
    }
  };
  if (!g->has_tables) {
    SKY_TRY(call_begin(g, &call));
    const double go = 1.0 - std::min(1.0f, std::max(0.0f, stop_prob));
    if (N && len) SKY_TRY(online_plan(g, seeds, N, len, go, &how, &call));
    if (how.enqueued) {
      walk();
      SKY_TRY(plan_for_starts(g, N, len, go, &how));
      if (how.enqueued) return call_end(g, sampled, seconds, lengths, N);
    }
    if (how.full) {  // the build is a call of its own, and so is the plan if it was made just now
      if (call) call_cancel(g);
      else SKY_TRY(call_end(g, nullptr, &plan_sec));
      SKY_TRY(build_all_tables(g, &build_sec));
    }
  }
  if (g->has_tables) {
    SKY_TRY(walk_offline(g, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds));
    if (seconds) *seconds += plan_sec + build_sec;
    return SKY_OK;
  }
  if (how.table_from != 0xFFFFFFFFu) {
    SKY_TRY(build_rows_from(g, how.table_from, call));
    call = nullptr;  // the build's first kernel is the call's, or the plan's was
  }
  walk();
  return call_end(g, sampled, seconds, lengths, N);
}

// ---------------------------------------------------------------- node2vec
// One walker per workgroup of T threads, for the whole walk; every step evaluates the one entry of its second-order
// table that the draw reads (draw_slot).  The weights of a step need, for every neighbour of the current vertex,
// whether it is a neighbour of the previous one too.  Both rows are sorted, so each wavefront moves through its part of
// the current row and, beside it, through the previous row a window of WIN ids at a time that it keeps in LDS: the ids of
// 256 slots are searched there together.  (A binary search per neighbour in the row in memory, 15 to 17 dependent loads,
// in every pass, and a launch per step that waited for its slowest walker: 480 us a step for 2,000 walkers on the scale-18
// graph, 1.1 M entries.)  What the search found stays in LDS, two bits per slot, for the passes that follow.
constexpr uint32_t N2V_CODES = 65536;    // slots of a row whose result is kept
constexpr uint32_t N2V_WEIGHTS = N2V_CODES / 16;  // slots of a row whose weights are, in the same LDS
constexpr uint32_t N2V_SPARSE = 32;      // previous row longer than the current one by this factor: searched in memory

// number of ids of row[lo .. n) that lie below key, plus lo; a wavefront probes 64 places at a time
__device__ __forceinline__ uint32_t wave_lower_bound(const uint32_t* __restrict__ row, uint32_t lo, uint32_t n, uint32_t key) {
  const uint32_t lane = threadIdx.x & 63;
  uint32_t len = n - lo;
  while (len > 64u) {
    const uint32_t step = len / 65u + 1u, end = lo + len, p = lo + (lane + 1) * step - 1;
    const uint32_t c = (uint32_t)__popcll(__ballot(p < end && row[p] < key));
    lo += c * step;
    len = min(step, end - lo);
  }
  return lo + (uint32_t)__popcll(__ballot(lane < len && row[lo + lane] < key));
}

// WIN: ids of the previous row in LDS, per wavefront
template <uint32_t WIN>
struct N2vRow {
  static constexpr int U = 1;
  static constexpr WaveRows WAVE = WAVE_NONE;
  static constexpr int HELD = 16;
  const float* w;
  const uint32_t* nbr;
  const uint32_t* prow;
  uint32_t d, pdeg, prev;
  bool has_prev;
  bool times;  // p and q are reciprocals, which are exact: products instead of quotients
  float p, q;
  uint32_t* win;   // [WIN], this wavefront's own
  uint8_t* codes;  // [N2V_CODES / 4]: per slot 0 neighbour of both, 1 the previous vertex, 2 neither.  Or the weights of a row
                   // of up to N2V_WEIGHTS slots: what follows the first pass then waits for no memory
  uint32_t wpos, wlen;  // window: ids wpos .. wpos + wlen of the previous row

  // weight of the edge in slot k after the second-order factor (src/api/bias_node2vec.cu:15-27)
  __device__ __forceinline__ float weigh(float x, uint32_t code) const {
    const float by = code == 1u ? p : code == 2u ? q : 1.0f;
    return clamp_weight(times ? x * by : __fdiv_rn(x, by));
  }
  __device__ __forceinline__ void load_window(uint32_t from) {
    const uint32_t lane = threadIdx.x & 63;
    wpos = from;
    wlen = min(WIN, pdeg - from);
    uint4u x[WIN / 256];
#pragma unroll
    for (int j = 0; j < (int)(WIN / 256); ++j) {
      const uint32_t k = 256u * j + 4u * lane;
      x[j] = uint4u{0, 0, 0, 0};
      if (k < wlen) x[j] = *reinterpret_cast<const uint4u*>(prow + from + k);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // searches of the window before are done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < (int)(WIN / 256); ++j) {
      const uint32_t k = 256u * j + 4u * lane;
      win[k] = k < wlen ? x[j].x : 0xFFFFFFFFu;  // no vertex has this id
      win[k + 1] = k + 1 < wlen ? x[j].y : 0xFFFFFFFFu;
      win[k + 2] = k + 2 < wlen ? x[j].z : 0xFFFFFFFFu;
      win[k + 3] = k + 3 < wlen ? x[j].w : 0xFFFFFFFFu;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // codes of the four slots k .. (two bits each); all lanes of the wavefront together, 4 slots per lane in slot order
  __device__ __forceinline__ uint32_t find(uint32_t k, const uint32_t (&t)[4]) {
    uint32_t code = 0;
    if (pdeg > N2V_SPARSE * d) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j < d) code |= (t[j] == prev ? 1u : row_contains(prow, pdeg, t[j]) ? 0u : 2u) << (2 * j);
      return code;
    }
    // ids of the wavefront's first and last slot (lane 0 is always inside the row)
    const uint32_t lane = threadIdx.x & 63, kw = (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)t[0]);
    const uint32_t last_slot = min(255u, d - 1 - kw), lj = last_slot & 3u;
    const uint32_t mine = lj == 0 ? t[0] : lj == 1 ? t[1] : lj == 2 ? t[2] : t[3];
    const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)(last_slot >> 2));
    (void)lane;
    bool hit[4] = {false, false, false, false};
    if (wlen == 0 || win[wlen - 1] < first) {  // the window lies wholly below these slots
      const uint32_t from = wpos + wlen;
      if (from < pdeg) {
        // a short way is one more window; a long one is searched
        const uint32_t at = prow[min(from + WIN, pdeg) - 1] >= first ? from : wave_lower_bound(prow, from, pdeg, first);
        if (at < pdeg) load_window(at);
        else { wpos = pdeg; wlen = 0; }
      }
    }
    while (wlen) {
      uint32_t steps = 1u;
      while (steps < wlen) steps *= 2;  // wlen <= steps <= WIN; the places past wlen hold the largest id
      uint32_t at[4] = {0, 0, 0, 0};
      for (uint32_t h = steps / 2; h; h /= 2) {
        uint32_t x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = win[at[j] + h - 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) at[j] += x[j] < t[j] ? h : 0u;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) hit[j] = hit[j] || win[at[j]] == t[j];
      if (win[wlen - 1] >= last || wpos + wlen >= pdeg) break;
      load_window(wpos + wlen);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (k + j < d) code |= (t[j] == prev ? 1u : hit[j] ? 0u : 2u) << (2 * j);
    return code;
  }
  __device__ __forceinline__ void first(uint32_t k, float (&x)[4]) {
    uint32_t t[4] = {0, 0, 0, 0};
    x[0] = x[1] = x[2] = x[3] = 0.0f;
    if (k < d) {
      const float4u a = *reinterpret_cast<const float4u*>(w + k);
      x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
      if (has_prev) {
        const uint4u b = *reinterpret_cast<const uint4u*>(nbr + k);
        t[0] = b.x; t[1] = b.y; t[2] = b.z; t[3] = b.w;
      }
    }
    uint32_t code = 0;
    if (has_prev) {
      code = find(k, t);
      if (d > N2V_WEIGHTS && d <= N2V_CODES && k < d) codes[k >> 2] = (uint8_t)code;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = k + j < d ? weigh(x[j], (code >> (2 * j)) & 3u) : 0.0f;
    if (d <= N2V_WEIGHTS && k < d) reinterpret_cast<float4*>(codes)[k >> 2] = make_float4(x[0], x[1], x[2], x[3]);
  }
  __device__ __forceinline__ void again(uint32_t k, float (&x)[4]) const {
    x[0] = x[1] = x[2] = x[3] = 0.0f;
    if (k >= d) return;
    if (d <= N2V_WEIGHTS) {
      const float4 c = reinterpret_cast<const float4*>(codes)[k >> 2];
      x[0] = c.x; x[1] = c.y; x[2] = c.z; x[3] = c.w;
      return;
    }
    const float4u a = *reinterpret_cast<const float4u*>(w + k);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    uint32_t code = 0;
    if (has_prev) {
      if (d <= N2V_CODES) {
        code = codes[k >> 2];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (k + j < d) code |= (nbr[k + j] == prev ? 1u : row_contains(prow, pdeg, nbr[k + j]) ? 0u : 2u) << (2 * j);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = k + j < d ? weigh(x[j], (code >> (2 * j)) & 3u) : 0.0f;
  }
};

template <int T, uint32_t WIN>
__global__ __launch_bounds__(T, WIN == 512 ? 5 : 4) void walk_n2v_table_kernel(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
                                                           const float* __restrict__ wgt, const uint32_t* __restrict__ seeds,
                                                           uint32_t first, uint32_t V, uint32_t len, float p, float q,
                                                           float stop_prob, uint64_t seed, bool times, uint32_t* __restrict__ paths,
                                                           uint32_t* __restrict__ lengths, CallDevice* __restrict__ call) {
  __shared__ DrawLds<T> lds;
  __shared__ uint32_t s_win[T / 64][WIN];
  __shared__ __align__(16) uint8_t s_codes[N2V_CODES / 4];
  call_stamp(call);
  const uint32_t i = first + blockIdx.x;
  uint32_t* const path = paths + (size_t)i * (len + 1);
  uint32_t v = seeds[i], s = 0, prev = 0, prev_off = 0, prev_deg = 0;
  if (threadIdx.x == 0) path[0] = v;
  for (; s < len && v < V; ++s) {
    const u32x4 r = philox(seed, i, s, 0, DOM_WALK);
    if (stop_prob > 0.0f && u24(r.z) < stop_prob) break;
    const uint32_t off = xadj[v], d = xadj[v + 1] - off;
    if (d == 0) break;
    N2vRow<WIN> row;
    row.w = wgt + off;
    row.nbr = adjncy + off;
    row.prow = adjncy + prev_off;
    row.d = d;
    row.pdeg = prev_deg;
    row.prev = prev;
    row.has_prev = s > 0;
    row.times = times;
    row.p = p;
    row.q = q;
    row.win = s_win[threadIdx.x >> 6];
    row.codes = s_codes;
    row.wpos = row.wlen = 0;
    const uint32_t cand = draw_slot<T>(row, d, r, lds);
    if (cand == NONE_SLOT) break;
    prev = v;
    prev_off = off;
    prev_deg = d;
    v = row.nbr[cand];
    if (threadIdx.x == 0) path[s + 1] = v;
  }
  if (threadIdx.x == 0) lengths[i] = s;
}

// The same walk on a graph of few enough vertices that a bit for each fits beside the walkers of a CU in LDS: the bits of the
// previous row's vertices are set once a step, and a slot then tests one bit, where the search of the window is ten dependent
// reads; with no state from slot to slot the loads of U times 256 slots are in flight at once.
// Four walkers of four wavefronts to a CU, or two of eight while these hold all of them that walk (700 walkers x 20 on the scale-17 graph
// 242 us with four wavefronts, 201 with eight; 2,000 x 40 there 452 and 667): twice as many bits leave two walkers to a CU.  The line
// is where four go, not where the bits stop to pay: with two of eight wavefronts to a CU the scale-19 graph would take 371 us for 490 with
// 200 walkers x 40, 409 for 739 with 768, 767 for 863 with 2,000.
// Against the windows: 2,000 x 40 with p = 2, q = 1/2 on the scale-18 graph 736 -> 550 us, on the scale-17 graph 617 -> 456, 1,500 x 30
// with 40 edges a vertex, scale 13, 482 -> 320, 200 x 40 with 30, scale 16, 526 -> 358.
constexpr uint32_t MAP_VERTICES = 1u << 18;  // 32 KB
constexpr uint32_t MAP_ROW = 32768;          // longer previous rows of N2V_SPARSE times the current one are searched in memory
constexpr uint32_t MAP_KEEP = 4096;          // slots of a row whose weights are kept, or what room there is
constexpr uint32_t MAP_FEW = 768;
struct N2vMapRow {
  static constexpr int U = 2;
  static constexpr WaveRows WAVE = WAVE_ONE;
  static constexpr int HELD = 16;
  const float* w;
  const uint32_t* nbr;
  const uint32_t* prow;
  const uint32_t* map;  // bit t: vertex t is a neighbour of prev
  float* kept;          // weights of the row's slots, if it has at most `keep`
  uint32_t d, pdeg, prev, keep;
  bool has_prev, search;
  bool times;  // p and q are reciprocals, which are exact: products instead of quotients
  float p, q;

  // weight of the edge to t after the second-order factor (src/api/bias_node2vec.cu:15-27)
  __device__ __forceinline__ float weigh(float x, uint32_t t, bool in) const {
    if (has_prev) {
      const bool both = search ? in && row_contains(prow, pdeg, t) : (map[t >> 5] >> (t & 31)) & 1u;
      const float by = t == prev ? p : both ? 1.0f : q;
      x = times ? x * by : __fdiv_rn(x, by);
    }
    return masked_weight(x, in);
  }
  __device__ __forceinline__ void many(uint32_t k, uint32_t end, bool again, float (&x)[U][4]) const {
    if (again && d <= keep) {
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint32_t at = min(k + 256u * j, (d - 1) & ~3u);
        const float4 c = reinterpret_cast<const float4*>(kept)[at >> 2];
        const float y[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) x[j][t] = k + 256u * j + t < end ? y[t] : 0.0f;
      }
      return;
    }
    float4u a[U];
    uint4u b[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t at = min(k + 256u * j, (d - 1) & ~3u);
      a[j] = *reinterpret_cast<const float4u*>(w + at);
      b[j] = *reinterpret_cast<const uint4u*>(nbr + at);
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t at = k + 256u * j;
      x[j][0] = x[j][1] = x[j][2] = x[j][3] = 0.0f;
      if (at - 4 * (threadIdx.x & 63) >= end) continue;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bool in = at + t < end;
        x[j][t] = weigh(a[j][t], in ? b[j][t] : 0u, in);  // past the row's end lies another's vertex, or none
      }
      if (!again && d <= keep && at < end) reinterpret_cast<float4*>(kept)[at >> 2] = make_float4(x[j][0], x[j][1], x[j][2], x[j][3]);
    }
  }
  __device__ __forceinline__ void load(uint32_t k, float (&x)[1]) const {
    const uint32_t at = min(k, d - 1);
    x[0] = weigh(w[at], nbr[at], k < d);
  }
  __device__ __forceinline__ void load(uint32_t k, float (&x)[4]) const {
    const uint32_t at = min(k, (d - 1) & ~3u);
    const float4u a = *reinterpret_cast<const float4u*>(w + at);
    const uint4u b = *reinterpret_cast<const uint4u*>(nbr + at);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = weigh(a[t], k + t < d ? b[t] : 0u, k + t < d);
  }
  __device__ __forceinline__ void again(uint32_t k, float (&x)[4]) const {
    x[0] = x[1] = x[2] = x[3] = 0.0f;
    if (k >= d) return;
    if (d <= keep) {
      const float4 c = reinterpret_cast<const float4*>(kept)[k >> 2];
      x[0] = c.x; x[1] = c.y; x[2] = c.z; x[3] = c.w;
      return;
    }
    const float4u a = *reinterpret_cast<const float4u*>(w + k);
    const uint4u b = *reinterpret_cast<const uint4u*>(nbr + k);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = weigh(a[t], k + t < d ? b[t] : 0u, k + t < d);
  }
};

template <int T>
__global__ __launch_bounds__(T) void walk_n2v_map_kernel(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
                                                         const float* __restrict__ wgt, const uint32_t* __restrict__ seeds,
                                                         uint32_t first, uint32_t V, uint32_t len, float p, float q,
                                                         float stop_prob, uint64_t seed, bool times, uint32_t map_words, uint32_t keep,
                                                         uint32_t* __restrict__ paths, uint32_t* __restrict__ lengths,
                                                         CallDevice* __restrict__ call) {
  __shared__ DrawLds<T> lds;
  extern __shared__ __align__(16) uint32_t s_map[];  // [map_words], a multiple of 4, then the kept weights
  call_stamp(call);
  const uint32_t i = first + blockIdx.x;
  uint32_t* const path = paths + (size_t)i * (len + 1);
  uint32_t v = seeds[i], s = 0, prev = 0, prev_off = 0, prev_deg = 0;
  if (threadIdx.x == 0) path[0] = v;
  for (; s < len && v < V; ++s) {
    const u32x4 r = philox(seed, i, s, 0, DOM_WALK);
    if (stop_prob > 0.0f && u24(r.z) < stop_prob) break;
    const uint32_t off = xadj[v], end = xadj[v + 1];
    auto mark = [&] {  // the previous row, while the bounds of this one are on their way
      constexpr int M = 2;
      const uint32_t* const prow = adjncy + prev_off;
      for (uint64_t from = 0; from < prev_deg; from += 4 * T * M) {
        const uint32_t k = (uint32_t)from + 4 * threadIdx.x;
        uint4u x[M];
#pragma unroll
        for (int j = 0; j < M; ++j) x[j] = *reinterpret_cast<const uint4u*>(prow + min(k + 4 * T * j, (prev_deg - 1) & ~3u));
        if (from == 0) {
          __syncthreads();  // the draw before may still be reading bits
          for (uint32_t c = threadIdx.x; c < map_words / 4; c += T) reinterpret_cast<uint4*>(s_map)[c] = make_uint4(0, 0, 0, 0);
          __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < M; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (k + 4 * T * j + t < prev_deg) atomicOr(&s_map[x[j][t] >> 5], 1u << (x[j][t] & 31));
      }
    };  // the draw starts with a barrier
    if (s > 0 && prev_deg <= MAP_ROW) mark();
    const uint32_t d = end - off;
    if (d == 0) break;
    const bool search = prev_deg > MAP_ROW && prev_deg / N2V_SPARSE > d;
    if (prev_deg > MAP_ROW && !search) mark();
    N2vMapRow row;
    row.w = wgt + off;
    row.nbr = adjncy + off;
    row.prow = adjncy + prev_off;
    row.map = s_map;
    row.kept = reinterpret_cast<float*>(s_map + map_words);
    row.d = d;
    row.pdeg = prev_deg;
    row.prev = prev;
    row.keep = keep;
    row.has_prev = s > 0;
    row.search = search;
    row.times = times;
    row.p = p;
    row.q = q;
    const uint32_t cand = draw_slot<T>(row, d, r, lds);
    if (cand == NONE_SLOT) break;
    prev = v;
    prev_off = off;
    prev_deg = d;
    v = row.nbr[cand];
    if (threadIdx.x == 0) path[s + 1] = v;
  }
  if (threadIdx.x == 0) lengths[i] = s;
}

int walk_online_node2vec(sky_graph* g, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                         float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                         double* seconds) {
  hipStream_t st = g->stream;
  CallDevice* call = nullptr;
  SKY_TRY(call_begin(g, &call));
  // Four wavefronts per walker, eight while that leaves CUs without one.  A window of 1024 ids per wavefront makes 37 KB
  // of LDS, four walkers to a CU; more walkers than that get windows of 512, 29 KB, five to a CU, so that fewer of them
  // wait for a CU (2,000 walkers x 40 steps on the scale-18 graph 901 -> 761 us; 900 walkers on the scale-17 graph 538
  // with 1024 ids, 555 with 512).  Less LDS still, by fewer slots whose result is kept or smaller windows, was slower.
  constexpr uint32_t FEW = 512, RESIDENT = 1024;
  // A power of two divides as its reciprocal multiplies, to the last bit: 12 instructions an entry fewer.
  auto power = [](float x) {
    int e;
    return std::frexp(x, &e) == 0.5f && std::abs(e) < 100;
  };
  const bool times = power(p) && power(q);
  const float by_p = times ? 1.0f / p : p, by_q = times ? 1.0f / q : q;
  const uint32_t most = 0xFFFFFFFFu / 512;  // walkers of one launch: below 2^32 threads
  for (uint32_t f = 0; f < N; f += std::min(most, N - f)) {
    const dim3 grid(std::min(most, N - f));
    auto go = [&](auto kernel, uint32_t threads) {
      hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, st, g->xadj, g->adjncy, g->adjwgt, seeds, f, g->V, len, by_p, by_q, stop_prob,
                         seed, times, paths, lengths, call);
    };
    if (g->V <= MAP_VERTICES) {
      const uint32_t words = (g->V + 127u) / 128u * 4u;
      auto map = [&](auto kernel, uint32_t threads, uint32_t walkers, size_t fixed) {  // walkers of a CU
        const uint32_t keep = std::min(MAP_KEEP, ((160u << 10) / walkers - (uint32_t)fixed - 4u * words) / 16u * 4u);
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 4u * (words + keep), st, g->xadj, g->adjncy, g->adjwgt, seeds, f, g->V, len,
                           by_p, by_q, stop_prob, seed, times, words, keep, paths, lengths, call);
      };
      if (N <= MAP_FEW) map(walk_n2v_map_kernel<512>, 512, 2, sizeof(DrawLds<512>));
      else map(walk_n2v_map_kernel<256>, 256, 4, sizeof(DrawLds<256>));
    } else if (N <= FEW) go(walk_n2v_table_kernel<512, 1024>, 512);
    else if (N <= RESIDENT) go(walk_n2v_table_kernel<256, 1024>, 256);
    else go(walk_n2v_table_kernel<256, 512>, 256);
    call = nullptr;
  }
  return call_end(g, sampled, seconds, lengths, N);
}

}  // namespace sky
