// Builds in few launches (sky_build_fused.hip): what a graph keeps for them, and the rows of a frontier.
#pragma once
#include "sky_graph.h"

namespace sky {

struct TiledRow;
struct TileGeom;
struct TileTotals;

// What follows from the row offsets alone and is therefore made once per graph: the rows of more than 32 entries by
// class, and the geometry of the rows that are built tile by tile, with the scratch of their passes.
struct BuildPlan {
  RowRef* rows = nullptr;  // classes CLS_G16 .. back to back
  uint32_t start[CLS_COUNT] = {0};
  uint64_t listed = 0;
  long long narrow_limit = 0;  // option stream_min_edges the plan was made under
  int t_first = 0;             // classes t_first .. CLS_HUGE have geometry to be built tile by tile ...
  int t_all = 0;               // ... and t_all .. CLS_HUGE are, by every build
  uint32_t wide_row = 0, wide_tile = 0;  // first row and tile of the latter, when the two differ
  uint32_t n_trows = 0, n_tiles = 0;  // n_tiles: an upper bound, tiles that do not exist have span 0
  TiledRow* trows = nullptr;
  void* tiles = nullptr;  // the allocation of the arrays below
  TileGeom* geom = nullptr;
  u128* tsum = nullptr;
  TileTotals* ttot = nullptr;
  uint64_t *BL = nullptr, *BH = nullptr;
  uint32_t* nfh = nullptr;
  uint4* ranges = nullptr;
  BuildPlan() = default;
  BuildPlan(const BuildPlan&) = delete;
  ~BuildPlan();
};

// Segments of a frontier's rows: class c from start[c] on, as many as the device word counts[c] says.  The classes
// tiled_from .. CLS_HUGE have none: their rows are known to the plan, and the frontier's bitmap says which to build.
struct FrontierLists {
  RowRef* list = nullptr;
  uint32_t start[CLS_COUNT] = {0}, cap[CLS_COUNT] = {0};
  int tiled_from = 0;
  bool few = false;  // at most SMALL_FRONTIER rows
};
// A frontier's bitmap: the bit of vertex v.  A word serves its atomics one after another, and a graph's busiest vertices tend to
// have neighbouring ids (R-MAT: one draw in a hundred lands on 32 of 4 M); an odd factor, modulo the number of bits, a power of
// two, puts them into words of their own.  Collecting the 1 M draws of a 40,000-seed batch 88 -> 27 us.
__device__ __forceinline__ uint32_t frontier_bit(uint32_t v, uint32_t mask) { return (v * 2654435769u) & mask; }
inline uint32_t frontier_mask(uint32_t V) {
  uint32_t m = 31;
  while (V && m < V - 1) m = 2 * m + 1;
  return m;
}
constexpr uint32_t FRONTIER_WORDS = 32;  // device words of counts per frontier
static_assert(FRONTIER_WORDS > CLS_COUNT, "one word per class, and one for the launch of the longest rows");

bool fused_possible(const sky_graph* g);
// The graph's plan, made if there is none or a knob has changed.  *first as in bin_all_rows: making the plan is part of the
// call that needs it, and of its time.
int ensure_plan(sky_graph* g, CallDevice** first);
// All rows; needs the plan and vertices, and the end of the call behind it.
int build_all_fused(sky_graph* g, CallDevice* call);
// The rows of at least min_degree entries alone (a class boundary of 33 or more); needs the plan.  `call` is stamped (null: another kernel was).
int build_rows_from(sky_graph* g, uint32_t min_degree, CallDevice* call);
// Segments for a frontier of at most n_upper rows, in `buf`, which grows when it has to.  `p` is a plan of the graph, the same
// for all frontiers of a call.
int frontier_lists(sky_graph* g, const BuildPlan& p, uint32_t n_upper, sky_graph::PoolBuf* buf, FrontierLists* f);
// Builds the rows in the segments (counts: their lengths, on the device, and behind them a word that is 0 the first time; `again`: not
// the first time with these counts) and those of the tiled classes whose bit is set, unless another hop has: `built`, a word for each row of the
// plan that has geometry, the call's own, 0 at first, then holds the hop's number + 1.  Nothing waits for the device.
int build_frontier(sky_graph* g, const BuildPlan& p, const FrontierLists& f, uint32_t* counts, bool again, const uint32_t* bitmap,
                   uint32_t* built, uint32_t hop);

// Appends the vertices of the calling workgroup's lanes whose `fresh` is set to their classes' segments: one global atomic
// per class that occurs.  All threads of the workgroup call it; s_cnt and s_base hold CLS_COUNT words of LDS each.
__device__ __forceinline__ void append_rows(bool fresh, uint32_t v, const uint32_t* __restrict__ xadj,
                                            int8_t* __restrict__ valid, const FrontierLists& f, uint32_t* __restrict__ counts,
                                            uint32_t* s_cnt, uint32_t* s_base) {
  if (threadIdx.x < CLS_COUNT) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  uint32_t off = 0, d = 0, rank = 0;
  int c = CLS_EMPTY;
  if (fresh) {
    off = xadj[v];
    d = xadj[v + 1] - off;
    c = degree_class(d);
    if (c == CLS_EMPTY) valid[v] = 0;
    if (c >= f.tiled_from && c <= CLS_HUGE) c = CLS_EMPTY;
    if (c != CLS_EMPTY) rank = atomicAdd(&s_cnt[c], 1u);
  }
  __syncthreads();
  if (threadIdx.x < CLS_COUNT && s_cnt[threadIdx.x]) s_base[threadIdx.x] = atomicAdd(&counts[threadIdx.x], s_cnt[threadIdx.x]);
  __syncthreads();
  if (c != CLS_EMPTY) f.list[f.start[c] + s_base[c] + rank] = RowRef{v, off, d, 0};
}

// Appends the vertices of the calling workgroup's lanes whose `fresh` is set to a plain list: one global atomic.
// s_n holds one word of LDS per wavefront and one more.
__device__ __forceinline__ void append_list(bool fresh, uint32_t v, uint32_t* __restrict__ list, uint32_t* __restrict__ count,
                                            uint32_t* s_n) {
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const unsigned long long m = __ballot(fresh);
  if (lane == 0) s_n[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t n = 0;
    for (uint32_t w = 0; w < waves; ++w) n += s_n[w];
    s_n[waves] = n ? atomicAdd(count, n) : 0u;
  }
  __syncthreads();
  if (fresh) {
    uint32_t base = s_n[waves];
    for (uint32_t w = 0; w < wave; ++w) base += s_n[w];
    list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = v;
  }
}

}  // namespace sky
