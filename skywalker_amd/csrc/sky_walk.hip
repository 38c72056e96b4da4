// Biased walk on prebuilt alias tables (replaces sample_kernel_static / _buffer / sample_kernel and
// OfflineWalk of the reference, src/offline_walk.cu:10-230), with the PPR stop test the reference
// only has in its online kernel (src/online_walk.cu:109-110).
//
// One walker per lane.  Step s of walker i draws r = Philox(seed; i, s, 0, DOM_WALK):
//   stop when stop_prob > 0 and u24(r.z) < stop_prob, or the vertex has no out-edge,
//   col = mulhi(r.x, deg); cand = u24(r.y) < prob[off+col] ? col : alias[off+col];
//   stop when cand == SKY_INVALID (row of zero total weight); next = adjncy[off + cand].
// The result depends on (seed, i, s) only, never on scheduling.
#include "sky_graph.h"

namespace sky {

constexpr int WALK_BLOCK = 256;
constexpr int WALK_STAGE = 4;  // steps whose vertices leave together as one 16-byte store

typedef uint32_t path4u __attribute__((ext_vector_type(4), aligned(4)));

// What a step reads first: the bounds of the row of v, eight bytes that need not be aligned to eight.
typedef uint32_t bounds2u __attribute__((ext_vector_type(2), aligned(4)));

// One draw from the row [off, off + deg) of deg > 0 entries.  With the walk index one 16-byte entry holds both possible
// next vertices (two cache lines per step: xadj and the entry); without it the neighbour id is a third gather.
template <bool INDEXED, bool ONCE>
__device__ __forceinline__ bool walk_draw(const uint32_t* __restrict__ adjncy, const AliasEntry* __restrict__ table,
                                          const WalkEntry* __restrict__ index, const u32x4& r, uint32_t off, uint32_t deg,
                                          uint32_t& next) {
  const uint32_t col = __umulhi(r.x, deg);
  if (INDEXED) {
    // like the table entry below: read once, so it should not push the row offsets out of L2
    typedef uint32_t idx4 __attribute__((ext_vector_type(4)));
    const idx4* ep = reinterpret_cast<const idx4*>(index + off + col);
    const idx4 eb = ONCE ? __builtin_nontemporal_load(ep) : *ep;
    WalkEntry e;
    e.prob = __uint_as_float(eb.x);
    e.alias = eb.y;
    e.nbr_col = eb.z;
    e.nbr_alias = eb.w;
    const bool keep = u24(r.y) < e.prob;
    if (!keep && e.alias == SKY_INVALID) return false;
    next = keep ? e.nbr_col : e.nbr_alias;
  } else {
    // On a graph whose tables are far larger than the caches the entry and the neighbour id are read once per
    // step, the row offsets of the well-connected vertices many times by many walkers: the two gathers then go
    // past the cache's usual replacement order so that they do not evict the offsets (1 M walkers x 80 steps on the
    // scale-26 graph: 2.16 -> 1.86 ms).  On a small graph the entries are hit again and stay ordinary loads.
    const AliasEntry e = ONCE ? load_entry_once(table + off + col) : table[off + col];
    const uint32_t cand = u24(r.y) < e.prob ? col : e.alias;
    if (cand == SKY_INVALID) return false;
    next = ONCE ? __builtin_nontemporal_load(adjncy + off + cand) : adjncy[off + cand];
  }
  return true;
}

// Steps [s, s_end) of one walker that has a wavefront for itself; the arguments are the same in every lane.  Returns the step it
// has come to, s_end unless it stopped.  Everything a step depends on is in scalar registers and its gathers are scalar
// loads, the lanes hold the random numbers and the vertices of 64 steps, and the neighbour of the drawn column is requested
// beside the table entry (half of the draws keep the column: two round trips to memory instead of three).
// VEC: entry and neighbour through the vector cache instead: the scalar caches, one to two CUs, answer some 20 G misses a second
// on the whole chip, which several thousand walkers ask for.
template <bool INDEXED, bool VEC>
__device__ __forceinline__ uint32_t walk_alone(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
                                               const AliasEntry* __restrict__ table, const WalkEntry* __restrict__ index,
                                               float stop_prob, uint64_t seed, uint32_t i, uint32_t v, uint32_t s,
                                               uint32_t s_end, uint32_t* __restrict__ path) {
  auto uniform = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
  const uint32_t lane = threadIdx.x & 63;
  while (s < s_end) {
    const u32x4 r = philox(seed, i, s + lane, 0, DOM_WALK);
    const uint32_t ubits = __float_as_uint(u24(r.y));
    const unsigned long long stop = __ballot(u24(r.z) < stop_prob);
    const uint32_t n = min(64u, s_end - s);
    uint32_t mine = 0, k = 0;
    for (; k < n; ++k) {
      if ((stop >> k) & 1) break;
      const bounds2u x = *reinterpret_cast<const bounds2u*>(xadj + v);
      const uint32_t off = x.x, deg = x.y - x.x;
      if (deg == 0) break;
      const float u = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)ubits, (int)k));
      uint32_t at = off + __umulhi((uint32_t)__builtin_amdgcn_readlane((int)r.x, (int)k), deg);
      if (VEC) asm volatile("" : "+v"(at));
      if (INDEXED) {
        const WalkEntry e = index[at];
        const bool keep = u < __uint_as_float(uniform(__float_as_uint(e.prob)));
        if (!keep && uniform(e.alias) == SKY_INVALID) break;
        v = uniform(keep ? e.nbr_col : e.nbr_alias);
      } else {
        const AliasEntry e = table[at];
        uint32_t straight = adjncy[at];
        if (VEC) asm volatile("" : "+v"(straight));  // here, not where it turns out to be needed
        else asm volatile("" : "+s"(straight));
        if (u < __uint_as_float(uniform(__float_as_uint(e.prob)))) {
          v = uniform(straight);
        } else {
          const uint32_t alias = uniform(e.alias);
          if (alias == SKY_INVALID) break;
          v = uniform(adjncy[off + alias]);
        }
      }
      if (lane == k) mine = v;
    }
    if (lane < k) path[s + 1 + lane] = mine;
    s += k;
    if (k < n) break;
  }
  return s;
}

// Few walkers, a wavefront each.  What bounds a walk of a few thousand walkers is the latency of its steps, and a wavefront of
// 64 walkers waits in every one of them for the slowest of 64 gathers.  4,096 walkers x 80 steps on the scale-16 graph 94.8 ->
// 55.8 us, 100 walkers 49.4 -> 34.8, 2,048 on the scale-24 graph 96 -> 49.
template <bool INDEXED, bool VEC>
__global__ __launch_bounds__(64) void walk_alone_kernel(const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
                                                        const AliasEntry* __restrict__ table,
                                                        const WalkEntry* __restrict__ index,
                                                        const uint32_t* __restrict__ seeds, uint32_t V, uint32_t len,
                                                        float stop_prob, uint64_t seed, uint32_t* __restrict__ paths,
                                                        uint32_t* __restrict__ lengths, CallDevice* __restrict__ call) {
  call_stamp(call);
  const uint32_t i = blockIdx.x;
  uint32_t* const path = paths + (size_t)i * (len + 1);
  const uint32_t v = seeds[i];
  if (threadIdx.x == 0) path[0] = v;
  uint32_t s = 0;
  if (v < V) s = walk_alone<INDEXED, VEC>(xadj, adjncy, table, index, stop_prob, seed, i, v, 0, len, path);
  if (threadIdx.x == 0) lengths[i] = s;
}

// Steps [s_begin, s_end) of the walkers listed in `live` (null: walkers 0..n_live-1, which then also record
// their start vertex).  A walker that is still walking at s_end is appended to `next_live` when that list is
// given: the next launch then runs on full wavefronts again (walkers that reached a vertex without out-edges
// or stopped no longer hold a lane).  The vertices of WALK_STAGE steps leave as one store.
template <bool INDEXED, bool ONCE>
__global__ __launch_bounds__(WALK_BLOCK) void walk_offline_kernel(
    const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy, const AliasEntry* __restrict__ table,
    const WalkEntry* __restrict__ index, const uint32_t* __restrict__ seeds, const uint32_t* __restrict__ live,
    const uint32_t* __restrict__ n_live_dev, uint32_t n_live, uint32_t V, uint32_t len, uint32_t s_begin,
    uint32_t s_end, float stop_prob, uint64_t seed, uint32_t* __restrict__ paths, uint32_t* __restrict__ lengths,
    uint32_t* __restrict__ next_live, uint32_t* __restrict__ n_next, CallDevice* __restrict__ call, uint32_t parts,
    unsigned long long* __restrict__ block_partials, uint32_t per) {
  if (s_begin == 0) call_stamp(call);
  __shared__ unsigned long long s_part[WALK_BLOCK / 64];
  const uint32_t wave = blockIdx.x * (WALK_BLOCK / 64) + (threadIdx.x >> 6);
  const uint32_t t = (threadIdx.x & 63) < per ? wave * per + (threadIdx.x & 63) : 0xFFFFFFFFu;
  if (n_live_dev) n_live = min(n_live, *n_live_dev);  // the list's length is only known on the device
  uint32_t steps = 0;
  bool walking = false;
  bool alone = false;  // the last of the wavefront that still walks
  uint32_t i = 0, v = 0, s = s_begin;
  auto finish = [&] {
    steps = s - s_begin;
    if (!walking || s_end == len) lengths[i] = s;
    walking = walking && s_end < len;
  };
  if (t < n_live) {
    i = live ? live[t] : t;
    uint32_t* path = paths + (size_t)i * (len + 1);
    if (s_begin == 0) {
      v = seeds[i];
      path[0] = v;
    } else {
      v = path[s_begin];
    }
    walking = v < V;  // a start vertex that does not exist is recorded and never left
    // The random numbers of a step do not depend on where the walker stands: those of the next step are computed
    // while the row bounds of this one are on their way (ten rounds, a tenth of a step's time: 250,000 PPR walkers with the
    // index 91 -> 74 us).  Requesting the neighbour of col beside the table entry gains nothing here: of 64 walkers some
    // take the alias in every step.
    u32x4 r = philox(seed, i, s, 0, DOM_WALK);
    while (walking && s < s_end) {
      if (!ONCE) {
        alone = __popcll(__ballot(true)) == 1;
        if (alone) break;
      }
      uint32_t b[WALK_STAGE];
      uint32_t got = 0;
#pragma unroll
      for (int k = 0; k < WALK_STAGE; ++k) {
        b[k] = 0;
        if (walking && s + got < s_end) {
          if (stop_prob > 0.0f && u24(r.z) < stop_prob) {
            walking = false;
          } else {
            const bounds2u x = *reinterpret_cast<const bounds2u*>(xadj + v);
            u32x4 rn = philox(seed, i, s + got + 1, 0, DOM_WALK);
            asm volatile("" : "+v"(rn.x), "+v"(rn.y), "+v"(rn.z));  // here, not where it is used
            uint32_t nx = 0;
            if (x.y == x.x || !walk_draw<INDEXED, ONCE>(adjncy, table, index, r, x.x, x.y - x.x, nx)) {
              walking = false;
            } else {
              v = nx;
              b[k] = nx;
              got = k + 1;
            }
            r = rn;
          }
        }
      }
      uint32_t* dst = path + s + 1;
      if (got == WALK_STAGE) {
        path4u o;
        o.x = b[0]; o.y = b[1]; o.z = b[2]; o.w = b[3];
        *reinterpret_cast<path4u*>(dst) = o;
      } else {
#pragma unroll
        for (int k = 0; k < WALK_STAGE - 1; ++k)
          if ((uint32_t)k < got) dst[k] = b[k];
      }
      s += got;
    }
    if (ONCE) finish();
  }
  if (const unsigned long long m = ONCE ? 0ull : __ballot(alone)) {
    // The longest walks decide how long a launch lasts, and they end with their wavefronts to themselves (20,000 PPR walkers
    // on the scale-24 graph 48 -> 43 us, 1 M 330 -> 310, 1 M walkers x 80 steps 1615 -> 1575).  Not where entries are read once:
    // there the lines moved decide, and the scalar loads would keep what is not needed again.
    const int l = __ffsll((long long)m) - 1;
    auto of = [&](uint32_t x) { return (uint32_t)__builtin_amdgcn_readlane((int)x, l); };
    const uint32_t to = walk_alone<INDEXED, false>(xadj, adjncy, table, index, stop_prob, seed, of(i), of(v), of(s), s_end,
                                                   paths + (size_t)of(i) * (len + 1));
    if (alone) {
      s = to;
      walking = to == s_end;
    }
  }
  if (!ONCE && t < n_live) finish();
  if (next_live) {  // survivors, one atomic per wavefront
    const unsigned long long m = __ballot(walking);
    if (m) {
      const int lane = threadIdx.x & 63;
      uint32_t base = 0;
      if (lane == __ffsll((long long)m) - 1) base = atomicAdd(n_next, (uint32_t)__popcll(m));
      base = (uint32_t)__shfl((int)base, __ffsll((long long)m) - 1, 64);
      if (walking) next_live[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = i;
    }
  }
  // exact 64-bit count of sampled edges (the reference reduces lengths through float, sampler_result.cuh:57-67)
  unsigned long long tot = steps;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) tot += shfl_xor_u64(tot, m);
  if (block_partials) {  // one sum per workgroup, added up by reduce_partials_kernel: no counter to clear
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = tot;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned long long b = 0;
#pragma unroll
      for (int w = 0; w < WALK_BLOCK / 64; ++w) b += s_part[w];
      block_partials[blockIdx.x] = b;
    }
  } else if ((threadIdx.x & 63) == 0) {
    call_sampled(call, wave, parts, tot);
  }
}

// Options walk_compact_every (0: one launch, every walker keeps its lane for the whole walk) and walk_read_once
// (-1: by the size of the tables, 0 / 1: never / always load entries as read-once data).
// Tables of more than 2 GiB (the last-level cache holds 256 MiB) are gathered from as read-once data.
static bool walk_reads_once(const sky_graph* g) {
  const long long mode = option(g, OPT_WALK_READ_ONCE);
  return mode < 0 ? (uint64_t)g->E * sizeof(AliasEntry) > (2ull << 30) : mode != 0;
}

template <bool INDEXED>
static void launch_walk(sky_graph* g, const uint32_t* seeds, const uint32_t* live, const uint32_t* n_live_dev,
                        uint32_t n_live, uint32_t len, uint32_t s_begin, uint32_t s_end, float stop_prob, uint64_t seed,
                        uint32_t* paths, uint32_t* lengths, uint32_t* next_live, uint32_t* n_next,
                        CallDevice* call, unsigned long long* partials, uint32_t per = 64) {
  const uint32_t walkers = WALK_BLOCK / 64 * per;  // of a workgroup
  const dim3 grid((n_live + walkers - 1) / walkers), block(WALK_BLOCK);
  if (walk_reads_once(g))
    hipLaunchKernelGGL((walk_offline_kernel<INDEXED, true>), grid, block, 0, g->stream, g->xadj, g->adjncy, g->table,
                       INDEXED ? g->walk_index : nullptr, seeds, live, n_live_dev, n_live, g->V, len, s_begin, s_end, stop_prob,
                       seed, paths, lengths, next_live, n_next, call, g->call.parts, partials, per);
  else
    hipLaunchKernelGGL((walk_offline_kernel<INDEXED, false>), grid, block, 0, g->stream, g->xadj, g->adjncy, g->table,
                       INDEXED ? g->walk_index : nullptr, seeds, live, n_live_dev, n_live, g->V, len, s_begin, s_end, stop_prob,
                       seed, paths, lengths, next_live, n_next, call, g->call.parts, partials, per);
}

// Few walkers get a wavefront each.  Beyond ALONE_SCALAR the vector cache takes part (4,096 walkers x 80 steps on the scale-16 graph
// 60.8 us all scalar, 54.9 with it; 1,000 walkers 35.4 and 37.5), and with the walk index, whose entries leave no load to
// request ahead, a lane each is as fast (4,000 walkers on the scale-22 graph 70 us both ways; 2,000 walkers 45 -> 37).
// Up to 8,192 are as many wavefronts as the GPU holds (twice as many walk in two turns: 130 us, 97 with a lane each), but
// where a lane's gathers come from L2 or the walk is short half as many are the limit (8,000 walkers, a lane / a wavefront each:
// scale 14, 30 steps 31.6 / 36.8; scale 21, 30 steps 47.8 / 38.5, 6 steps 20.4 / 23; 4,000: scale 14, 6 steps 19.3 / 20.1,
// 16 steps 24.0 / 23.9, 30 steps 31 / 29).
constexpr uint32_t ALONE_SCALAR = 2048;
static uint32_t alone_walkers(const sky_graph* g, uint32_t len) {
  if (g->has_walk_index || len < 16) return ALONE_SCALAR;
  return len >= 24 && (uint64_t)g->E * sizeof(AliasEntry) > (4u << 20) ? 8192u : 4096u;
}
// Walkers of a wavefront beyond that: 16 while three such wavefronts to a SIMD hold them all, because each waits in every step for the
// slowest of its gathers.  Not on tables that L2 holds, where it does not wait long.  (64 / 16, us: 10,000 PPR walkers on the scale-24 graph
// with the index 33.9 / 30.7, 30,000 45 / 42.7, 50,000 without 57.5 / 54, 10,000 on the scale-22 graph 44.6 / 38, 12,000 x 80, scale 20,
// 124 / 112, 20,000 x 80 on the scale-25 graph with 30 edges a vertex 162 / 152; 60,000 x 40, scale 20, 87 / 88, 130,000 with the index 59.5 / 60.7;
// 30,000 x 60, scale 18, 78.7 / 80.2, 50,000 x 50 on the scale-14 graph 42.5 / 48.4.  32: in between.)
static uint32_t lane_walkers(const sky_graph* g, uint32_t N) {
  return N <= 3u * 1024u * 16u && (uint64_t)g->E * sizeof(AliasEntry) > (32u << 20) ? 16u : 64u;
}
int walk_offline(sky_graph* g, const uint32_t* seeds, uint32_t N, uint32_t len, float stop_prob, uint64_t seed,
                 uint32_t* paths, uint32_t* lengths, uint64_t* sampled, double* seconds) {
  hipStream_t st = g->stream;
  CallDevice* call = nullptr;
  SKY_TRY(call_begin(g, &call));
  const uint32_t every = (uint32_t)option(g, OPT_WALK_COMPACT_EVERY);
  const bool segmented = every > 0 && every < len && N > 0;
  const uint32_t nseg = segmented ? (len + every - 1) / every : 1;
  uint32_t *lists = nullptr, *counts = nullptr;
  if (segmented) {  // two lists of walker numbers used in turn, one survivor count per segment
    SKY_TRY(pool_get(g, sky_graph::POOL_WALK_LIST, (size_t)2 * N * 4, (void**)&lists));
    SKY_TRY(pool_get(g, sky_graph::POOL_WALK_COUNTS, (size_t)(nseg + 1) * 4, (void**)&counts));
    SKY_HIP(hipMemsetAsync(counts, 0, (size_t)(nseg + 1) * 4, st));
  }
  auto run = [&](auto... a) {
    if (g->has_walk_index) launch_walk<true>(g, a...);
    else launch_walk<false>(g, a...);
  };
  if (N && N <= alone_walkers(g, len) && !segmented) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(N), dim3(64), 0, st, g->xadj, g->adjncy, g->table, g->walk_index, seeds, g->V, len, stop_prob,
                         seed, paths, lengths, call);
    };
    const bool vec = N > ALONE_SCALAR;
    if (g->has_walk_index) go(walk_alone_kernel<true, false>);
    else vec ? go(walk_alone_kernel<false, true>) : go(walk_alone_kernel<false, false>);
    return call_end(g, sampled, seconds, lengths, N);
  }
  const uint32_t per = segmented ? 64u : lane_walkers(g, N);
  g->call.parts = call_parts((N + per - 1ull) / per);
  if (N && !segmented) {
    run(seeds, (const uint32_t*)nullptr, (const uint32_t*)nullptr, N, len, 0u, len, stop_prob, seed, paths, lengths,
        (uint32_t*)nullptr, (uint32_t*)nullptr, call, (unsigned long long*)nullptr, per);
  } else if (N) {
    for (uint32_t k = 0; k < nseg; ++k) {
      const uint32_t s0 = k * every, s1 = std::min(len, s0 + every);
      const uint32_t* in = k ? lists + (size_t)((k - 1) & 1) * N : nullptr;
      uint32_t* out = s1 < len ? lists + (size_t)(k & 1) * N : nullptr;
      // the survivors of segment k - 1 are counted in counts[k]; the grid covers all N, blocks past the count leave
      run(seeds, in, k ? counts + k : (const uint32_t*)nullptr, N, len, s0, s1, stop_prob, seed, paths, lengths, out,
          counts + k + 1, call, (unsigned long long*)nullptr);
    }
  }
  return call_end(g, sampled, seconds);
}

// ---------------------------------------------------------------- walk index
// Optional 16-byte entries {prob, alias, neighbour of this slot, neighbour of the alias slot} beside the 8-byte
// table: a step then reads one entry and needs no gather from adjncy.  Built from the finished tables by one pass
// over the slots; a tile of 1024 slots finds its rows through the row that holds the tile's first slot.
constexpr uint32_t IDX_TILE = 1024;
constexpr uint32_t IDX_ROWS = 4096;  // row offsets of a tile kept in LDS; tiles that span more rows search xadj itself

__global__ __launch_bounds__(256) void index_tile_rows_kernel(const uint32_t* __restrict__ xadj, uint32_t V,
                                                              uint32_t* __restrict__ row_of_tile,
                                                              CallDevice* __restrict__ call) {
  call_stamp(call);
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= V) return;
  const uint32_t lo = xadj[v], hi = xadj[v + 1];
  for (uint64_t t = ((uint64_t)lo + IDX_TILE - 1) / IDX_TILE; t * IDX_TILE < hi; ++t) row_of_tile[t] = v;
}

__global__ __launch_bounds__(256) void index_fill_kernel(const uint32_t* __restrict__ xadj,
                                                         const uint32_t* __restrict__ adjncy,
                                                         const AliasEntry* __restrict__ table,
                                                         const uint32_t* __restrict__ row_of_tile, uint32_t ntiles,
                                                         uint32_t V, uint32_t E, WalkEntry* __restrict__ index) {
  __shared__ uint32_t s_x[IDX_ROWS];
  const uint32_t t = blockIdx.x;
  const uint32_t v0 = row_of_tile[t], v1 = t + 1 < ntiles ? row_of_tile[t + 1] : V - 1;
  const uint32_t rows = v1 - v0 + 1;  // rows v0..v1 hold every slot of the tile
  const bool in_lds = rows <= IDX_ROWS;
  if (in_lds)
    for (uint32_t k = threadIdx.x; k < rows; k += 256u) s_x[k] = xadj[v0 + k];
  __syncthreads();
  const uint32_t* x = in_lds ? s_x : xadj + v0;
#pragma unroll
  for (int k = 0; k < (int)(IDX_TILE / 256); ++k) {
    const uint32_t i = t * IDX_TILE + k * 256u + threadIdx.x;
    if (i >= E) continue;
    // the last row of v0..v1 that starts at or before slot i (rows without entries share their start with the
    // next row and are passed over)
    uint32_t lo = 0, n = rows;
    while (n > 1) {
      const uint32_t half = n >> 1;
      lo = x[lo + half] <= i ? lo + half : lo;
      n -= half;
    }
    const uint32_t off = x[lo];
    const AliasEntry e = table[i];
    WalkEntry w;
    w.prob = e.prob;
    w.alias = e.alias;
    w.nbr_col = adjncy[i];
    w.nbr_alias = e.alias == SKY_INVALID ? SKY_INVALID : adjncy[off + e.alias];
    index[i] = w;
  }
}

int build_walk_index(sky_graph* g, double* seconds) {
  hipStream_t st = g->stream;
  if (seconds) *seconds = 0;
  if (!g->walk_index) SKY_TRY(alloc_padded(&g->walk_index, (size_t)g->E));
  if (g->E == 0) return SKY_OK;
  const uint32_t ntiles = (g->E + IDX_TILE - 1) / IDX_TILE;
  uint32_t* row_of_tile = nullptr;
  SKY_TRY(pool_get(g, sky_graph::POOL_WALK_LIST, (size_t)ntiles * 4, (void**)&row_of_tile));
  CallDevice* call = nullptr;
  SKY_TRY(call_begin(g, &call));
  hipLaunchKernelGGL(index_tile_rows_kernel, dim3((g->V + 255) / 256), dim3(256), 0, st, g->xadj, g->V, row_of_tile, call);
  hipLaunchKernelGGL(index_fill_kernel, dim3(ntiles), dim3(256), 0, st, g->xadj, g->adjncy, g->table, row_of_tile,
                     ntiles, g->V, g->E, g->walk_index);
  SKY_TRY(call_end(g, nullptr, seconds));
  g->has_walk_index = true;
  return SKY_OK;
}

// ---------------------------------------------------------------- the same walk without any allocation
// For callers that cannot allocate (HIP graph capture, serving loops): the per-workgroup counts of sampled
// edges go to a file-scope device array instead of a counter from hipMalloc, a second kernel adds them up into
// the caller's own device word, no event is created and nothing is copied to the host.  Every call on a GPU
// shares that GPU's array: calls that overlap on one GPU race.  Nothing in it needs clearing (each workgroup of
// a call writes its own element before the sum reads it).
constexpr uint32_t NOALLOC_MAX_BLOCKS = 16384;  // 128 KiB of device memory per GPU, held until the process ends
constexpr int NOALLOC_MAX_DEVICES = 64;
static __device__ __align__(256) unsigned long long scratch[NOALLOC_MAX_BLOCKS];
static unsigned long long* g_scratch_ptr[NOALLOC_MAX_DEVICES];  // device address of `scratch` on each GPU

__global__ __launch_bounds__(1024) void reduce_partials_kernel(const unsigned long long* __restrict__ partials,
                                                               uint32_t n, unsigned long long* __restrict__ out) {
  __shared__ unsigned long long s_w[16];
  unsigned long long t = 0;
  for (uint32_t k = threadIdx.x; k < n; k += 1024u) t += partials[k];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) t += shfl_xor_u64(t, m);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long b = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) b += s_w[w];
    *out = b;
  }
}

int walk_offline_noalloc(sky_graph* g, const uint32_t* seeds, uint32_t N, uint32_t len, float stop_prob,
                         uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled_device) {
  const uint64_t max_walkers = (uint64_t)NOALLOC_MAX_BLOCKS * WALK_BLOCK;
  if (N > max_walkers)
    return fail(SKY_ERR_LIMIT, "sky_walk_offline_noalloc: " + std::to_string(N) + " walkers, the static scratch holds " +
                                   std::to_string(max_walkers) + " (split the batch)");
  int dev = 0;
  SKY_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return fail(SKY_ERR_LIMIT, "sky_walk_offline_noalloc: device index beyond 63");
  if (dev != g->device)  // the scratch array of the current device would be handed to kernels that read another device's graph
    return fail(SKY_ERR_STATE, "sky_walk_offline_noalloc: the graph lives on device " + std::to_string(g->device) +
                                   ", the current device is " + std::to_string(dev));
  if (!g_scratch_ptr[dev]) {  // once per device, with that device current: each GPU holds its own copy of the array
    unsigned long long* p = nullptr;
    SKY_HIP(hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = p;
  }
  unsigned long long* const partials = g_scratch_ptr[dev];
  hipStream_t st = g->stream;
  const uint32_t blocks = (N + WALK_BLOCK - 1) / WALK_BLOCK;
  if (blocks) {
    if (g->has_walk_index)
      launch_walk<true>(g, seeds, nullptr, nullptr, N, len, 0u, len, stop_prob, seed, paths, lengths, nullptr, nullptr,
                        nullptr, partials);
    else
      launch_walk<false>(g, seeds, nullptr, nullptr, N, len, 0u, len, stop_prob, seed, paths, lengths, nullptr, nullptr,
                         nullptr, partials);
  }
  if (sampled_device)
    hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(1024), 0, st, partials, blocks,
                       reinterpret_cast<unsigned long long*>(sampled_device));
  SKY_HIP(hipGetLastError());
  return SKY_OK;
}

// ---------------------------------------------------------------- node2vec by rejection
// The second-order law of a step, w(v,x) * f(x) with f = 1/p for the previous vertex, 1 for its
// neighbours and 1/q for the rest (src/api/bias_node2vec.cu:15-27), is sampled without building the
// step's table: trial t draws a candidate from the first-order table of the current vertex with
// r_t = Philox(seed; i, s, t, DOM_WALK) (trial 0 shares the counter of the stop test) and keeps it when
// u24(r_t.w) * fmax < f(candidate), fmax = max(1/p, 1, 1/q); the 65537th candidate is kept whatever
// it is.  One membership search in the previous vertex's sorted row per trial, instead of one
// per neighbour of the current vertex.  The reference's unbiased node2vec walker rejects the same way
// (src/unbiased_walk.cu:14-60).
//
// G lanes per walker, which hold its state alike and share the work of a step: the random numbers, which cost more
// instructions than everything else in a trial, are computed for several trials of several steps at once, one lane each, and
// all search the previous row together, G probes per round.  Most trials need no search at all: whether the candidate is
// kept depends on its being a neighbour of the previous vertex only when the drawn number lies between the two cases'
// limits.  The bounds of the candidate's own row are requested before the search, for the step after.  The first probe, a line of memory for
// every lane where the previous row is long, goes out with the table's entry, but only for a drawn number between the limits: lines are what
// bounds large graphs (40,000 x 80 on the scale-24 graph read 10.6 M of them, 32 G a second of the 50 that random reads reach; us, for every step /
// for such numbers: 40,000 x 80 345 / 325, 1,000 x 80 with q = 1/2 there 143 / 117, 50,000 x 40, scale 20, 175 / 168, 8,000 x 30, scale 22,
// p = q = 2, 138 / 130, 150,000 x 30, scale 22, 286 / 275, 10,000 x 50, scale 21, p = 1/2, q = 1, 152 / 137; in turns of four trials one of which
// nearly always asks 273 / 297, so there it stays with the move; behind the entry's load instead of in front of it 324 / 368: what waits for the
// entry then waits for a probe too).  Leaving it until it is known to be needed or reading the next step's entry during the search as if the
// candidate were kept was slower, and doing the whole search beside the next step's loads and taking a refused step back gains on the largest
// graphs what it costs elsewhere several times (40,000 x 80 on the scale-24 graph 324 / 312, but 50,000 x 40, scale 20, 167 / 187, 500 x 60, scale 14,
// 68 / 99, 8,000 x 30, scale 22, q = 2, 129 / 231).
//
// A turn of the loop is TR trials of every walker of the wavefront, whichever step each of them is in: where a turn was a step,
// every walker waited in each for the one with the most trials.
//
// A walk lasts as long as its longest chain of dependent loads, so G is the largest whose wavefronts are all resident at
// once (seven on each of the 1024 SIMDs); once the walkers alone fill the GPU the lanes are worth more as walkers.
// Where no trial is in need of a search (q = 1) two lanes, that hold the next trial's numbers and the next step's, are as good as many
// (p = 4, 50,000 walkers x 40 on the scale-20 graph: 2 lanes 110 us, 8 191; 8,000 x 30 on the scale-22 graph: 2 59, 4 60, 32 102;
// 500 x 60, scale 16: 2 89, 4 74, 64 77).
// TR: where half of the trials fail or more, four are drawn at once, a lane each, and the first that is kept ends the step, or, of
// two that depend on the previous row, the first is searched for and the other left to the next turn; the first that ends the walk, if it
// comes before, ends it.  (One at a time / four, us: p = 1/4,
// q = 1: 500 x 60, scale 16, 224 / 121, 8,000 x 30, scale 22, 256 / 143, 50,000 x 40, scale 20, 371 / 273; p = 1/2, q = 2: 220 / 143, 275 / 178,
// 490 / 396.  Where three in four are kept, p = 2, q = 1/2: 91 / 101, 120 / 134, 222 / 294; where the walkers alone fill the GPU, 150,000 x 30,
// scale 22, p = 1/4, q = 1: 482 / 637.)
constexpr uint64_t N2V_LANES = 7ull * 1024 * 64;
constexpr int N2V_TRIALS = 4;
template <int G>
__device__ __forceinline__ unsigned long long group_ballot(bool p) {
  const unsigned long long b = __ballot(p) >> (lane_id() & (64u - G));
  return G == 64 ? b : b & ((1ull << (G & 63)) - 1ull);
}
// Every lane of the group must call this together with the same row, n and key.
// The first round's probes depend on the row alone: group_first_probe loads them as soon as the row is known
// (a step before the key is), and group_row_has takes the value.
template <int G>
__device__ __forceinline__ uint32_t group_first_probe(const uint32_t* __restrict__ row, uint32_t n) {
  const uint32_t gl = lane_id() & (G - 1);
  if (n <= (uint32_t)G) return gl < n ? row[gl] : 0xFFFFFFFFu;
  const uint32_t p = (gl + 1) * (n / (G + 1) + 1) - 1;
  return p < n ? row[p] : 0xFFFFFFFFu;  // no vertex has this id
}
template <int G>
__device__ __forceinline__ bool group_row_has(const uint32_t* __restrict__ row, uint32_t n, uint32_t key, uint32_t x0) {
  const uint32_t gl = lane_id() & (G - 1);
  if (n <= (uint32_t)G) return group_ballot<G>(x0 == key) != 0;
  uint32_t lo = 0, len = n;  // if the key is in the row it is in [lo, lo + len)
  bool first_round = true;
  while (len > (uint32_t)G) {
    const uint32_t step = len / (G + 1) + 1, end = lo + len;
    const uint32_t p = lo + (gl + 1) * step - 1;           // probe gl: last element of part gl
    const uint32_t x = first_round ? x0 : (p < end ? row[p] : 0xFFFFFFFFu);
    first_round = false;
    const uint32_t c = (uint32_t)__popcll(group_ballot<G>(x < key));  // parts that lie wholly below the key
    lo += c * step;
    len = min(step, end - lo);
  }
  return group_ballot<G>(gl < len && row[lo + gl] == key) != 0;
}

template <int G, int TR>
__global__ __launch_bounds__(WALK_BLOCK) void walk_n2v_reject_group_kernel(
    const uint32_t* __restrict__ xadj, const uint32_t* __restrict__ adjncy,
    const AliasEntry* __restrict__ table, const uint32_t* __restrict__ seeds, uint32_t walker0, uint32_t N, uint32_t V, uint32_t len,
    float fp, float fq, float fmax, float stop_prob, uint64_t seed, bool once, uint32_t* __restrict__ paths,
    uint32_t* __restrict__ lengths, CallDevice* __restrict__ call, uint32_t parts) {
  // One trial a turn: the numbers of the next one and of the next step's first are kept, which takes two lanes.  Four: those of the turn.
  static_assert(TR == 1 ? G >= 2 : TR == N2V_TRIALS && G >= TR, "a lane for every number that is kept");
  // Numbers kept of a step, a lane each, of the last one fewer.
  constexpr uint32_t TRIALS = TR == 1 ? (G < 4 ? 1 : G < 16 ? 3 : G < 32 ? 4 : 8) : G < 16 ? TR : 2 * TR;
  if (walker0 == 0) call_stamp(call);
  const uint64_t wi = walker0 + ((uint64_t)blockIdx.x * WALK_BLOCK + threadIdx.x) / G;
  const uint32_t i = (uint32_t)wi, gl = threadIdx.x & (G - 1), my = gl & (TR - 1);
  const int base = (int)(lane_id() & (64u - G));  // first lane of the group
  const bool first = gl == 0;                     // the lane that writes for the group
  uint32_t s = 0;
  if (wi < N) {
    uint32_t* path = paths + (size_t)i * (len + 1);
    uint32_t v = seeds[i];
    if (first) path[0] = v;
    if (v < V && len) {
      bounds2u x = *reinterpret_cast<const bounds2u*>(xadj + v);
      uint32_t off = x.x, deg = x.y - x.x, t = 0;
      uint32_t prev = 0, prev_off = 0, prev_deg = 0, x0 = 0xFFFFFFFFu;
      // lane gl: trial sb_t + gl of step sb, then trial gl % TRIALS of step sb + gl / TRIALS
      uint32_t sb = 0, tb = 0;
      auto numbers = [&] { return philox(seed, i, sb + gl / TRIALS, gl % TRIALS + (gl < TRIALS ? tb : 0u), DOM_WALK); };
      auto lane_of = [&](uint32_t step, uint32_t trial) -> uint32_t {  // G or more: not among the kept ones
        const uint32_t k = step == sb ? trial - tb : trial;
        return k < TRIALS ? (step - sb) * TRIALS + k : (uint32_t)G;
      };
      // what lane l holds; the only walker of a wavefront needs no exchange through LDS for it
      auto of = [&](uint32_t x, int l) -> uint32_t {
        if (G == 64 && TR == 1) return (uint32_t)__builtin_amdgcn_readlane((int)x, __builtin_amdgcn_readfirstlane(l));
        return (uint32_t)__shfl((int)x, l, 64);
      };
      u32x4 mine = numbers();
      const float lo = fminf(1.0f, fq), hi = fmaxf(1.0f, fq);
      for (;;) {
        if (TR > 1 && __any(lane_of(s, t) >= (uint32_t)G || lane_of(s, t + TR - 1) >= (uint32_t)G)) {
          sb = s;
          tb = t;
          mine = numbers();
        }
        const int from = base + (int)lane_of(s, t);
        if (t == 0 && ((stop_prob > 0.0f && u24(of(mine.z, from)) < stop_prob) || deg == 0)) break;
        const uint32_t rx = of(mine.x, from + (int)my), ry = of(mine.y, from + (int)my), rw = of(mine.w, from + (int)my);
        const float need = u24(rw) * fmax;
        // The previous row can only be asked about a candidate drawn with such a number: its first probe is on its way then, beside the entry.
        if (TR == 1) x0 = group_first_probe<G>(adjncy + prev_off, need >= lo && need < hi ? prev_deg : 0u);  // no row before the first step
        const uint32_t col = __umulhi(rx, deg);
        const AliasEntry e = once ? load_entry_once(table + off + col) : table[off + col];
        // The numbers of what may come next, while the entry is on its way: all walkers of the wavefront together.
        if (G > TR && __any((TR == 1 && lane_of(s, t + 1) >= (uint32_t)G) || lane_of(s + 1, TR - 1) >= (uint32_t)G)) {
          sb = s;
          tb = t + 1;
          mine = numbers();
          asm volatile("" : "+v"(mine.x), "+v"(mine.y), "+v"(mine.z), "+v"(mine.w));
        }
        const uint32_t cand = u24(ry) < e.prob ? col : e.alias;
        // The walk ends at a row without weight.  A table from outside may keep the column in some of its entries, or for some numbers: in
        // a turn of several trials a lane then ends the walk while its neighbours do not, and the group decides below.
        const bool ends = cand == SKY_INVALID;
        if (TR == 1 && ends) break;
        uint32_t next = adjncy[off + (TR > 1 && ends ? col : cand)];
        x = *reinterpret_cast<const bounds2u*>(xadj + next);
        bool keep = s == 0 || t + my >= 65536u, ask = false;
        if (!keep) {
          if (next == prev) keep = need < fp;
          else if (need < lo) keep = true;
          else ask = need < hi;
        }
        uint32_t went = 1;  // trials that this turn has decided
        if (TR == 1) {
          if (ask) keep = need < (group_row_has<G>(adjncy + prev_off, prev_deg, next, x0) ? 1.0f : fq);
        } else {
          // bit j: trial t + j is kept; bit 8 + j: that depends on the previous row; bit 16 + j: it ends the walk
          uint32_t b = (ends ? 65536u : keep ? 1u : ask ? 256u : 0u) << my;
          b |= dpp0<DPP_QUAD_XOR1, 0xF>(b);
          b |= dpp0<DPP_QUAD_XOR2, 0xF>(b);
          const uint32_t kept = b & 255u, asked = (b >> 8) & 255u, ended = b >> 16;
          uint32_t left = kept | asked | ended | 1u << TR;
          went = (uint32_t)__ffs((int)left) - 1u;
          if ((asked >> went) & 1u) {
            const int l = base + (int)went;
            const uint32_t key = (uint32_t)__shfl((int)next, l, 64);
            const float limit = __shfl(need, l, 64);
            if (!(limit < (group_row_has<G>(adjncy + prev_off, prev_deg, key, x0) ? 1.0f : fq))) {  // on to the next one that may be kept
              left &= left - 1u;
              went = (uint32_t)__ffs((int)left) - 1u;
              keep = (kept >> went) & 1u;
            } else {
              keep = true;
            }
          } else {
            keep = (kept >> went) & 1u;
          }
          if ((ended >> went) & 1u) break;
          if (keep) {
            const int l = base + (int)went;
            next = (uint32_t)__shfl((int)next, l, 64);
            x.x = (uint32_t)__shfl((int)x.x, l, 64);
            x.y = (uint32_t)__shfl((int)x.y, l, 64);
          }
        }
        if (keep) {
          prev = v;
          prev_off = off;
          prev_deg = deg;
          if (TR > 1 && lo < hi) x0 = group_first_probe<G>(adjncy + off, deg);  // some trial of four asks; in flight during the loads of the step
          v = next;
          off = x.x;
          deg = x.y - x.x;
          t = 0;
          ++s;
          if (first) path[s] = v;
          if (s == len) break;
        } else {
          t += went;
        }
      }
    }
    if (first) lengths[i] = s;
  }
  unsigned long long t = first ? s : 0u;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) t += shfl_xor_u64(t, m);
  if ((threadIdx.x & 63) == 0) call_sampled(call, blockIdx.x * (WALK_BLOCK / 64) + threadIdx.x / 64, parts, t);
}

int walk_node2vec_reject(sky_graph* g, float p, float q, const uint32_t* seeds, uint32_t N, uint32_t len,
                         float stop_prob, uint64_t seed, uint32_t* paths, uint32_t* lengths, uint64_t* sampled,
                         double* seconds) {
  hipStream_t st = g->stream;
  double build_sec = 0;
  if (!g->has_tables) SKY_TRY(build_all_tables(g, &build_sec));  // first-order tables, built on demand
  const float fp = 1.0f / p, fq = 1.0f / q;
  const float fmax = fmaxf(1.0f, fmaxf(fp, fq));
  // every candidate is kept: the first-order walk, whose trial 0 shares the counters, and whose one launch has a lane for each walker
  if (fp == 1.0f && fq == 1.0f && N <= 0xFFFFFFFFu / WALK_BLOCK * WALK_BLOCK) {
    SKY_TRY(walk_offline(g, seeds, N, len, stop_prob, seed, paths, lengths, sampled, seconds));
    if (seconds) *seconds += build_sec;
    return SKY_OK;
  }
  CallDevice* call = nullptr;
  SKY_TRY(call_begin(g, &call));
  auto run = [&](auto lanes, auto trials) {
    constexpr int G = decltype(lanes)::value;
    g->call.parts = call_parts((uint64_t)N * G / 64);
    const uint64_t most = 0x80000000ull / G;  // walkers of one launch: below 2^32 threads
    for (uint64_t f = 0; f < N; f += most) {
      const uint64_t threads = std::min<uint64_t>(most, N - f) * G;
      hipLaunchKernelGGL((walk_n2v_reject_group_kernel<G, decltype(trials)::value>), dim3((uint32_t)((threads + WALK_BLOCK - 1) / WALK_BLOCK)),
                         dim3(WALK_BLOCK), 0, st, g->xadj, g->adjncy, g->table, seeds, (uint32_t)f, N, g->V, len, fp, fq, fmax,
                         stop_prob, seed, walk_reads_once(g), paths, lengths, call, g->call.parts);
    }
  };
  using One = std::integral_constant<int, 1>;
  using Four = std::integral_constant<int, N2V_TRIALS>;
  uint64_t lanes = N ? N2V_LANES / N : 0;  // per walker
  // (1 + 1 / q) / 2 / fmax of the candidates are kept where one in two is a neighbour of the previous vertex.
  const bool four = lanes >= 8 && (1.0f + fq) <= fmax;
  if (fq == 1.0f) lanes = four ? std::max<uint64_t>(N2V_TRIALS, lanes / 2) : lanes >= 32 ? 4 : 2;
  auto pick = [&](auto width) {
    if (four) run(width, Four{});
    else run(width, One{});
  };
  if (lanes >= 64) pick(std::integral_constant<int, 64>{});
  else if (lanes >= 32) pick(std::integral_constant<int, 32>{});
  else if (lanes >= 16) pick(std::integral_constant<int, 16>{});
  else if (lanes >= 8) pick(std::integral_constant<int, 8>{});
  else if (lanes >= 4) pick(std::integral_constant<int, 4>{});
  else if (N) run(std::integral_constant<int, 2>{}, One{});
  SKY_TRY(call_end(g, sampled, seconds));
  if (seconds) *seconds += build_sec;
  return SKY_OK;
}

}  // namespace sky
