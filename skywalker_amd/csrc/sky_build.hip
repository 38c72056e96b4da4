// Offline alias-table construction for every vertex (replaces ConstructAliasTableKernel /
// ConstructTable of the reference, src/createTable.cu:48-179, and the constructors of
// include/alias_table_new.cuh it calls).
//
// The table of a row is a pure function of its weights, defined with exact integer
// prefix sums so that no kernel below can change a bit of it by changing how it
// parallelises:
//   S     = sum floor(w_i 2^64)  (128 bit)        scale = deg / double(S)      p_i = w_i * scale
//   F     = 40 fraction bits (62 - floor(log2 deg) for rows of 2^22 entries and more)
//   t_i   = (p_i - 1) 2^F  ;  heavy iff t_i >= 0.5 : surplus U_i = max(rint(t_i), 1)
//                             light otherwise      : deficit D_i = rint(-t_i)      (ties to even)
//   SL(i) = inclusive prefix sum of deficits over slots <= i,  SH(i) likewise of surpluses
//   light i : prob = float(p_i), alias = first slot m with SH(m) > SL(i) - D_i
//             (the last heavy if there is none; itself if the row has no heavy)
//   heavy j : last heavy of the row -> prob 1, alias itself; otherwise with y = SH(j):
//             l = first slot with SL(l) >= y;  found -> prob = (2^F + y - SL(l)) 2^-F, alias = next heavy
//                                              none  -> prob 1, alias itself
// This is the pairing a sequential two-pointer Vose sweep over (lights in slot order,
// heavies in slot order) produces, written so that every entry is resolved by two
// prefix sums and a binary search: no queues, no float atomics, no rollback.
//
// Dispatch is by degree class (sky_graph.h): one lane per vertex (deg <= 2), 2 to 32 lanes per vertex with the prefix
// arrays in a per-wave LDS strip (deg <= 192), 64 to 512 threads per vertex that pair by a merge in LDS (deg <= 5117),
// 512 threads that hold or stream the row (sky_build_stream.hip), and the tile-parallel path of sky_build_tiled.hip for
// longer rows.  Builds of up to FUSED_MAX_ENTRIES send the same row builders out in few launches (sky_build_fused.hip).
#include <algorithm>
#include <vector>

#include "sky_build_fused.h"
#include "sky_build_rows.h"
#include "sky_graph.h"

namespace sky {

// Class kernels: `vlist` is the class's segment of the row list, `count` its length.  Every row's builder writes its flag
// (1, or 0 for a row without weight): a build may follow one that found other weights.
template <int G, int PER>
__global__ __launch_bounds__(256) void build_group_kernel(const RowRef* __restrict__ vlist, uint32_t count,
                                                          const float* __restrict__ wgt,
                                                          AliasEntry* __restrict__ table,
                                                          int8_t* __restrict__ valid) {
  __shared__ uint64_t smem[(group_lds_bytes(G, PER, 256) + 7) / 8];
  const uint32_t grp = blockIdx.x * (256 / G) + threadIdx.x / G;
  RowRef rr{0, 0, 0, 0};
  if (grp < count) rr = vlist[grp];
  const bool ok = group_build_row<G, PER>(rr.off, rr.d, wgt, table, smem);
  if ((threadIdx.x & (G - 1)) == 0 && grp < count) valid[rr.v] = ok ? 1 : 0;
}

__global__ __launch_bounds__(128) void build_begin_kernel(uint32_t* __restrict__ counters, uint32_t words,
                                                          CallDevice* call, ForkMark fork) {
  call_stamp(call);
  fork_mark(fork);
  for (uint32_t i = threadIdx.x; i < words; i += 128u) counters[i] = 0;
}

// ---------------------------------------------------------------- binning
// `src` lists the vertices to bin (n of them); a null src means vertices 0..n-1.  Block b of the
// count and scatter kernels owns the items [b * per_block, (b + 1) * per_block): the count kernel
// leaves one row of class counts per block, bin_offsets_kernel turns the rows into each block's
// first position inside every class segment, and the scatter kernel hands out positions from
// cursors it keeps in LDS, so no global atomic is involved and the lists come out grouped by block.
constexpr int BIN_BLOCKS = 4096;  // most blocks a binning pass uses
constexpr int BIN_ITEMS = 4;      // vertices per thread and step
// at most BIN_BLOCKS blocks, each a multiple of one scatter step
static uint32_t bin_per_block(uint32_t n) {
  const uint32_t step = 256u * BIN_ITEMS;
  return ((n + BIN_BLOCKS - 1) / BIN_BLOCKS + step - 1) / step * step;
}

__global__ __launch_bounds__(256) void bin_count_kernel(const uint32_t* __restrict__ xadj,
                                                        const uint32_t* __restrict__ src, uint32_t n,
                                                        uint32_t per_block,
                                                        uint32_t* __restrict__ blk_cnt,
                                                        unsigned long long* __restrict__ class_edges) {
  __shared__ uint32_t s_cnt[CLS_COUNT];
  __shared__ unsigned long long s_edges[CLS_COUNT];
  if (threadIdx.x < CLS_COUNT) {
    s_cnt[threadIdx.x] = 0;
    s_edges[threadIdx.x] = 0;
  }
  __syncthreads();
  const uint32_t lo = blockIdx.x * per_block, hi = min(n, lo + per_block);
  uint32_t tiny_edges = 0;  // rows of 1..2 entries, the commonest kind of a power-law graph, stay out of the LDS atomics
  // four vertices per thread and step: their loads are in flight together (one at a time, the loop waits a
  // memory round trip per vertex)
  for (uint32_t chunk = lo; chunk < hi; chunk += 256u * BIN_ITEMS) {
    uint32_t d[BIN_ITEMS];
#pragma unroll
    for (int k = 0; k < BIN_ITEMS; ++k) {
      const uint32_t i = chunk + k * 256u + threadIdx.x;
      d[k] = 0;
      if (i < hi) {
        const uint32_t v = src ? src[i] : i;
        d[k] = xadj[v + 1] - xadj[v];
      }
    }
#pragma unroll
    for (int k = 0; k < BIN_ITEMS; ++k) {
      const int c = degree_class(d[k]);
      if (c >= CLS_G2) {
        atomicAdd(&s_cnt[c], 1u);
        atomicAdd(&s_edges[c], (unsigned long long)d[k]);
      } else {
        tiny_edges += d[k];  // 0 for an empty row
      }
    }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) tiny_edges += (uint32_t)__shfl_xor((int)tiny_edges, m, 64);
  if ((threadIdx.x & 63) == 0 && tiny_edges) atomicAdd(&s_edges[CLS_TINY], (unsigned long long)tiny_edges);
  __syncthreads();
  if (threadIdx.x < CLS_COUNT) {
    blk_cnt[blockIdx.x * CLS_COUNT + threadIdx.x] = s_cnt[threadIdx.x];
    if (s_edges[threadIdx.x]) atomicAdd(&class_edges[threadIdx.x], s_edges[threadIdx.x]);
  }
}

// One workgroup per class: exclusive prefix of the class's per-block counts (in place), total to counts[c].
// Thread t owns a run of consecutive blocks: its loads do not wait for one another.
__global__ __launch_bounds__(256) void bin_offsets_kernel(uint32_t* __restrict__ blk_cnt, uint32_t blocks,
                                                          uint32_t* __restrict__ counts) {
  __shared__ uint32_t s_w[4];
  const uint32_t c = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr uint32_t RUN = (BIN_BLOCKS + 255) / 256;
  const uint32_t b0 = tid * RUN;
  uint32_t x[RUN], sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < RUN; ++k) {
    x[k] = b0 + k < blocks ? blk_cnt[(b0 + k) * CLS_COUNT + c] : 0u;
    sum += x[k];
  }
  const uint32_t inc = group_scan_u32<64>(sum);
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  uint32_t run = inc - sum;
  for (uint32_t w = 0; w < wave; ++w) run += s_w[w];
#pragma unroll
  for (uint32_t k = 0; k < RUN; ++k) {
    if (b0 + k < blocks) blk_cnt[(b0 + k) * CLS_COUNT + c] = run;
    run += x[k];
  }
  if (tid == 0) counts[c] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Writes each row of class >= CLS_G2 into its class segment of vlist, and finishes
// the classes that need no cooperation: deg 0 (valid = 0) and deg 1..2 (closed form).  The rows of one
// or two entries that a wavefront meets in a step go to a list of its own in LDS first and are then
// built with its lanes side by side (they are a fifth of the vertices of a power-law graph: built where
// they are met, every step would pay for them with most lanes idle).
__global__ __launch_bounds__(256) void bin_scatter_kernel(const uint32_t* __restrict__ xadj,
                                                          const float* __restrict__ wgt,
                                                          const uint32_t* __restrict__ src, uint32_t n,
                                                          uint32_t per_block, int listed_from,
                                                          const uint32_t* __restrict__ counts,
                                                          const uint32_t* __restrict__ blk_off,
                                                          RowRef* __restrict__ vlist,
                                                          AliasEntry* __restrict__ table,
                                                          int8_t* __restrict__ valid) {
  __shared__ uint32_t s_cur[CLS_COUNT];
  __shared__ uint2 s_tiny[4][64 * BIN_ITEMS];  // per wavefront: {offset, vertex} of its rows of 1..2 entries
  __shared__ uint8_t s_tiny_d[4][64 * BIN_ITEMS];
  if (threadIdx.x < CLS_COUNT) {  // the class lists lie back to back in class order
    uint32_t start = 0;
    for (uint32_t c = (uint32_t)listed_from; c < threadIdx.x; ++c) start += counts[c];  // classes below have no list
    s_cur[threadIdx.x] = start + blk_off[blockIdx.x * CLS_COUNT + threadIdx.x];
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t lo = blockIdx.x * per_block, hi = min(n, lo + per_block);
  for (uint32_t chunk = lo; chunk < hi; chunk += 256u * BIN_ITEMS) {
    uint32_t nt = 0;  // wave-uniform: rows in this wavefront's list
#pragma unroll
    for (int i = 0; i < BIN_ITEMS; ++i) {
      const uint32_t item = chunk + i * 256u + threadIdx.x;
      int c = -1;
      uint32_t v = 0, off = 0, d = 0;
      if (item < hi) {
        v = src ? src[item] : item;
        off = xadj[v];
        d = xadj[v + 1] - off;
        c = degree_class(d);
      }
      // listed_from > CLS_G2: the rows of the classes below it, empty rows included, belong to small_rows_kernel
      const bool tiny_here = c == CLS_TINY && listed_from == CLS_G2;
      const unsigned long long m = __ballot(tiny_here);
      if (tiny_here) {
        const uint32_t p = nt + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        s_tiny[wave][p] = make_uint2(off, v);
        s_tiny_d[wave][p] = (uint8_t)d;
      } else if (c >= listed_from) {
        vlist[atomicAdd(&s_cur[c], 1u)] = RowRef{v, off, d, 0};
      }
      nt += (uint32_t)__popcll(m);
      // Written here, next to its neighbours' flags; a row without weight clears it later.  Lists that a graph keeps for
      // later builds are made without touching the flags: they belong to whatever tables there are.
      if (c >= 0 && listed_from == CLS_G2) valid[v] = c != CLS_EMPTY;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (uint32_t t = lane; t < nt; t += 64u) {
      const uint2 rec = s_tiny[wave][t];
      if (!tiny_row(rec.x, s_tiny_d[wave][t], wgt, table)) valid[rec.y] = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the next step's list entries stay behind these reads
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------- rows of at most 32 entries, where they lie
__global__ __launch_bounds__(64) void small_rows_kernel(const uint32_t* __restrict__ xadj,
                                                        const float* __restrict__ wgt,
                                                        const uint32_t* __restrict__ src, uint32_t n,
                                                        uint32_t per_wave, AliasEntry* __restrict__ table,
                                                        int8_t* __restrict__ valid) {
  __shared__ uint64_t smem[(SMALL_LDS_BYTES + 7) / 8];
  small_rows_range(spread_units(blockIdx.x, gridDim.x) * per_wave, xadj, wgt, src, n, per_wave, table, valid, smem);
}

// ---------------------------------------------------------------- one row per workgroup, prefix arrays in LDS
// ROWT threads cooperate on one row of at most ROWT*4*T slots (counted from the row's 16-byte
// aligned start).  Weights are read once as aligned float4 quads; every entry is classified once
// and keeps its search key in registers; SL and SH of every slot live in LDS.  Each entry then
// does exactly one binary search, lights in SH and heavies in SL, four searches interleaved; the
// next heavy after each heavy and the last heavy of the row come from a suffix scan, not a search.
template <int ROWT, int T>
__global__ __launch_bounds__(ROWT) void build_lds_kernel(const RowRef* __restrict__ vlist,
                                                         const uint32_t* __restrict__ xadj,
                                                         const float* __restrict__ wgt,
                                                         AliasEntry* __restrict__ table, int8_t* __restrict__ valid) {
  constexpr int CAP = ROWT * 4 * T;
  constexpr int NW = ROWT / 64;
  extern __shared__ __align__(16) uint64_t smem[];
  uint64_t* s_sl = smem;
  uint64_t* s_sh = smem + CAP;
  __shared__ u128 s_wsum[NW];
  __shared__ uint64_t s_ex[2 * T * NW];
  __shared__ uint32_t s_fh[T][NW], s_lh[T][NW];

  const RowRef rr = vlist[blockIdx.x];
  const uint32_t v = rr.v, off = rr.off, d = rr.d;
  const uint32_t base = off & ~3u, lead = off - base, span = lead + d;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;

  float w[T][4];
  u128 sum{0, 0};
  uint32_t live = 0;       // bit q*4+k: slot belongs to the row
  uint32_t wave_live = 0;  // bit t: some slot of this wave's strip of sub-tile t belongs to the row
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const uint32_t pos = 4u * (t * ROWT + tid);
    if (4u * (t * ROWT + wave * 64) >= span) {  // wave-uniform: nothing of the row here
#pragma unroll
      for (int k = 0; k < 4; ++k) w[t][k] = 0.0f;
      continue;
    }
    wave_live |= 1u << t;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pos < span) x = *reinterpret_cast<const float4*>(wgt + base + pos);
    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t idx = pos + k;
      const bool in = idx - lead < d;  // one unsigned compare: slots before the row wrap around
      if (in) live |= 1u << (t * 4 + k);
      w[t][k] = in ? clamp_weight(xs[k]) : 0.0f;
      sum = add128(sum, weight_fixed(w[t][k]));
    }
  }
  sum = group_sum_u128<64>(sum);
  if (NW > 1) {
    if (lane == 0) s_wsum[wave] = sum;
    __syncthreads();
    sum = s_wsum[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) sum = add128(sum, s_wsum[i]);
  }
  if ((sum.lo | sum.hi) == 0) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if ((live >> (t * 4 + k)) & 1) {
          const uint32_t idx = 4u * (t * ROWT + tid) + k;
          table[base + idx] = AliasEntry{0.0f, SKY_INVALID};
        }
    if (tid == 0) valid[v] = 0;
    return;
  }
  if (tid == 0) valid[v] = 1;
  const Ledger L = make_ledger(d, sum);

  // classify once; amounts -> prefix sums; first / last heavy of every (sub-tile, wave)
  uint64_t dl[T][4], dh[T][4], sl[T][4], sh[T][4];
  float op[T][4];
  uint32_t heavy = 0;
  uint64_t hb_mask[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (!((wave_live >> t) & 1)) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        dl[t][k] = dh[t][k] = 0;
        op[t][k] = 0.0f;
      }
      hb_mask[t] = 0;
      if (lane == 0) {
        s_fh[t][wave] = NONE32;
        s_lh[t][wave] = 0;
      }
      continue;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int b = t * 4 + k;
      const Entry e = classify(w[t][k], L);
      const bool in = (live >> b) & 1;
      dl[t][k] = (in && !e.heavy) ? e.amount : 0;
      dh[t][k] = (in && e.heavy) ? e.amount : 0;
      op[t][k] = e.heavy ? 1.0f : (float)e.p;
      if (in && e.heavy) heavy |= 1u << b;
    }
    // first and last heavy slot of this (sub-tile, wave), from a ballot over the quads that hold a heavy
    const uint32_t m = (heavy >> (t * 4)) & 15u;
    const uint64_t bal = __ballot(m != 0);
    hb_mask[t] = bal;
    // readlane must see every lane's m: keep it out of divergent code
    uint32_t fh = NONE32, lh = 0;  // lh holds index + 1, 0 = none
    if (bal) {
      const int l0 = __ffsll((unsigned long long)bal) - 1, l1 = 63 - __clzll((long long)bal);
      const uint32_t m0 = (uint32_t)__builtin_amdgcn_readlane((int)m, l0);
      const uint32_t m1 = (uint32_t)__builtin_amdgcn_readlane((int)m, l1);
      fh = 4u * (t * ROWT + wave * 64 + l0) + (uint32_t)(__ffs((int)m0) - 1);
      lh = 4u * (t * ROWT + wave * 64 + l1) + (uint32_t)(31 - __clz((int)m1)) + 1;
    }
    if (lane == 0) {
      s_fh[t][wave] = fh;
      s_lh[t][wave] = lh;
    }
  }
  uint64_t total_l, total_h;
  block_scan2_as<ROWT, T, false>(dl, dh, s_ex, sl, sh, total_l, total_h, wave_live);  // its barrier also publishes s_fh / s_lh
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const uint32_t pos = 4u * (t * ROWT + tid);
    if (!((wave_live >> t) & 1)) continue;  // slots beyond the row are never searched
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s_sl[pos + k] = sl[t][k];
      s_sh[pos + k] = sh[t][k];
    }
  }
  // next heavy after each quad: later lanes of the wave, later waves of the sub-tile, later sub-tiles
  uint32_t last_heavy = 0;
  uint32_t nh_after[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    // next quad of this wave that holds a heavy: first ballot bit above this lane
    const uint32_t m = (heavy >> (t * 4)) & 15u;
    const uint64_t above = hb_mask[t] & ~((2ull << lane) - 1);
    const int ln = above ? __ffsll((unsigned long long)above) - 1 : lane;
    const uint32_t mn = (uint32_t)__shfl((int)m, ln, 64);
    uint32_t nx = above ? 4u * (t * ROWT + wave * 64 + ln) + (uint32_t)(__ffs((int)mn) - 1) : NONE32;
#pragma unroll
    for (int wv = 0; wv < NW; ++wv) {
      if (wv > wave) nx = min(nx, s_fh[t][wv]);
#pragma unroll
      for (int t2 = t + 1; t2 < T; ++t2) nx = min(nx, s_fh[t2][wv]);
      last_heavy = max(last_heavy, s_lh[t][wv]);
    }
    nh_after[t] = nx;
  }
  __syncthreads();  // s_sl / s_sh are complete

  const uint64_t* a_l = s_sl + lead;
  const uint32_t off_l = lead * 8u, off_h = (CAP + lead) * 8u;  // byte offsets of the row inside smem
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const uint32_t pos = 4u * (t * ROWT + tid);
    if (pos >= span) continue;
    uint32_t arr[4];
    uint64_t key[4];
    uint32_t nh[4], oa[4], at[4];
    uint32_t nxt = nh_after[t];
#pragma unroll
    for (int k = 3; k >= 0; --k) {
      nh[k] = nxt;
      if ((heavy >> (t * 4 + k)) & 1) nxt = pos + k;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool hv = (heavy >> (t * 4 + k)) & 1;
      arr[k] = hv ? off_l : off_h;                          // a heavy looks for its retiring light in SL
      key[k] = hv ? sh[t][k] - 1 : sl[t][k] - dl[t][k];      // first SL >= y  <=>  first SL > y - 1
    }
    search4(smem, arr, key, d, at);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool hv = (heavy >> (t * 4 + k)) & 1;
      const uint32_t self = pos + k - lead;
      if (!hv) {
        oa[k] = at[k] < d ? at[k] : (last_heavy ? last_heavy - 1 - lead : self);
      } else if (nh[k] != NONE32 && at[k] < d) {
        op[t][k] = residual_prob(L.one + sh[t][k] - a_l[at[k]], L);
        oa[k] = nh[k] - lead;
      } else {
        oa[k] = self;  // op is already 1
      }
    }
    if (pos >= lead && pos + 4 <= span) {
      store_entries4(table + base + pos, op[t], oa);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if ((live >> (t * 4 + k)) & 1) {
          table[base + pos + k] = AliasEntry{op[t][k], oa[k]};
        }
    }
  }
}

// ---------------------------------------------------------------- one row per workgroup, pairing by merge (merge_row)
// MINW: wavefronts per SIMD the registers must leave room for; 3 where LDS (50 KB for 256 threads of 14 slots) allows no
// more anyway.  Rows of one class each, 30 M entries, lognormal(0, 2), TB/s of 12 bytes an entry, with integer sums, masks and moves
// of a thread's own slots, and as it is: 382..509 entries 2.57 and 3.26, 1022..1533 3.03 and 3.30, 2046..2557 2.70 and 3.34,
// 4606..5117 2.37 and 3.09; on the scale-26 graph, whose rows fill their classes, 2.97 and 4.18, 3.75 and 4.12 for the first two.
template <int ROWT, int PER, int MINW = 4>
__global__ __launch_bounds__(ROWT, MINW) void build_merge_kernel(const RowRef* __restrict__ vlist, const float* __restrict__ wgt,
                                                           AliasEntry* __restrict__ table, int8_t* __restrict__ valid) {
  extern __shared__ __align__(16) uint64_t smem[];
  __shared__ uint64_t s_aux[8 * (ROWT / 64)];
  const RowRef rr = vlist[blockIdx.x];
  const bool ok = merge_row<ROWT, PER>(rr, smem, s_aux, wgt, table);
  if (threadIdx.x == 0) valid[rr.v] = ok ? 1 : 0;
}

// ---------------------------------------------------------------- rows beyond LDS: global scratch
// 1024 threads stream one row three times: exact sum; prefix sums written to a scratch
// region private to the row (16 bytes per slot); searches over that scratch.
constexpr int HUGE_T = 1024;

__device__ __forceinline__ u128 block_sum_u128(u128 v, u128* s_tmp) {
  v = group_sum_u128<64>(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) s_tmp[wave] = v;
  __syncthreads();
  u128 r = s_tmp[0];
  for (int i = 1; i < HUGE_T / 64; ++i) r = add128(r, s_tmp[i]);
  return r;
}

__device__ __forceinline__ bool streaming_row(uint32_t off, uint32_t d, uint32_t max_tiles) {
  return ((off & 3u) + d + TILED_TILE - 1) / TILED_TILE > max_tiles;  // rows the tile-parallel path leaves alone
}

__global__ __launch_bounds__(HUGE_T) void build_huge_kernel(const RowRef* __restrict__ vlist, uint32_t count,
                                                            uint32_t max_tiles,
                                                            const uint64_t* __restrict__ scratch_off,
                                                            const uint32_t* __restrict__ xadj,
                                                            const float* __restrict__ wgt,
                                                            uint64_t* __restrict__ scratch,
                                                            AliasEntry* __restrict__ table,
                                                            int8_t* __restrict__ valid) {
  constexpr int NW = HUGE_T / 64;
  __shared__ u128 s_tmp[NW];
  __shared__ uint64_t s_wl[NW], s_wh[NW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (uint32_t r = blockIdx.x; r < count; r += gridDim.x) {
    const uint32_t v = vlist[r].v;
    const uint32_t off = xadj[v], d = xadj[v + 1] - off;
    if (!streaming_row(off, d, max_tiles)) continue;
    const float* wr = wgt + off;
    uint64_t* g_sl = scratch + 2 * scratch_off[r];
    uint64_t* g_sh = g_sl + d;

    u128 sum{0, 0};
    for (uint32_t i = tid; i < d; i += HUGE_T) sum = add128(sum, weight_fixed(clamp_weight(wr[i])));
    sum = block_sum_u128(sum, s_tmp);
    if ((sum.lo | sum.hi) == 0) {
      for (uint32_t i = tid; i < d; i += HUGE_T) {
        table[off + i] = AliasEntry{0.0f, SKY_INVALID};
      }
      if (tid == 0) valid[v] = 0;
      continue;
    }
    if (tid == 0) valid[v] = 1;
    const Ledger L = make_ledger(d, sum);

    uint64_t carry_l = 0, carry_h = 0;
    for (uint32_t tile = 0; tile < d; tile += HUGE_T) {
      const uint32_t i = tile + tid;
      uint64_t dl = 0, dh = 0;
      if (i < d) {
        const Entry e = classify(clamp_weight(wr[i]), L);
        if (e.heavy) dh = e.amount; else dl = e.amount;
      }
      const uint64_t il = group_scan_u64<64>(dl), ih = group_scan_sat_u64<64>(dh);
      __syncthreads();
      if (lane == 63) { s_wl[wave] = il; s_wh[wave] = ih; }
      __syncthreads();
      uint64_t bl = carry_l, bh = carry_h, tl = 0, th = 0;
      for (int k = 0; k < NW; ++k) {
        if (k == wave) { bl += tl; bh = add_sat(bh, th); }
        tl += s_wl[k];
        th = add_sat(th, s_wh[k]);
      }
      if (i < d) {
        g_sl[i] = bl + il;
        g_sh[i] = add_sat(bh, ih);
      }
      carry_l += tl;
      carry_h = add_sat(carry_h, th);
    }
    const uint64_t total_h = carry_h;
    __threadfence();
    __syncthreads();

    for (uint32_t i = tid; i < d; i += HUGE_T) {
      const Entry e = classify(clamp_weight(wr[i]), L);
      float op;
      uint32_t oa;
      if (!e.heavy) {
        const uint64_t x = g_sl[i] - e.amount;
        const uint32_t m = first_greater(g_sh, 0, d, x);
        op = (float)e.p;
        if (m < d) oa = m;
        else if (total_h) oa = first_greater(g_sh, 0, d, total_h - 1);
        else oa = i;
      } else {
        const uint64_t y = g_sh[i];
        const uint32_t nxt = first_greater(g_sh, i + 1, d, y);
        const uint32_t li = nxt < d ? first_greater(g_sl, 0, d, y - 1) : d;
        if (li < d) {
          op = residual_prob(L.one + y - g_sl[li], L);
          oa = nxt;
        } else {
          op = 1.0f;
          oa = i;
        }
      }
      table[off + i] = AliasEntry{op, oa};
    }
    __syncthreads();
  }
}

// Exclusive prefix sum of the degrees of the huge rows (a few thousand at most per launch of
// 1024 threads; longer lists are walked in chunks by the same block).
__global__ __launch_bounds__(1024) void huge_prefix_kernel(const RowRef* __restrict__ vlist, uint32_t count,
                                                           uint32_t max_tiles, const uint32_t* __restrict__ xadj,
                                                           uint64_t* __restrict__ scratch_off,
                                                           uint64_t* __restrict__ total) {
  __shared__ uint64_t s_w[16];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  uint64_t carry = 0;
  for (uint32_t chunk = 0; chunk < count; chunk += 1024) {
    const uint32_t r = chunk + tid;
    uint64_t d = 0;
    if (r < count) {
      const uint32_t v = vlist[r].v;
      d = xadj[v + 1] - xadj[v];
      if (!streaming_row(xadj[v], (uint32_t)d, max_tiles)) d = 0;
    }
    const uint64_t inc = group_scan_u64<64>(d);
    __syncthreads();
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    uint64_t b = carry, t = 0;
    for (int k = 0; k < 16; ++k) {
      if (k == wave) b += t;
      t += s_w[k];
    }
    if (r < count) scratch_off[r] = b + inc - d;
    carry += t;
  }
  if (tid == 0) *total = carry;
}

// ---------------------------------------------------------------- host driver
namespace {

constexpr size_t COUNTER_BYTES = 2 * CLS_COUNT * 4 + CLS_COUNT * 8;

struct BuildScratch {
  RowRef* vlist = nullptr;       // [vcap]
  uint32_t* counters = nullptr;  // [2*CLS_COUNT] class counts (the second half is unused), then CLS_COUNT 64-bit edge totals
  uint32_t* blk_cnt = nullptr;   // [BIN_BLOCKS * CLS_COUNT] class counts of every binning block, then their prefixes
  uint64_t* huge_off = nullptr;  // [huge_cap + 1], last = total
  uint64_t* huge_scratch = nullptr;
  uint32_t vcap = 0, huge_cap = 0;
  uint64_t huge_scratch_cap = 0;
};
bool g_lds_enabled = false;  // the kernels' LDS limits are raised once per process

template <class K>
int enable_big_lds(K kernel, size_t bytes) {
  SKY_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)bytes));
  return SKY_OK;
}

// The graph's build scratch, created on first use.
BuildScratch& scratch_of(sky_graph* g) {
  if (!g->build_scratch) g->build_scratch = new BuildScratch();
  return *static_cast<BuildScratch*>(g->build_scratch);
}

}  // namespace

void free_build_scratch(sky_graph* g) {
  if (!g->build_scratch) return;
  BuildScratch* sc = static_cast<BuildScratch*>(g->build_scratch);
  void* ptrs[] = {sc->vlist, sc->counters, sc->blk_cnt, sc->huge_off, sc->huge_scratch};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  delete sc;
  g->build_scratch = nullptr;
}

int buf_grow(sky_graph::PoolBuf* b, size_t bytes) {
  if (b->cap >= bytes && b->p) return SKY_OK;
  if (b->p) SKY_HIP(hipFree(b->p));
  b->p = nullptr;
  b->cap = 0;
  SKY_HIP(hipMalloc(&b->p, bytes + 16));
  b->cap = bytes;
  return SKY_OK;
}
int pool_get(sky_graph* g, int slot, size_t bytes, void** out) {
  SKY_TRY(buf_grow(&g->pool[slot], bytes));
  *out = g->pool[slot].p;
  return SKY_OK;
}
void pool_release(sky_graph* g) {
  for (auto& b : g->pool) {
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
  }
}

// The class kernels of one build are independent of one another once their lists are there: they go out over the graph's stream
// and three side streams (a class of few rows takes as long as one row, and the tail of one kernel is filled by another), and the
// graph's stream waits for the others at the end.  Not used when every kernel is timed on its own.
// (With events for the waits, and one stream for the classes of builds of 1 G entries and more / now, us: scale 26 with 8 edges a vertex
// 2,435 / 2,368, with 28 8,013 / 8,010, means of ten processes a side, of which those of the latter differ by 200; scale 23 with 40
// 1,535 / 1,495, scale 22 with 50 965 / 937, scale 24 with 16 1,235 / 1,230.  The streaming kernel in front of the merge kernels, the
// short rows behind them, or two streams instead of four: the same or up to 5 % slower.  Smaller builds, which come here by other
// knobs, in order / over four streams: 2.1 M entries in rows of up to 5,000 178 / 146, 4 M of up to 50,000 247 / 190, scale 20 with 6 207 / 177.)
constexpr uint64_t FAN_MIN_EDGES = 2000000;
struct StreamFan {
  Beside b;
  hipStream_t main;
  bool on = false;
  uint64_t load[SIDE_STREAMS + 1] = {0, 0, 0, 0};
  explicit StreamFan(hipStream_t m) : main(m) {}
  // One side stream, whatever start() does later; join() waits for it.
  int branch(int k, hipStream_t* out) {
    *out = main;
    if (!b.stream[k]) return SKY_OK;
    SKY_TRY(beside_fork(&b, k));
    *out = b.stream[k];
    return SKY_OK;
  }
  void start() { on = b.stream[0] != nullptr; }
  // The stream that carries the least work so far (`work`: the launch's entries, weighted by the caller where a
  // kernel is slow): a kernel queued behind a long one waits for it while other streams run dry.
  int next(uint64_t work, hipStream_t* out) {
    *out = main;
    if (!on) return SKY_OK;
    int k = 0;
    for (int i = 1; i <= SIDE_STREAMS; ++i)
      if (load[i] < load[k]) k = i;
    load[k] += work + 1;
    return k == SIDE_STREAMS ? SKY_OK : branch(k, out);
  }
  int join() {
    on = false;
    return beside_join(&b);
  }
  ~StreamFan() { beside_drop(&b); }  // after an error in between
};
// The graph's stream replaced for the duration of a call that takes it from the graph.
struct StreamSwap {
  sky_graph* g;
  hipStream_t saved;
  StreamSwap(sky_graph* g_, hipStream_t s) : g(g_), saved(g_->stream) { g->stream = s; }
  ~StreamSwap() { g->stream = saved; }
};

int EventTimer::mark(const char* name, uint64_t e) {
  hipEvent_t x;
  SKY_HIP(hipEventCreate(&x));
  SKY_HIP(hipEventRecord(x, stream));
  ev.push_back(x);
  names.push_back(name);
  edges.push_back(e);
  return SKY_OK;
}
int EventTimer::finish(std::vector<sky_graph::ProfileEntry>* profile, double* seconds) {
  SKY_HIP(hipStreamSynchronize(stream));
  SKY_HIP(hipGetLastError());
  profile->clear();
  for (size_t i = 1; i < ev.size(); ++i) {
    float ms = 0;
    SKY_HIP(hipEventElapsedTime(&ms, ev[i - 1], ev[i]));
    profile->push_back({names[i], ms, edges[i]});
  }
  float total_ms = 0;
  if (ev.size() >= 2) SKY_HIP(hipEventElapsedTime(&total_ms, ev.front(), ev.back()));
  if (seconds) *seconds = total_ms * 1e-3;
  return SKY_OK;
}
EventTimer::~EventTimer() {
  for (hipEvent_t e : ev) (void)hipEventDestroy(e);
}

int ensure_table_storage(sky_graph* g) {
  if (!g->table) SKY_TRY(alloc_padded(&g->table, (size_t)g->E));
  if (!g->valid) SKY_TRY(alloc_padded(&g->valid, (size_t)g->V));
  return SKY_OK;
}

int prepare_build_scratch(sky_graph* g, uint32_t max_rows) {
  BuildScratch& sc = scratch_of(g);
  if (sc.vcap < max_rows) {
    if (sc.vlist) SKY_HIP(hipFree(sc.vlist));
    sc.vlist = nullptr;
    sc.vcap = 0;
    SKY_HIP(hipMalloc((void**)&sc.vlist, (size_t)max_rows * sizeof(RowRef) + 16));
    sc.vcap = max_rows;
  }
  if (!sc.counters) SKY_HIP(hipMalloc((void**)&sc.counters, COUNTER_BYTES));
  if (!sc.blk_cnt) SKY_HIP(hipMalloc((void**)&sc.blk_cnt, (size_t)BIN_BLOCKS * CLS_COUNT * 4));
  if (!g_lds_enabled) {
    SKY_TRY(enable_big_lds(build_lds_kernel<512, 2>, 512 * 4 * 2 * 16));
    SKY_TRY(enable_big_lds(build_merge_kernel<512, 10>, (int)merge_lds_bytes(512, 10)));
    g_lds_enabled = true;
  }
  return SKY_OK;
}

// Largest build that goes out in the few launches of sky_build_fused.hip.  Above, a class fills the GPU by itself, and short
// rows beside the others in a kernel of their own are worth more than fewer launches.  (In few launches / by class, us, one after
// another and, in brackets, with the device waited for in between, which takes 35 us more where all side streams have had work: scale 22 with
// 16 edges a vertex 352 / 409, with 18 425 / 460, with 22 493 / 467 (507 / 522), with 31 652 / 647 (665 / 707), scale 20 with 120 763 / 749 (775 / 826), scale 21
// with 60 698 / 689 (710 / 749), scale 23 with 10 420 / 422, with 14 613 / 587 (627 / 641), scale 24 with 5 453 / 438 (486 / 491), with 7 626 / 696, 100 M
// entries in rows of up to 50,000 594 / 612, 110 M of up to 3,000 607 / 574 (621 / 613).)
constexpr uint64_t FUSED_MAX_ENTRIES = 1ull << 27;

// Whether a build leaves its rows of at most 32 entries to small_rows_kernel, which builds them where they lie,
// without lists.  Taken alone it is slower than the class kernels of these rows (1.39 against 1.12 ms on the
// scale-26 graph), but it depends on no list: on a side stream it runs beside the kernels of the long rows (it waits on
// memory, they on the vector ALU).  A build of all vertices then needs no binning either: the lists of the longer rows
// are in the graph's plan.  Every build of all vertices that is too large for few launches gains by that (R-MAT
// lognormal, by class / in place, us: scale 24 with 16 edges a vertex 1613 / 1535, with 56 5172 / 4888, scale 23 with 40
// 2069 / 1928, scale 22 with 66 1772 / 1668); a list of vertices has to be binned, and takes it from 2^25 rows on.
static bool small_rows_in_place(const sky_graph* g, const uint32_t* src, uint32_t n) {
  const long long sip = option(g, OPT_SMALL_IN_PLACE);
  return sip < 0 ? n >= (1u << 25) || (src == nullptr && n == g->V && g->E > FUSED_MAX_ENTRIES) : sip != 0;
}

// Builds the rows listed in `src` (device array of n vertex ids; null = vertices 0..n-1).
// prepare_build_scratch(n) (not needed for a build of all vertices with small_rows_in_place) and ensure_table_storage must have been called.
int build_rows(sky_graph* g, const uint32_t* src, uint32_t n, EventTimer* tm, CallDevice* call) {
  hipStream_t st = g->stream;
  g->has_walk_index = false;  // the table entries it was made from are about to change
  BuildScratch& sc = scratch_of(g);
  uint32_t counts[CLS_COUNT] = {0}, starts[CLS_COUNT] = {0};
  struct {
    uint32_t counts[2 * CLS_COUNT];
    unsigned long long edges[CLS_COUNT];
  } host = {};
  static_assert(sizeof(host) == COUNTER_BYTES, "counter block layout");
  const bool small_in_place = small_rows_in_place(g, src, n);
  const int listed_from = small_in_place ? CLS_G16 : CLS_G2;
  StreamFan fan(st);
  auto launch_small = [&](hipStream_t s) {
    const uint32_t per_wave = std::max(256u, std::min(SMALL_RANGE, n / 16384u / 64u * 64u));
    hipLaunchKernelGGL(small_rows_kernel, dim3((n + per_wave - 1) / per_wave), dim3(64), 0, s, g->xadj, g->adjwgt, src, n,
                       per_wave, g->table, g->valid);
  };
  // A build of all vertices that leaves the short rows where they lie takes the lists of the others from the graph's
  // plan: they depend on the row offsets alone, and binning 67 M vertices again took 0.35 ms.
  const bool all_rows = src == nullptr && n == g->V;
  const bool planned = all_rows && small_in_place && n > 0;
  if (planned) SKY_TRY(ensure_plan(g, &call));
  RowRef* vlist = planned ? g->plan->rows : sc.vlist;
  // clears the counters of the binning pass and, unless the plan's first kernel has, notes when the call began
  ForkMark fork{nullptr, 0};
  if (!tm && n > 0 && (small_in_place || std::min<uint64_t>(g->E, (uint64_t)n * g->max_degree) >= FAN_MIN_EDGES))
    SKY_TRY(beside_begin(g, &fan.b, &fork, SIDE_STREAMS));
  hipLaunchKernelGGL(build_begin_kernel, dim3(1), dim3(128), 0, st, sc.counters, (uint32_t)(COUNTER_BYTES / 4), call, fork);
  SKY_HIP(hipGetLastError());
  if (n > 0) {
    if (small_in_place && !tm) {
      hipStream_t side;
      SKY_TRY(fan.branch(SIDE_STREAMS - 1, &side));
      launch_small(side);
    }
    if (planned) {
      for (int c = 0; c < CLS_COUNT; ++c) {
        host.counts[c] = g->bin_counts[c];
        host.edges[c] = g->bin_edges[c];
      }
    } else {
      // The class sizes decide the launches that follow.
      const uint32_t per_block = bin_per_block(n), blocks = (n + per_block - 1) / per_block;
      hipLaunchKernelGGL(bin_count_kernel, dim3(blocks), dim3(256), 0, st, g->xadj, src, n, per_block, sc.blk_cnt,
                         reinterpret_cast<unsigned long long*>(sc.counters + 2 * CLS_COUNT));
      hipLaunchKernelGGL(bin_offsets_kernel, dim3(CLS_COUNT), dim3(256), 0, st, sc.blk_cnt, blocks, sc.counters);
      hipLaunchKernelGGL(bin_scatter_kernel, dim3(blocks), dim3(256), 0, st, g->xadj, g->adjwgt, src, n, per_block, listed_from,
                         sc.counters, sc.blk_cnt, sc.vlist, g->table, g->valid);
      SKY_HIP(hipMemcpyAsync(&host, sc.counters, COUNTER_BYTES, hipMemcpyDeviceToHost, st));
      SKY_HIP(hipStreamSynchronize(st));
    }
    for (int c = listed_from; c < CLS_COUNT; ++c) counts[c] = host.counts[c];
    uint32_t acc = 0;
    for (int c = 0; c < CLS_COUNT; ++c) {
      starts[c] = acc;
      acc += counts[c];
    }
  }
  const uint64_t small_edges = host.edges[CLS_TINY] + host.edges[CLS_G2] + host.edges[CLS_G4] + host.edges[CLS_G8];
  if (tm) SKY_TRY(tm->mark("bin", small_in_place ? 0 : host.edges[CLS_TINY]));
  if (tm && small_in_place && n > 0) {
    launch_small(st);
    SKY_TRY(tm->mark("small", small_edges));
  }
  uint64_t call_edges = 0;
  for (int c = 0; c < CLS_COUNT; ++c) call_edges += host.edges[c];
  if (!tm && option(g, OPT_BUILD_STREAMS) && call_edges >= FAN_MIN_EDGES) fan.start();

  auto grp = [&](int cls, auto kernel, int G, const char* name) -> int {
    const uint32_t cnt = counts[cls];
    if (cnt) {
      const uint32_t per_block = 256 / G;
      hipStream_t on;
      SKY_TRY(fan.next(host.edges[cls], &on));
      hipLaunchKernelGGL(kernel, dim3((cnt + per_block - 1) / per_block), dim3(256), 0, on, vlist + starts[cls],
                         cnt, g->adjwgt, g->table, g->valid);
    }
    return (tm && cnt) ? tm->mark(name, host.edges[cls]) : SKY_OK;  // no bracket for an empty class
  };
  const bool row_merge = option(g, OPT_ROW_MERGE) != 0;
  // Rows of 8190..STREAM_MAX_DEG entries: one workgroup streams a row.  A small streaming class is not worth its
  // own launch (too few workgroups to fill the GPU): its rows then go to the tile-parallel path together with the
  // HUGE class.  The rows above 65533 entries keep one workgroup busy for up to 1.5 ms; they join the launch (and
  // start first) only when it holds enough other rows to run that long anyway, else they are built tile by tile.
  // The lists lie back to back: STREAM_LAST, STREAM, STREAM_WIDE, HUGE.
  const uint32_t narrow_rows = counts[CLS_STREAM] + counts[CLS_STREAM_LAST];
  const uint64_t narrow_edges = host.edges[CLS_STREAM] + host.edges[CLS_STREAM_LAST];
  const uint64_t all_stream_edges = narrow_edges + host.edges[CLS_STREAM_WIDE];
  const bool stream_to_tiled = !row_merge || all_stream_edges <= (uint64_t)option(g, OPT_STREAM_MIN_EDGES);
  const bool wide_streamed = !stream_to_tiled && all_stream_edges >= (uint64_t)option(g, OPT_STREAM_WIDE_MIN_EDGES);
  const uint32_t wide_rows = wide_streamed ? counts[CLS_STREAM_WIDE] : 0;
  auto lds = [&](int cls, auto kernel, int rowt, int t, const char* name) -> int {
    const uint32_t cnt = counts[cls];
    if (cnt) {
      const size_t bytes = (size_t)rowt * 4 * t * 16;
      hipStream_t on;
      SKY_TRY(fan.next(host.edges[cls], &on));
      hipLaunchKernelGGL(kernel, dim3(cnt), dim3(rowt), bytes, on, vlist + starts[cls], g->xadj, g->adjwgt,
                         g->table, g->valid);
    }
    return (tm && cnt) ? tm->mark(name, host.edges[cls]) : SKY_OK;  // no bracket for an empty class
  };
  auto mrg = [&](int cls, auto kernel, int rowt, int per, const char* name) -> int {
    const uint32_t cnt = counts[cls];
    if (cnt) {
      const size_t bytes = merge_lds_bytes(rowt, per);
      hipStream_t on;
      SKY_TRY(fan.next(host.edges[cls], &on));
      hipLaunchKernelGGL(kernel, dim3(cnt), dim3(rowt), bytes, on, vlist + starts[cls],
                         g->adjwgt, g->table, g->valid);
    }
    return (tm && cnt) ? tm->mark(name, host.edges[cls]) : SKY_OK;  // no bracket for an empty class
  };
  static const char* const mw_name[9] = {"mw2", "mw3", "mw4", "mw5", "mw6", "mw7", "mw8", "mw9", "mw10"};
  if (row_merge) {
    SKY_TRY(mrg(CLS_LDS_W1, build_merge_kernel<64, 4>, 64, 4, "lds_w1"));
    SKY_TRY(mrg(CLS_LDS_W6, build_merge_kernel<64, 6>, 64, 6, "lds_w6"));
    SKY_TRY(mrg(CLS_LDS_W2, build_merge_kernel<64, 8>, 64, 8, "lds_w2"));
    SKY_TRY(mrg(CLS_MW2_6, build_merge_kernel<128, 6>, 128, 6, "mw2_6"));
#define SKY_MW(NW) SKY_TRY(mrg(CLS_MW2 + NW - 2, build_merge_kernel<64 * NW, 8>, 64 * NW, 8, mw_name[NW - 2]))
    // Class nw holds rows that fit 512 nw slots.  Where a shape with an even number of slots per thread and a
    // multiple of 4 wavefronts covers that span exactly, it is used instead of nw wavefronts of 8 slots: every
    // SIMD of the CU then carries the same number of a workgroup's wavefronts.  768 threads of 6 slots, which would cover
    // nw = 9, need 86 registers: one workgroup per CU, 1.69 TB/s where 512 threads of 10 slots reach 2.85.
    SKY_MW(2);
    SKY_TRY(mrg(CLS_MW2 + 1, build_merge_kernel<256, 6>, 256, 6, mw_name[1]));
    SKY_MW(4);
    SKY_TRY(mrg(CLS_MW2 + 3, build_merge_kernel<256, 10>, 256, 10, mw_name[3]));
    SKY_TRY(mrg(CLS_MW2 + 4, build_merge_kernel<512, 6>, 512, 6, mw_name[4]));
    SKY_TRY(mrg(CLS_MW2 + 5, (build_merge_kernel<256, 14, 3>), 256, 14, mw_name[5]));
    SKY_MW(8);
    SKY_TRY(mrg(CLS_MW2 + 7, build_merge_kernel<512, 10>, 512, 10, mw_name[7]));
    SKY_TRY(mrg(CLS_MW2 + 8, build_merge_kernel<512, 10>, 512, 10, mw_name[8]));
#undef SKY_MW
  } else {
    SKY_TRY(lds(CLS_LDS_W1, build_lds_kernel<64, 1>, 64, 1, "lds_w1"));
    SKY_TRY(lds(CLS_LDS_W6, build_lds_kernel<64, 2>, 64, 2, "lds_w6"));
    SKY_TRY(lds(CLS_LDS_W2, build_lds_kernel<64, 2>, 64, 2, "lds_w2"));
    SKY_TRY(lds(CLS_MW2_6, build_lds_kernel<128, 2>, 128, 2, "mw2_6"));
    for (int nw = 2; nw <= MERGE_MAX_NW; ++nw) {
      const int cls = CLS_MW2 + nw - 2;
      if (nw <= 2) SKY_TRY(lds(cls, build_lds_kernel<128, 2>, 128, 2, mw_name[nw - 2]));
      else if (nw <= 4) SKY_TRY(lds(cls, build_lds_kernel<256, 2>, 256, 2, mw_name[nw - 2]));
      else if (nw <= 8) SKY_TRY(lds(cls, build_lds_kernel<512, 2>, 512, 2, mw_name[nw - 2]));
      else {  // this variant has no kernel for rows of 4094..5117 entries: tile-parallel path
        if (counts[cls]) {
          uint32_t skipped = 0;
          SKY_TRY(fan.join());  // the tile-parallel path's scratch serves one call at a time
          SKY_TRY(build_rows_tiled(g, vlist + starts[cls], counts[cls], &skipped, nullptr, 0));
          if (skipped) return fail(SKY_ERR_STATE, "tiled_max_tiles below 9 needs row_merge");
        }
        if (tm) SKY_TRY(tm->mark(mw_name[nw - 2], host.edges[cls]));
      }
    }
  }

  // After the merge kernels: two workgroups of it fill a CU's LDS, so nothing of small_rows_kernel would run beside it on a CU
  // (scale 26 8.25 -> 8.18 ms, scale 25 with 56 edges a vertex 8.8 -> 8.6); last of all, its longest rows would have no company.
  if (!stream_to_tiled && narrow_rows + wide_rows) {
    // the streaming kernel takes three times as long for an entry as the others when it shares the GPU with them
    hipStream_t on;
    SKY_TRY(fan.next(3 * (narrow_edges + (wide_streamed ? host.edges[CLS_STREAM_WIDE] : 0)), &on));
    StreamSwap sw(g, on);
    SKY_TRY(build_rows_stream(g, vlist + starts[CLS_STREAM_WIDE], wide_rows, vlist + starts[CLS_STREAM_LAST], narrow_rows));
    if (tm) SKY_TRY(tm->mark("stream", narrow_edges + (wide_streamed ? host.edges[CLS_STREAM_WIDE] : 0)));
  }
  // Rows of 5118..8189 entries: one workgroup holds the row (without row_merge they are built tile by tile).
  if (row_merge && counts[CLS_HOLD]) {
    {
      hipStream_t on;
      SKY_TRY(fan.next(2 * host.edges[CLS_HOLD], &on));
      StreamSwap sw(g, on);
      SKY_TRY(build_rows_hold(g, vlist + starts[CLS_HOLD], counts[CLS_HOLD]));
    }
    if (tm) SKY_TRY(tm->mark("hold", host.edges[CLS_HOLD]));
  }
  SKY_TRY(grp(CLS_G2, build_group_kernel<SHAPE_G2.lanes, SHAPE_G2.per>, SHAPE_G2.lanes, "g2"));
  SKY_TRY(grp(CLS_G4, build_group_kernel<SHAPE_G4.lanes, SHAPE_G4.per>, SHAPE_G4.lanes, "g4"));
  SKY_TRY(grp(CLS_G8, build_group_kernel<SHAPE_G8.lanes, SHAPE_G8.per>, SHAPE_G8.lanes, "g8"));
  SKY_TRY(grp(CLS_G16, build_group_kernel<SHAPE_G16.lanes, SHAPE_G16.per>, SHAPE_G16.lanes, "g16"));
  SKY_TRY(grp(CLS_G32, build_group_kernel<SHAPE_G32.lanes, SHAPE_G32.per>, SHAPE_G32.lanes, "g32"));
  SKY_TRY(grp(CLS_G32S, build_group_kernel<SHAPE_G32S.lanes, SHAPE_G32S.per>, SHAPE_G32S.lanes, "g32s"));
  SKY_TRY(grp(CLS_G32X, build_group_kernel<SHAPE_G32X.lanes, SHAPE_G32X.per>, SHAPE_G32X.lanes, "g32x"));

  // the lists HOLD, STREAM_LAST, STREAM, STREAM_WIDE, HUGE lie back to back (the class numbers between are unused)
  const uint32_t held_rows = row_merge ? 0 : counts[CLS_HOLD];
  const uint32_t tiled_rows =
      counts[CLS_HUGE] + (wide_streamed ? 0 : counts[CLS_STREAM_WIDE]) + (stream_to_tiled ? narrow_rows : 0) + held_rows;
  const uint64_t tiled_edges = host.edges[CLS_HUGE] + (wide_streamed ? 0 : host.edges[CLS_STREAM_WIDE]) +
                               (stream_to_tiled ? narrow_edges : 0) +
                               (row_merge ? 0 : host.edges[CLS_HOLD]);
  const RowRef* tiled_list =
      vlist + (held_rows ? starts[CLS_HOLD]
                         : stream_to_tiled ? starts[CLS_STREAM_LAST] : (wide_streamed ? starts[CLS_HUGE] : starts[CLS_STREAM_WIDE]));
  if (tiled_rows) {
    const uint32_t cnt = tiled_rows;
    uint32_t skipped = 0;
    {
      hipStream_t on;
      SKY_TRY(fan.next(2 * tiled_edges, &on));
      StreamSwap sw(g, on);
      SKY_TRY(build_rows_tiled(g, tiled_list, cnt, &skipped, tm, tiled_edges));
    }
    SKY_TRY(fan.join());
    if (skipped) {  // rows with more tiles than the tile-parallel path takes: one workgroup streams each
      const uint32_t max_tiles = tiled_max_tiles(g);
      if (sc.huge_cap < cnt) {
        if (sc.huge_off) SKY_HIP(hipFree(sc.huge_off));
        sc.huge_off = nullptr;
        sc.huge_cap = 0;
        SKY_HIP(hipMalloc((void**)&sc.huge_off, ((size_t)cnt + 1) * 8));
        sc.huge_cap = cnt;
      }
      hipLaunchKernelGGL(huge_prefix_kernel, dim3(1), dim3(1024), 0, st, tiled_list, cnt, max_tiles,
                         g->xadj, sc.huge_off, sc.huge_off + cnt);
      uint64_t total = 0;
      SKY_HIP(hipMemcpyAsync(&total, sc.huge_off + cnt, 8, hipMemcpyDeviceToHost, st));
      SKY_HIP(hipStreamSynchronize(st));
      if (sc.huge_scratch_cap < total) {
        if (sc.huge_scratch) SKY_HIP(hipFree(sc.huge_scratch));
        sc.huge_scratch = nullptr;
        sc.huge_scratch_cap = 0;
        SKY_HIP(hipMalloc((void**)&sc.huge_scratch, total * 16));
        sc.huge_scratch_cap = total;
      }
      hipLaunchKernelGGL(build_huge_kernel, dim3(std::min<uint32_t>(cnt, 512)), dim3(HUGE_T), 0, st,
                         tiled_list, cnt, max_tiles, sc.huge_off, g->xadj, g->adjwgt, sc.huge_scratch,
                         g->table, g->valid);
      if (tm) SKY_TRY(tm->mark("streamed", 0));
    }
  }
  return fan.join();
}

int bin_all_rows(sky_graph* g, int listed_from, RowRef** rows, uint32_t* start, CallDevice** first) {
  hipStream_t st = g->stream;
  SKY_TRY(ensure_table_storage(g));
  SKY_TRY(prepare_build_scratch(g, 0));
  BuildScratch& sc = scratch_of(g);
  struct {
    uint32_t counts[2 * CLS_COUNT];
    unsigned long long edges[CLS_COUNT];
  } host = {};
  const uint32_t n = g->V, per_block = bin_per_block(n), blocks = n ? (n + per_block - 1) / per_block : 0;
  if (n) {
    hipLaunchKernelGGL(build_begin_kernel, dim3(1), dim3(128), 0, st, sc.counters, (uint32_t)(COUNTER_BYTES / 4),
                       *first, ForkMark{nullptr, 0});
    *first = nullptr;
    hipLaunchKernelGGL(bin_count_kernel, dim3(blocks), dim3(256), 0, st, g->xadj, (const uint32_t*)nullptr, n, per_block,
                       sc.blk_cnt, reinterpret_cast<unsigned long long*>(sc.counters + 2 * CLS_COUNT));
    hipLaunchKernelGGL(bin_offsets_kernel, dim3(CLS_COUNT), dim3(256), 0, st, sc.blk_cnt, blocks, sc.counters);
    SKY_HIP(hipMemcpyAsync(&host, sc.counters, COUNTER_BYTES, hipMemcpyDeviceToHost, st));
    SKY_HIP(hipStreamSynchronize(st));
  }
  size_t listed = 0;
  for (int c = 0; c < CLS_COUNT; ++c) {
    g->bin_counts[c] = host.counts[c];
    g->bin_edges[c] = host.edges[c];
    start[c] = (uint32_t)listed;
    if (c >= listed_from) listed += host.counts[c];
  }
  SKY_HIP(hipMalloc((void**)rows, listed * sizeof(RowRef) + 16));
  if (listed)
    hipLaunchKernelGGL(bin_scatter_kernel, dim3(blocks), dim3(256), 0, st, g->xadj, g->adjwgt, (const uint32_t*)nullptr, n, per_block,
                       listed_from, sc.counters, sc.blk_cnt, *rows, g->table, g->valid);
  SKY_HIP(hipGetLastError());
  return SKY_OK;
}

int build_all_tables(sky_graph* g, double* seconds) {
  SKY_TRY(ensure_table_storage(g));
  // Knobs that name kernels of their own, and per-kernel timing, want the class kernels.
  const bool fused = fused_possible(g) && !option(g, OPT_BUILD_PROFILE) && option(g, OPT_SMALL_IN_PLACE) < 0 &&
                     option(g, OPT_BUILD_STREAMS) != 0 && g->E <= FUSED_MAX_ENTRIES && g->V;
  if (fused) {
    CallDevice* call = nullptr;
    double sec = 0;
    SKY_TRY(call_begin(g, &call));
    SKY_TRY(ensure_plan(g, &call));
    SKY_TRY(build_all_fused(g, call));
    SKY_TRY(call_end(g, nullptr, &sec));
    g->build_profile.assign(1, {"build", (float)(sec * 1e3), g->E});
    if (seconds) *seconds = sec;
    g->has_tables = true;
    return SKY_OK;
  }
  SKY_TRY(prepare_build_scratch(g, small_rows_in_place(g, nullptr, g->V) ? 0 : g->V));
  if (option(g, OPT_BUILD_PROFILE)) {
    EventTimer tm(g->stream);
    SKY_TRY(tm.mark("start", 0));
    SKY_TRY(build_rows(g, nullptr, g->V, &tm));
    SKY_TRY(tm.finish(&g->build_profile, seconds));
  } else {  // no event between the kernels
    CallDevice* call = nullptr;
    double sec = 0;
    SKY_TRY(call_begin(g, &call));
    SKY_TRY(build_rows(g, nullptr, g->V, nullptr, call));
    SKY_TRY(call_end(g, nullptr, &sec));
    g->build_profile.assign(1, {"build", (float)(sec * 1e3), g->E});
    if (seconds) *seconds = sec;
  }
  g->has_tables = true;
  return SKY_OK;
}

}  // namespace sky
