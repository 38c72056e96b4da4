// Builds whose launches, not their entries, would bound them: from a graph of a thousand edges up to FUSED_MAX_ENTRIES, and
// the rows of a frontier.
//
// The class kernels of sky_build.hip give every degree class a launch of its own.  That is right where a class fills
// the GPU for a millisecond; a build of 17 M entries spent 220 us on 27 launches of 5 to 25 us each, 2.4 us apart on
// the host and each with a tail of its own, and spreading them over four streams costs 30 us for the fork and the
// join by events alone.  Here one launch takes all classes whose rows need the same number of threads, and the passes of the
// rows that are built tile by tile, which depend on one another, ride along in the same launches:
//
//   fused_wave_kernel    64 threads    rows of up to 509 entries         tile sums
//   fused_pair_kernel    128 threads   rows of 510..1021                 row sums -> ledger, tile totals
//   fused_wide_kernel    512 threads   rows of 2558 and more             scan over a row's tiles
//   fused_block_kernel   256 threads   rows of 1022..2557                entries of the tiles
//   fused_mid_kernel     512 threads   rows of 2558..5117, where a fork (below) gives them a launch of their own
//
// A launch whose classes are empty is left out.  A small build with rows for more than the first of them, and none for tiles, goes
// out in one launch of 512 threads instead (fused_all_kernel).  Every row builder is the one the class kernels call, so the
// tables are the same bits.  The lists of rows by class and the geometry of the tiles depend on the row offsets alone:
// they are made by the first build of a graph and kept with it.
//
// Only the passes over tiles depend on one another.  In a whole build the sweep over the rows of up to 32 entries, and behind it the rows
// of 2558 and more, go out beside the rest (Beside, sky_call.h), so that the tails of four launches no longer follow one another.
// (In order / beside, us, three graphs in turn: scale 16 with 16 edges a vertex 46 / 42, scale 20 with 16 131 / 120, with 6 96 / 82, with 3
// 69 / 54, scale 23 with 4 253 / 233, with 10 437 / 433, 3 M entries in rows of up to 20,000 70 / 58, 40 M in rows of up to 300,007 331 / 319.
// Where the launches that follow one another fill the GPU the tails no longer count: BESIDE_MERGED.  On one graph again and again, with
// the long rows in front of the sweep scale 23 with 10 483 instead of 430; those on a third stream scale 20 with 6 69 instead of 82, with 16 110
// instead of 104, scale 16 with 16 45 instead of 42; rows of up to 107 entries alone, one launch in order, 128 / 138.)  The
// workgroups of a large frontier's launches stay until all units are done and leave no room beside them: those follow one another.  (The
// second hop of 40,000 seeds on the scale-22 graph with 32 edges a vertex takes 10 to 90 us longer beside one another.)
#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "sky_build_fused.h"
#include "sky_build_rules.h"
#include "sky_build_long.h"
#include "sky_build_rows.h"
#include "sky_build_tile.h"

namespace sky {

// What a unit of a launch's work is.
enum Section : uint32_t {
  SEC_SWEEP,  // 64 threads: a range of vertices, all their rows of at most 32 entries
  SEC_TINY,   //             64 listed rows of 1..2 entries
  SEC_G2, SEC_G4, SEC_G8, SEC_G16, SEC_G32, SEC_G32S, SEC_G32X, SEC_W1, SEC_W6, SEC_W2,
  SEC_SUM,    //             the sum of a tile
  SEC_P6, SEC_P8,                              // 128 threads
  SEC_TOTALS,                                  //             two tiles
  SEC_STREAM, SEC_B6, SEC_B8, SEC_B10,  // 512 threads
  SEC_SCAN,                                    //             a row's tiles
  SEC_M6, SEC_M8, SEC_M10, SEC_M14,            // 256 threads
  SEC_EMIT                                     //             a tile
};
struct SectionRef {
  uint32_t kind;
  uint32_t units;    // host-sized: units of this section; device-sized: not used
  uint32_t per;      // rows per unit
  uint32_t start;    // first row in the list
  int cls0, ncls;    // device-sized: classes whose rows lie back to back from `start` on
  uint32_t stride;   // device-sized: distance between the segments of consecutive classes
};
constexpr int MAX_SECTIONS = 14;
struct FusedArgs {
  const RowRef* list;
  const uint32_t* counts;  // device-sized: rows of every class (null: host-sized)
  const uint32_t* xadj;
  const float* wgt;
  AliasEntry* table;
  int8_t* valid;
  uint32_t V, per_wave;  // SEC_SWEEP
  bool split;            // a wavefront for every class of a range's rows, four that follow one another (SPLIT_SWEEP)
  // rows built tile by tile
  TiledRow* trows;
  const TileGeom* geom;
  u128* tsum;
  TileTotals* ttot;
  uint64_t *BL, *BH;
  uint32_t* nfh;
  uint4* ranges;
  const uint32_t* bitmap;  // frontier: bit set for every vertex whose row has been asked for (null: every row is built)
  uint32_t bit_mask;       // of the bitmap (frontier_bit)
  uint32_t* built;         // frontier: by row of trows, the hop (from 1 on) whose build in the same call has made it
  uint32_t hop;            // this one
  uint32_t* next;          // frontier: units of the wide launch that are taken, 0 at first (null: every grid-th for each workgroup)
  uint32_t tile0, trow0;  // first tile and row of those this build makes tile by tile
  bool ledgers_done;
  CallDevice* call;  // the call's first launch notes when it began
  ForkMark fork;     // and the first of a fork that it runs
  uint32_t nsec;
  uint32_t first[MAX_SECTIONS];  // host-sized: first unit of every section, 2^32 - 1 past the last
  SectionRef sec[MAX_SECTIONS];
};

// The section and the unit inside it that unit u of the launch is; false past the end.  Host-sized launches have
// one workgroup per unit and the sections' first units in their arguments; device-sized ones find out how many units
// each section has, section i in lane i of every wavefront, once per workgroup.
template <bool DEV>
struct UnitFinder;
template <>
struct UnitFinder<false> {
  __device__ __forceinline__ explicit UnitFinder(const FusedArgs&) {}
  __device__ __forceinline__ bool find(const FusedArgs& a, uint32_t u, SectionRef& s, uint32_t& unit, uint32_t& rows) const {
    uint32_t k = 0, first = 0;
#pragma unroll
    for (int i = 1; i < MAX_SECTIONS; ++i)
      if (u >= a.first[i]) {
        k = i;
        first = a.first[i];
      }
    s = a.sec[k];
    unit = u - first;
    rows = 0;
    return true;
  }
};
template <>
struct UnitFinder<true> {
  uint32_t incl, rows_of;
  __device__ __forceinline__ explicit UnitFinder(const FusedArgs& a) {
    const uint32_t lane = threadIdx.x & 63;
    uint32_t n = 0;
    rows_of = 0;
    if (lane < a.nsec) {
      const SectionRef s = a.sec[lane];
      n = s.units;
      if (s.cls0 >= 0) {
        for (int c = 0; c < s.ncls; ++c) rows_of += a.counts[s.cls0 + c];
        n = (rows_of + s.per - 1) / s.per;
      }
    }
    incl = group_scan_u32<16>(n);
  }
  __device__ __forceinline__ bool find(const FusedArgs& a, uint32_t u, SectionRef& s, uint32_t& unit, uint32_t& rows) const {
    const unsigned long long m = __ballot(u < incl) & ((1ull << MAX_SECTIONS) - 1ull);
    if (!m) return false;
    const int k = __ffsll((long long)m) - 1;
    s = a.sec[k];
    unit = u - (k ? (uint32_t)__builtin_amdgcn_readlane((int)incl, k - 1) : 0u);
    rows = (uint32_t)__builtin_amdgcn_readlane((int)rows_of, k);
    return true;
  }
};
// The next unit that no workgroup of the launch has.
__device__ __forceinline__ uint32_t next_unit(uint32_t* taken) {
  __shared__ uint32_t s_unit;
  __syncthreads();  // the unit before is done with LDS, and s_unit has been read
  if (threadIdx.x == 0) s_unit = gridDim.x + atomicAdd(taken, 1u);
  __syncthreads();
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)s_unit);
}
// Row `i` of a section (host-sized: `rows` holds none, the section's last unit may be partly empty).
template <bool DEV>
__device__ __forceinline__ bool row_at(const FusedArgs& a, const SectionRef& s, uint32_t i, uint32_t rows, RowRef& rr) {
  rr = RowRef{0, 0, 0, 0};
  if (!DEV) {
    if (i >= s.stride) return false;  // host-sized: stride holds the number of rows
    rr = a.list[s.start + i];
    return true;
  }
  if (i >= rows) return false;
  uint32_t at = s.start;
  for (int c = 0; c + 1 < s.ncls; ++c) {
    const uint32_t n = a.counts[s.cls0 + c];
    if (i < n) break;
    i -= n;
    at += s.stride;
  }
  rr = a.list[at + i];
  return true;
}

// Units first, first + stride, ... below n that are wanted, by a workgroup (each wavefront of it looks for itself and finds the same), 64
// of them looked at together, a lane each.  A build of a frontier passes over the tiles of every long row of the graph, of which it
// makes few: one after another that is a chain of two to four dependent loads for each (28,500 tiles of the scale-22 graph with 32
// edges a vertex, 43 us of a launch of 1,024 workgroups).
template <class Wanted, class Work>
__device__ __forceinline__ void each_wanted(uint32_t n, uint32_t first, uint32_t stride, Wanted wanted, Work work) {
  for (uint32_t u0 = first; u0 < n; u0 += 64u * stride) {
    const uint32_t u = u0 + (threadIdx.x & 63) * stride;
    for (unsigned long long m = __ballot(u < n && wanted(u)); m; m &= m - 1ull) work(u0 + ((uint32_t)__ffsll((long long)m) - 1u) * stride);
  }
}
// The first unit from n on for a workgroup of a device-sized launch, which has units of the n in front too; one of the others has one unit.
template <bool DEV>
__device__ __forceinline__ uint32_t unit_behind(uint32_t n) {
  return DEV ? first_behind(n, blockIdx.x, gridDim.x) : blockIdx.x;
}
// Whether the tile belongs to a row that the frontier asks for; its first tile says so to the passes behind.
__device__ __forceinline__ bool tile_asked(const FusedArgs& a, uint32_t tile) {
  const TileGeom tg = a.geom[tile];
  if (tg.span == 0) return false;  // there are fewer tiles than their bound
  const uint32_t b = frontier_bit(a.trows[tg.row].v, a.bit_mask);
  const uint32_t made = a.built[tg.row];
  const bool active = ((a.bitmap[b >> 5] >> (b & 31)) & 1u) && (made == 0 || made == a.hop);  // a hop may be built once more
  if (tg.T == 0) a.trows[tg.row].active = active ? 1u : 0u;
  return active;
}
__device__ __forceinline__ bool tile_active(const FusedArgs& a, uint32_t tile) {
  const TileGeom tg = a.geom[tile];
  return tg.span != 0 && a.trows[tg.row].active;
}

// The exact sum of tile `tile` by a wavefront: 16 slots per lane.
__device__ __forceinline__ void tile_sum_wave(const FusedArgs& a, uint32_t tile) {
  const uint32_t lane = threadIdx.x & 63;
  const TileGeom tg = a.geom[tile];
  if (tg.span == 0) return;
  float4 x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t pos = tg.T * TILE + 256u * k + 4u * lane;
    x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pos < tg.span) x[k] = *reinterpret_cast<const float4*>(a.wgt + tg.base + pos);
  }
  WSum3 sum{0.0, 0.0, 0.0};  // exact: a tile adds at most 1024 limbs below 2^32 + 1
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float xs[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t idx = tg.T * TILE + 256u * k + 4u * lane + j;
      wsum3_add(sum, (double)masked_weight(xs[j], idx - tg.lead < tg.span - tg.lead));
    }
  }
  sum = group_sum_wsum3<64>(sum);
  if (lane == 0) a.tsum[tile] = wsum3_to_u128(sum);
}

// Row sum -> ledger, and the totals of one tile, by a wavefront.  Every tile of a row adds up its row's tile sums, which
// spares a launch in between; where a row has so many that this would take long (LEDGER_TILES) there is that launch.
__device__ __forceinline__ void tile_totals_wave(const FusedArgs& a, uint32_t tile) {
  const uint32_t lane = threadIdx.x & 63;
  const TileGeom tg = a.geom[tile];
  if (tg.span == 0) return;
  TiledRow* row = a.trows + tg.row;
  float4 x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t pos = tg.T * TILE + 256u * k + 4u * lane;
    x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pos < tg.span) x[k] = *reinterpret_cast<const float4*>(a.wgt + tg.base + pos);
  }
  bool ok;
  Ledger L = {0.0, 0.0, 0.0, 0};
  if (a.ledgers_done) {
    ok = row->ok;
    L = row_ledger(*row);
  } else {
    u128 sum{0, 0};
    const uint32_t t0 = row->tile0, nt = row->ntiles;
    for (uint32_t t = lane; t < nt; t += 64) sum = add128(sum, a.tsum[t0 + t]);
    sum = group_sum_u128<64>(sum);
    ok = (sum.lo | sum.hi) != 0;
    if (ok) L = make_ledger(row->d, sum);
    if (tg.T == 0 && lane == 0) {
      row->ok = ok;
      row->scale = L.scale;
      row->fs = L.fs;
      row->inv_fs = L.inv_fs;
      row->one = L.one;
    }
  }
  if (!ok) return;
  auto totals = [&](auto may_wrap) {
    constexpr bool SAT = decltype(may_wrap)::value;
    uint64_t sd = 0, su = 0;
    uint32_t fh = NONE32, lh = 0;  // lh holds idx + 1 so that 0 means none
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float xs[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t idx = tg.T * TILE + 256u * k + 4u * lane + j;
        const bool in = idx - tg.lead < tg.span - tg.lead;
        const Entry e = classify_fast((double)masked_weight(xs[j], in), in, L);
        if (!in) continue;
        if (e.heavy) {
          su = add_sat<SAT>(su, e.amount);
          fh = min(fh, idx);
          lh = max(lh, idx + 1);
        } else {
          sd += e.amount;
        }
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      sd += shfl_xor_u64(sd, m);
      su = add_sat<SAT>(su, shfl_xor_u64(su, m));
      fh = min(fh, (uint32_t)__shfl_xor((int)fh, m, 64));
      lh = max(lh, (uint32_t)__shfl_xor((int)lh, m, 64));
    }
    if (lane == 0) a.ttot[tile] = TileTotals{sd, su, fh, lh ? lh - 1 : NONE32};
  };
  if (surpluses_may_wrap(L.scale)) totals(std::true_type{});
  else totals(std::false_type{});
}

__device__ __forceinline__ void sweep_unit(const FusedArgs& a, uint32_t unit, uint64_t* smem) {
  const uint32_t range = a.split ? unit / 4 : spread_units(unit, (a.V + a.per_wave - 1) / a.per_wave);
  small_rows_range(range * a.per_wave, a.xadj, a.wgt, nullptr, a.V, a.per_wave, a.table, a.valid, smem,
                   a.split ? 1u << (unit % 4) : 15u);
}

template <bool DEV, int G, int PER>
__device__ __forceinline__ void group_unit(const FusedArgs& a, const SectionRef& s, uint32_t unit, uint32_t rows,
                                           uint64_t* smem) {
  uint32_t t = threadIdx.x & 63;
  asm volatile("" : "+v"(t));  // what depends on the lane number stays inside this unit's code
  RowRef rr;
  const bool have = row_at<DEV>(a, s, unit * (64 / G) + t / G, rows, rr);
  const bool ok = group_build_row<G, PER, 64>(rr.off, rr.d, a.wgt, a.table, smem, t);
  if (have && (t & (G - 1)) == 0) a.valid[rr.v] = ok ? 1 : 0;
}
template <bool DEV, int ROWT, int PER>
__device__ __forceinline__ void merge_unit(const FusedArgs& a, const SectionRef& s, uint32_t unit, uint32_t rows,
                                           uint64_t* smem, uint64_t* s_aux) {
  RowRef rr;
  if (!row_at<DEV>(a, s, unit, rows, rr)) return;
  int t = ROWT == 64 ? threadIdx.x & 63 : threadIdx.x;
  asm volatile("" : "+v"(t));  // see group_unit
  const bool ok = merge_row<ROWT, PER>(rr, smem, s_aux, a.wgt, a.table, t);
  if (t == 0) a.valid[rr.v] = ok ? 1 : 0;
}

constexpr size_t cmax(size_t a, size_t b) { return a > b ? a : b; }
constexpr size_t WAVE_LDS = cmax(cmax(SMALL_LDS_BYTES, group_lds_bytes(SHAPE_G32X.lanes, SHAPE_G32X.per, 64)),
                                 cmax(merge_lds_bytes(64, 8), cmax(merge_lds_bytes(64, 6), merge_lds_bytes(64, 4))));
constexpr size_t PAIR_LDS = cmax(merge_lds_bytes(128, 8), merge_lds_bytes(128, 6));
constexpr size_t BLOCK_LDS = cmax(cmax(merge_lds_bytes(256, 10), merge_lds_bytes(256, 8)), cmax(merge_lds_bytes(256, 6), sizeof(TileEmitLds)));

// The second launch bounds: what LDS lets reside anyway (21 wavefronts, 10 pairs, 4 workgroups of 256 to a CU).  Left alone the
// device-sized kernels took 109, 104 and 132 registers, one workgroup in five and one in four less (the 134,652 rows of a
// 40,000-seed batch's second hop on the scale-22 graph: 79, 91 and 133 us, with the bounds 63, 70 and 81).
template <bool DEV>
__global__ __launch_bounds__(64, 5) void fused_wave_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[(WAVE_LDS + 7) / 8];
  __shared__ uint64_t s_aux[8];
  call_stamp(a.call);
  fork_mark(a.fork);
  const uint32_t tiles = DEV && a.sec[0].kind == SEC_SUM ? a.sec[0].units : 0u;
  if constexpr (DEV)
    each_wanted(tiles, blockIdx.x, gridDim.x, [&](uint32_t t) { return tile_asked(a, a.tile0 + t); },
                [&](uint32_t t) { tile_sum_wave(a, a.tile0 + t); });
  const UnitFinder<DEV> units(a);
  for (uint32_t u = unit_behind<DEV>(tiles);; u += gridDim.x) {
    SectionRef s;
    uint32_t unit = 0, rows = 0;
    if (!units.find(a, u, s, unit, rows)) return;
    switch (s.kind) {
      case SEC_SWEEP:
        if constexpr (!DEV)
          sweep_unit(a, unit, smem);
        break;
      case SEC_TINY:
        if constexpr (DEV) {
          RowRef rr;
          if (row_at<DEV>(a, s, unit * 64 + threadIdx.x, rows, rr)) a.valid[rr.v] = tiny_row(rr.off, rr.d, a.wgt, a.table) ? 1 : 0;
        }
        break;
      case SEC_G2: if constexpr (DEV) group_unit<DEV, SHAPE_G2.lanes, SHAPE_G2.per>(a, s, unit, rows, smem); break;
      case SEC_G4: if constexpr (DEV) group_unit<DEV, SHAPE_G4.lanes, SHAPE_G4.per>(a, s, unit, rows, smem); break;
      case SEC_G8: if constexpr (DEV) group_unit<DEV, SHAPE_G8.lanes, SHAPE_G8.per>(a, s, unit, rows, smem); break;
      case SEC_G16: group_unit<DEV, SHAPE_G16.lanes, SHAPE_G16.per>(a, s, unit, rows, smem); break;
      case SEC_G32: group_unit<DEV, SHAPE_G32.lanes, SHAPE_G32.per>(a, s, unit, rows, smem); break;
      case SEC_G32S: group_unit<DEV, SHAPE_G32S.lanes, SHAPE_G32S.per>(a, s, unit, rows, smem); break;
      case SEC_G32X: group_unit<DEV, SHAPE_G32X.lanes, SHAPE_G32X.per>(a, s, unit, rows, smem); break;
      case SEC_W1: merge_unit<DEV, 64, 4>(a, s, unit, rows, smem, s_aux); break;
      case SEC_W6: merge_unit<DEV, 64, 6>(a, s, unit, rows, smem, s_aux); break;
      case SEC_W2: merge_unit<DEV, 64, 8>(a, s, unit, rows, smem, s_aux); break;
      case SEC_SUM:
        if constexpr (!DEV) tile_sum_wave(a, a.tile0 + unit);
        break;
      default: break;
    }
    if (!DEV) return;
    __syncthreads();  // the next unit rewrites the arrays in LDS
  }
}

template <bool DEV>
__global__ __launch_bounds__(128, 5) void fused_pair_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[(PAIR_LDS + 7) / 8];
  __shared__ uint64_t s_aux[16];
  call_stamp(a.call);
  fork_mark(a.fork);
  const uint32_t pairs = DEV && a.sec[0].kind == SEC_TOTALS ? a.sec[0].units : 0u;
  if constexpr (DEV)
    each_wanted(pairs * 2, blockIdx.x * 2 + (threadIdx.x >> 6), gridDim.x * 2,
                [&](uint32_t t) { return t < a.sec[0].stride && tile_active(a, a.tile0 + t); },
                [&](uint32_t t) { tile_totals_wave(a, a.tile0 + t); });
  const UnitFinder<DEV> units(a);
  for (uint32_t u = unit_behind<DEV>(pairs);; u += gridDim.x) {
    SectionRef s;
    uint32_t unit = 0, rows = 0;
    if (!units.find(a, u, s, unit, rows)) return;
    switch (s.kind) {
      case SEC_P6: merge_unit<DEV, 128, 6>(a, s, unit, rows, smem, s_aux); break;
      case SEC_P8: merge_unit<DEV, 128, 8>(a, s, unit, rows, smem, s_aux); break;
      case SEC_TOTALS:
        if constexpr (!DEV) {
          const uint32_t t = unit * 2 + (threadIdx.x >> 6);
          if (t < s.stride) tile_totals_wave(a, a.tile0 + t);
        }
        break;
      default: break;
    }
    if (!DEV) return;
    __syncthreads();
  }
}

constexpr size_t WIDE_LDS = sizeof(StreamLds);  // two workgroups of it fill a CU
static_assert(WIDE_LDS % 8 == 0 && cmax(merge_lds_bytes(512, 10), cmax(merge_lds_bytes(512, 8), merge_lds_bytes(512, 6))) + 512 <= WIDE_LDS,
              "everything fits the same LDS");
template <bool DEV>
__global__ __launch_bounds__(512, 4) void fused_wide_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[(WIDE_LDS + 7) / 8];
  // the wavefronts' sums of merge_row, past the end of their arrays
  uint64_t* const s_aux = smem + (WIDE_LDS - 512) / 8;
  call_stamp(a.call);
  fork_mark(a.fork);
  auto scan = [&](uint32_t r) {
    if (a.trows[r].ntiles && a.trows[r].ok)
      tile_scan_row<512>(a.trows, r, a.ttot, a.BL, a.BH, a.nfh, a.ranges, *reinterpret_cast<TileScanLds<512>*>(smem));
  };
  // Rows of tiles by every grid-th workgroup; the rows behind them, where a.next is given, by the workgroup that is first free.
  const uint32_t scans = DEV && a.sec[0].kind == SEC_SCAN ? a.sec[0].units : 0u;
  if constexpr (DEV)
    each_wanted(scans, blockIdx.x, gridDim.x, [&](uint32_t r) { return a.trows[a.trow0 + r].active != 0; },
                [&](uint32_t r) {
                  scan(a.trow0 + r);
                  if (threadIdx.x == 0) a.built[a.trow0 + r] = a.hop;
                  __syncthreads();
                });
  const UnitFinder<DEV> units(a);
  for (uint32_t u = a.next ? scans + blockIdx.x : unit_behind<DEV>(scans);;) {
    SectionRef s;
    uint32_t unit = 0, rows = 0;
    if (!units.find(a, u, s, unit, rows)) return;
    switch (s.kind) {
      case SEC_STREAM: {
        RowRef rr;
        if (row_at<DEV>(a, s, unit, rows, rr)) {
          const bool ok = stream_row(rr, *reinterpret_cast<StreamLds*>(smem), a.wgt, a.table);
          if (threadIdx.x == 0) a.valid[rr.v] = ok ? 1 : 0;
        }
        break;
      }
      case SEC_B6: merge_unit<DEV, 512, 6>(a, s, unit, rows, smem, s_aux); break;
      case SEC_B8: merge_unit<DEV, 512, 8>(a, s, unit, rows, smem, s_aux); break;
      case SEC_B10: merge_unit<DEV, 512, 10>(a, s, unit, rows, smem, s_aux); break;
      case SEC_SCAN:
        if constexpr (!DEV) scan(a.trow0 + unit);
        break;
      default: break;
    }
    if (!DEV) return;
    if (!a.next) {
      u += gridDim.x;
      __syncthreads();
    } else {
      u = scans + next_unit(a.next);
    }
  }
}

// The rows of up to 5117 entries of that launch by themselves: without the streamed rows' LDS a CU holds three workgroups instead of two.
constexpr size_t MID_LDS = cmax(merge_lds_bytes(512, 10), cmax(merge_lds_bytes(512, 8), merge_lds_bytes(512, 6)));
__global__ __launch_bounds__(512, 6) void fused_mid_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[(MID_LDS + 7) / 8];
  __shared__ uint64_t s_aux[64];
  const UnitFinder<false> units(a);
  SectionRef s;
  uint32_t unit = 0, rows = 0;
  if (!units.find(a, blockIdx.x, s, unit, rows)) return;
  switch (s.kind) {
    case SEC_B6: merge_unit<false, 512, 6>(a, s, unit, rows, smem, s_aux); break;
    case SEC_B8: merge_unit<false, 512, 8>(a, s, unit, rows, smem, s_aux); break;
    case SEC_B10: merge_unit<false, 512, 10>(a, s, unit, rows, smem, s_aux); break;
    default: break;
  }
}

// Tiles in an order in which neighbours run on the same XCD (workgroup u on u mod 8), 64 in a row: a tile reads the weights of those
// it is paired with once more, and finds them in that XCD's cache.  (40 M entries, 11 M of them in tiles: 350 -> 345 us; 60 M: 531 -> 523.)
__device__ __forceinline__ uint32_t near_tile(uint32_t u, uint32_t n) {
  return (u | 511u) < n ? (u & ~511u) + (u & 7u) * 64u + ((u >> 3) & 63u) : u;
}

// LONGER: rows of 2558..3581 entries as well (block_takes_longer), for which a CU holds four workgroups instead of five.
template <bool DEV, bool LONGER>
__global__ __launch_bounds__(256, 4) void fused_block_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[((LONGER ? cmax(merge_lds_bytes(256, 14), BLOCK_LDS) : BLOCK_LDS) + 7) / 8];
  __shared__ uint64_t s_aux[32];
  call_stamp(a.call);
  fork_mark(a.fork);
  auto emit = [&](uint32_t tile) {
    tile_emit(a.geom[tile], tile, a.trows, a.wgt, a.BL, a.BH, a.nfh, a.ranges, a.table, a.valid, *reinterpret_cast<TileEmitLds*>(smem));
  };
  const uint32_t tiles = DEV && a.sec[0].kind == SEC_EMIT ? a.sec[0].units : 0u;
  if constexpr (DEV)
    each_wanted(tiles, blockIdx.x, gridDim.x, [&](uint32_t t) { return tile_active(a, a.tile0 + near_tile(t, tiles)); },
                [&](uint32_t t) {
                  emit(a.tile0 + near_tile(t, tiles));
                  __syncthreads();
                });
  const UnitFinder<DEV> units(a);
  for (uint32_t u = unit_behind<DEV>(tiles);; u += gridDim.x) {
    SectionRef s;
    uint32_t unit = 0, rows = 0;
    if (!units.find(a, u, s, unit, rows)) return;
    switch (s.kind) {
      case SEC_M6: merge_unit<DEV, 256, 6>(a, s, unit, rows, smem, s_aux); break;
      case SEC_M8: merge_unit<DEV, 256, 8>(a, s, unit, rows, smem, s_aux); break;
      case SEC_M14:
        if constexpr (LONGER) merge_unit<DEV, 256, 14>(a, s, unit, rows, smem, s_aux);
        break;
      case SEC_M10: merge_unit<DEV, 256, 10>(a, s, unit, rows, smem, s_aux); break;
      case SEC_EMIT:
        if constexpr (!DEV) {
          const uint32_t tile = a.tile0 + near_tile(unit, s.units);
          if (a.geom[tile].span) emit(tile);
        }
        break;
      default: break;
    }
    if (!DEV) return;
    __syncthreads();
  }
}

// Small builds in one launch.  Rows of up to 509 entries are a wavefront's, eight of which share a
// workgroup, any longer one has the workgroup to itself.
constexpr uint32_t ALL_WAVES = 8;
constexpr size_t ALL_SLICE = (WAVE_LDS + 64 + 15) / 16 * 16;  // of a wavefront, and its sums
static_assert(ALL_WAVES * ALL_SLICE <= WIDE_LDS, "eight wavefronts fit the same LDS");
__global__ __launch_bounds__(512, 4) void fused_all_kernel(FusedArgs a) {
  __shared__ __align__(16) uint64_t smem[(WIDE_LDS + 7) / 8];
  call_stamp(a.call);
  const UnitFinder<false> units(a);
  SectionRef s;
  uint32_t unit = 0, rows = 0;
  units.find(a, blockIdx.x, s, unit, rows);
  uint64_t* const s_aux = smem + (WIDE_LDS - 512) / 8;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), wunit = unit * ALL_WAVES + wave;
  uint64_t* const wmem = smem + wave * (ALL_SLICE / 8);
  uint64_t* const w_aux = wmem + (ALL_SLICE - 64) / 8;
  switch (s.kind) {
    case SEC_SWEEP: sweep_unit(a, wunit, wmem); break;
    case SEC_G16: group_unit<false, SHAPE_G16.lanes, SHAPE_G16.per>(a, s, wunit, rows, wmem); break;
    case SEC_G32: group_unit<false, SHAPE_G32.lanes, SHAPE_G32.per>(a, s, wunit, rows, wmem); break;
    case SEC_G32S: group_unit<false, SHAPE_G32S.lanes, SHAPE_G32S.per>(a, s, wunit, rows, wmem); break;
    case SEC_G32X: group_unit<false, SHAPE_G32X.lanes, SHAPE_G32X.per>(a, s, wunit, rows, wmem); break;
    case SEC_W1: merge_unit<false, 64, 4>(a, s, wunit, rows, wmem, w_aux); break;
    case SEC_W6: merge_unit<false, 64, 6>(a, s, wunit, rows, wmem, w_aux); break;
    case SEC_W2: merge_unit<false, 64, 8>(a, s, wunit, rows, wmem, w_aux); break;
    case SEC_B6: merge_unit<false, 512, 6>(a, s, unit, rows, smem, s_aux); break;
    case SEC_B10: merge_unit<false, 512, 10>(a, s, unit, rows, smem, s_aux); break;
    case SEC_STREAM: {
      RowRef rr;
      if (row_at<false>(a, s, unit, rows, rr)) {
        const bool ok = stream_row(rr, *reinterpret_cast<StreamLds*>(smem), a.wgt, a.table);
        if (threadIdx.x == 0) a.valid[rr.v] = ok ? 1 : 0;
      }
      break;
    }
    default: break;
  }
}

// ---------------------------------------------------------------- plan of a graph
// Geometry of the rows that are built tile by tile, in list order: one workgroup, once per graph.
__global__ __launch_bounds__(1024) void plan_rows_kernel(const RowRef* __restrict__ list, uint32_t n, TiledRow* __restrict__ rows,
                                                         uint32_t row0, uint32_t tile0) {
  __shared__ uint32_t s_w[16];
  const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  uint32_t carry = 0;
  for (uint32_t c = 0; c < n; c += 1024u) {
    const uint32_t r = c + tid;
    uint32_t nt = 0;
    RowRef rr{0, 0, 0, 0};
    if (r < n) {
      rr = list[r];
      nt = ((rr.off & 3u) + rr.d + TILE - 1) / TILE;
    }
    const uint32_t inc = group_scan_u32<64>(nt);
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    uint32_t before = carry, total = 0;
    for (uint32_t w = 0; w < 16; ++w) {
      if (w == wave) before += total;
      total += s_w[w];
    }
    if (r < n) {
      TiledRow& o = rows[row0 + r];
      o.v = rr.v;
      o.off = rr.off;
      o.d = rr.d;
      o.base = rr.off & ~3u;
      o.lead = rr.off & 3u;
      o.span = o.lead + rr.d;
      o.ntiles = nt;
      o.tile0 = tile0 + before + inc - nt;
      o.bofs = o.tile0 + row0 + r;  // every row owns ntiles + 1 prefix slots
      o.active = 0;
    }
    carry += total;
    __syncthreads();
  }
}
__global__ __launch_bounds__(256) void plan_tiles_kernel(const TiledRow* __restrict__ rows, TileGeom* __restrict__ geom) {
  const TiledRow& row = rows[blockIdx.x];
  for (uint32_t t = threadIdx.x; t < row.ntiles; t += 256)
    geom[row.tile0 + t] = TileGeom{blockIdx.x, t, row.base, row.lead, row.span, {0, 0, 0}};
}
__global__ __launch_bounds__(64) void fused_ledger_kernel(TiledRow* __restrict__ rows, uint32_t row0, const u128* __restrict__ tsum,
                                                          bool frontier) {
  TiledRow& row = rows[row0 + blockIdx.x];
  if (row.ntiles == 0 || (frontier && !row.active)) return;
  u128 sum{0, 0};
  for (uint32_t t = threadIdx.x; t < row.ntiles; t += 64) sum = add128(sum, tsum[row.tile0 + t]);
  sum = group_sum_u128<64>(sum);
  if (threadIdx.x == 0) {
    const bool ok = (sum.lo | sum.hi) != 0;
    row.ok = ok;
    if (ok) {
      const Ledger L = make_ledger(row.d, sum);
      row.scale = L.scale;
      row.fs = L.fs;
      row.inv_fs = L.inv_fs;
      row.one = L.one;
    }
  }
}

namespace {
// Rows of more tiles than this get their ledger from a launch of its own: 2048 tiles add up 2048 x 2048 sums of 16
// bytes, 67 MB out of L2, when every tile does it.
constexpr uint32_t LEDGER_TILES = 2048;

// Builds of at most so many workgroups of 512 threads, and without longer rows than this, go out in one launch: each of the
// others costs 5 to 15 us, mostly of waiting for the last row.  With more workgroups their LDS and registers, which leave fewer
// wavefronts on a CU than the four kernels do, cost more; a longer row takes longer to stream (29 us for this one) than the
// passes over its tiles.  (Four launches / one, us: scale 10 with 8 edges a vertex 32 / 23, scale 13 with 16 45 / 24, scale 16 with 4
// 51 / 24, scale 20 with 3 80 / 59; rebuilds by workgroups: 2,300 75 / 53, 4,000 110 / 86, 12,000 141 / 151; by the longest
// row: 8,600 56 / 36, 15,400 with few others 62 / 76.)
constexpr uint64_t ALL_MOST = 4096;
constexpr uint32_t ALL_LONGEST = 12288;
static_assert(ALL_LONGEST <= 24576, "none is of class CLS_STREAM");

// Graphs of at most so many vertices sweep their rows of up to 32 entries with four wavefronts a range, one to a class: nothing but
// the chain of a wavefront's batches bounds so few rows, and there one batch is left of four.  More vertices keep the GPU busy
// without, and four wavefronts that share their lines read and write them four times (one wavefront / four, us: scale 9 with 5
// edges a vertex 17.2 / 13.6, scale 10 with 8 17.7 / 13.6, scale 13 with 8 19.6 / 14.9, scale 15 with 3 19.0 / 15.5, with 20 32.3 / 32.5,
// scale 16 with 8 25.5 / 26, scale 17 with 4 19.7 / 20.5, scale 18 with 3 25.7 / 28, scale 20 with 16 137 / 171).
constexpr uint32_t SPLIT_SWEEP = 1u << 15;

// Whole builds of at least so many entries that go out beside one another send out the rows of 2558..5117 entries in a launch of
// their own, beside the others on a third stream, which costs smaller ones more (in the launch of the longer rows / by
// themselves, us: scale 16 with 16 edges a vertex 43 / 46, scale 20 with 6 82 / 86, 10 M entries in rows of up to 50,000 100 / 103, of
// up to 7,000 87 / 87, scale 20 with 16 119 / 119, with 30 193 / 187, scale 22 with 16 357 / 348, scale 23 with 10 432 / 421, 40 M entries in rows of
// up to 5,000 249 / 232, of up to 300,007 319 / 314, 60 M of up to 9,000 362 / 365, scale 21 with 40 456 / 461).
constexpr uint32_t MID_ALONE = 1u << 24;

// Rows of 5118..8189 entries from which they are a launch of their own (10,000 rows of 6,500 streamed 478 us, held 402; 20,000
// 885 and 745): fewer save less than a launch costs.
constexpr uint32_t HOLD_ALONE = 2048;

// Entries of a graph from which a build of its longer rows alone, which has no sweep, is worth a fork (in order / beside, us: walks without tables of
// 10,000 x 8 on the scale-22 graph 195 / 188, of 836 x 10 on the scale-16 graph with 47 edges a vertex 75 / 79).
constexpr uint32_t PART_BESIDE = 1u << 24;
// Entries to build from which it is not any more: the launches then fill the GPU one after another, and share caches and LDS beside one
// another.  (In order / beside, us, entries to build: walks of 10,000 x 8 on the scale-22 graph with 16 edges a vertex, 12.8 M, 183 / 176,
// scale 23 with 10, 13.6 M, 175 / 169, with 12, 16.3 M, 235 / 234, with 16, 21.7 M, 279 / 282, scale 22 with 24, 19 M, 271 / 273, with 32, 25 M, 353 / 352;
// 2,000 x 8 on the scale-24 graph with 16, 13.4 M, 266 / 220; 30,000 x 12 on scale 23 with 16, 43 M, 434 / 443, with 20, 54 M, 547 / 563, 40,000 x 16, scale
// 22 with 24, 56 M, 524 / 531.)
constexpr uint64_t PART_MOST = 16000000;

// Entries in rows of 510..2557, which the launches of the tile passes take, from which a whole build goes out in order for the same reason.
// (In order / beside, us, their number: scale 23 with 8 edges a vertex, 10.7 M, 371 / 364, with 10, 14.8 M, 433 / 419, scale 24 with 6, 14.7 M, 525 / 516,
// 80 M entries in rows of up to 300,007, 9.2 M, 598 / 576, scale 22 with 16, 17 M, 364 / 348; scale 21 with 45, 18.9 M, 499 / 504, 110 M in rows of up
// to 3,000, 22.8 M, 606 / 607, scale 22 with 31, 25.7 M, 651 / 659, scale 24 with 7, 27.8 M, 626 / 629, scale 22 with 18, 27.9 M, 425 / 435, with 22, 34 M, 491 /
// 500, scale 23 with 14, 41 M, 612 / 619.)
constexpr uint64_t BESIDE_MERGED = 18000000;

// Tiles of a graph's plan from which a frontier of few rows has launches of their own for them (build_frontier).
constexpr uint32_t TILES_APART = 8192;

// Frontiers of at most this many rows make the rows of 8190..65533 entries tile by tile.
constexpr uint32_t SMALL_FRONTIER = 65536;

int alloc(void** p, size_t bytes) {
  SKY_HIP(hipMalloc(p, bytes + 16));
  return SKY_OK;
}
}  // namespace

BuildPlan::~BuildPlan() {
  void* ptrs[] = {rows, trows, tiles};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
}

int ensure_plan(sky_graph* g, CallDevice** first) {
  const long long narrow_limit = option(g, OPT_STREAM_MIN_EDGES);
  if (g->plan && g->plan->narrow_limit == narrow_limit) return SKY_OK;
  g->plan.reset();
  hipStream_t st = g->stream;
  g->plan = std::make_shared<BuildPlan>();
  BuildPlan& p = *g->plan;
  auto body = [&]() -> int {
    SKY_TRY(bin_all_rows(g, CLS_G16, &p.rows, p.start, first));
    p.listed = 0;
    for (int c = CLS_G16; c < CLS_COUNT; ++c) p.listed += g->bin_counts[c];
    p.narrow_limit = narrow_limit;
    // Those of 8190..65533 entries by narrow_rows; small frontiers make them tile by tile, for which they need geometry.  A graph with very
    // many of them does without: 65536 tiles that a frontier may have to pass over take 20 us a launch.
    const uint64_t last = g->bin_edges[CLS_STREAM_LAST], narrow = g->bin_edges[CLS_STREAM] + last;
    uint64_t wide = g->bin_edges[CLS_HOLD];
    for (int c = CLS_MW2 + 4; c <= CLS_MW2 + MERGE_MAX_NW - 2; ++c) wide += g->bin_edges[c];
    switch (narrow_rows(narrow_limit, last, g->bin_edges[CLS_STREAM], wide, g->max_degree)) {
      case NarrowRows::STREAMED: p.t_all = CLS_STREAM_WIDE; break;
      case NarrowRows::TO_24576_STREAMED: p.t_all = CLS_STREAM; break;
      case NarrowRows::TILED: p.t_all = CLS_STREAM_LAST; break;
    }
    p.t_first = p.t_all == CLS_STREAM_LAST || narrow <= 65536ull * TILE ? CLS_STREAM_LAST : p.t_all;
    // Tiles of the rows that only small frontiers make tile by tile, then those of the others, from a bound of the former on: that is
    // known without asking the device, and the places between are no tiles.
    uint64_t edges = 0, early_edges = 0;
    for (int c = p.t_first; c <= CLS_HUGE; ++c) {
      p.n_trows += g->bin_counts[c];
      edges += g->bin_edges[c];
      if (c < p.t_all) {
        p.wide_row += g->bin_counts[c];
        early_edges += g->bin_edges[c];
      }
    }
    if (!p.n_trows) return SKY_OK;
    const uint64_t wide_tile = early_edges / TILE + 2ull * p.wide_row;
    const uint64_t bound = wide_tile + (edges - early_edges) / TILE + 2ull * (p.n_trows - p.wide_row);
    if (bound >= (1ull << 31)) return fail(SKY_ERR_LIMIT, "the number of tiles has no usable bound");
    p.wide_tile = (uint32_t)wide_tile;
    p.n_tiles = (uint32_t)bound;
    SKY_TRY(alloc((void**)&p.trows, (size_t)p.n_trows * sizeof(TiledRow)));
    const size_t nb = (size_t)p.n_tiles + p.n_trows;
    // one allocation for everything that has one entry per tile
    const size_t bytes = (size_t)p.n_tiles * (sizeof(TileGeom) + sizeof(u128) + sizeof(uint4) + sizeof(TileTotals) + 4) + nb * 16;
    char* at = nullptr;
    SKY_TRY(alloc((void**)&at, bytes));
    p.tiles = at;
    auto take = [&](auto& ptr, size_t n) {
      ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(at);
      at += n * sizeof(*ptr);
    };
    take(p.geom, p.n_tiles);
    take(p.tsum, p.n_tiles);
    take(p.ranges, p.n_tiles);
    take(p.ttot, p.n_tiles);
    take(p.BL, nb);
    take(p.BH, nb);
    take(p.nfh, p.n_tiles);
    SKY_HIP(hipMemsetAsync(p.geom, 0, (size_t)p.n_tiles * sizeof(TileGeom), st));  // span 0: no such tile
    const RowRef* const list = p.rows + p.start[p.t_first];
    if (p.wide_row) hipLaunchKernelGGL(plan_rows_kernel, dim3(1), dim3(1024), 0, st, list, p.wide_row, p.trows, 0u, 0u);
    if (p.wide_row < p.n_trows)
      hipLaunchKernelGGL(plan_rows_kernel, dim3(1), dim3(1024), 0, st, list + p.wide_row, p.n_trows - p.wide_row, p.trows, p.wide_row,
                         p.wide_tile);
    hipLaunchKernelGGL(plan_tiles_kernel, dim3(p.n_trows), dim3(256), 0, st, p.trows, p.geom);
    SKY_HIP(hipGetLastError());
    return SKY_OK;
  };
  const int rc = body();
  if (rc != SKY_OK) g->plan.reset();
  return rc;
}

namespace {
struct Launch {
  FusedArgs a;
  uint64_t units = 0;
  uint32_t threads;
  Launch(const FusedArgs& base, uint32_t t) : a(base), threads(t) {
    a.nsec = 0;
    for (uint32_t& f : a.first) f = 0xFFFFFFFFu;
  }
  // host-sized: `rows` rows from `start` on
  void add(Section k, uint32_t rows, uint32_t per, uint32_t start) {
    if (!rows) return;
    a.first[a.nsec] = (uint32_t)units;
    a.sec[a.nsec++] = SectionRef{k, (rows + per - 1) / per, per, start, -1, 0, rows};
    units += (rows + per - 1) / per;
  }
  // device-sized: at most `upper` rows in the segments of the classes cls .. cls + ncls - 1
  void add_dev(Section k, uint32_t upper, uint32_t per, uint32_t start, int cls, int ncls, uint32_t stride) {
    if (!upper) return;
    a.sec[a.nsec++] = SectionRef{k, 0, per, start, cls, ncls, stride};
    units += (upper + per - 1) / per;
  }
};

FusedArgs common_args(sky_graph* g, const BuildPlan& p, int tiled_from) {
  FusedArgs a = {};
  a.xadj = g->xadj;
  a.wgt = g->adjwgt;
  a.table = g->table;
  a.valid = g->valid;
  a.V = g->V;
  a.trows = p.trows;
  a.geom = p.geom;
  a.tsum = p.tsum;
  a.ttot = p.ttot;
  a.BL = p.BL;
  a.BH = p.BH;
  a.nfh = p.nfh;
  a.ranges = p.ranges;
  a.trow0 = tiled_from == p.t_first ? 0u : p.wide_row;
  a.tile0 = tiled_from == p.t_first ? 0u : p.wide_tile;
  a.ledgers_done = p.n_trows > a.trow0 && ((uint64_t)g->max_degree + 3 + TILE - 1) / TILE > LEDGER_TILES;
  return a;
}

// Whether the rows of 2558..3581 entries (CLS_MW2 + 4 and + 5) go out with the launch of 256 threads, 14 slots each, rather than in
// that of the streamed rows, whose LDS leaves two workgroups of 512 to a CU (in the streamed rows' launch / here, us: scale 22 with 31 edges a vertex
// 674 / 652, scale 21 with 45 510 / 499, 110 M entries in rows of up to 3,000 617 / 607, 40,000 seeds 25 x 10 on the scale-22 graph with 32 714 / 671).
// With their LDS a CU holds four workgroups of that launch instead of five, which costs tiles more (16 M entries in tiles 543 -> 570 us),
// and where they have a launch of their own (MID_ALONE) there is nothing to be had by it (there / here: scale 22 with 10 238 / 245, with 11
// 263 / 269).
constexpr double LONGER_ENTRIES = 4e6, LONGER_PER_TILED = 2;
bool block_takes_longer(const sky_graph* g, int tiled_from) {
  double tiled = 0;
  for (int c = tiled_from; c <= CLS_HUGE; ++c) tiled += (double)g->bin_edges[c];
  const double longer = (double)g->bin_edges[CLS_MW2 + 4] + (double)g->bin_edges[CLS_MW2 + 5];
  return longer >= std::max(LONGER_ENTRIES, LONGER_PER_TILED * tiled);
}

// Whether the workgroups of a frontier's wide launch ask for their next unit instead of taking every 512th.  A streamed row of 60,000
// entries takes seven times as long as one of 8,000, and who asks waits 2 us: not where merges, of some 8 us, are most of the units.
// (40,000 seeds 25 x 10 on the scale-22 graph with 32 edges a vertex, 1,800 streamed rows: 177 us, asked for 162; with 7,300 merges
// beside them 297, asked for 330.)
bool streams_by_queue(const sky_graph* g, int tiled_from, bool longer) {
  if (tiled_from == CLS_STREAM_LAST) return false;
  uint64_t merges = 0;
  for (int c = CLS_MW2 + (longer ? 6 : 4); c <= CLS_MW2 + 8; ++c) merges += g->bin_counts[c];
  return merges <= (uint64_t)g->bin_counts[CLS_STREAM_LAST] + (tiled_from > CLS_STREAM ? g->bin_counts[CLS_STREAM] : 0u);
}

// One launch, if it has anything to do.  Device-sized ones know a bound of their units only: as many workgroups as the GPU holds at a time
// stride over what there is; of the pairs and of 256 threads, whose units differ most, three and two times as many, of which the last go where
// there is room first.  (Once / so many times, us: 40,000 seeds 25 x 10 on the scale-22 graph with 32 edges a vertex 671 / 666, 5,000 x 15 x 10 x 5
// 537 / 530, 300 x 25 x 10 236 / 223, 40,000 x 25 x 10, scale 20, 298 / 293.  Twice as many of 64 or 512 threads: 2 to 7 us more.)
template <bool DEV>
int enqueue(const BuildPlan& p, const Launch& l, bool longer, hipStream_t st) {
  if (!l.units) return SKY_OK;
  const uint32_t resident = l.threads == 64 ? 5120 : l.threads == 128 ? 3 * 2560 : l.threads == 256 ? 2 * 1024 : 512;
  const dim3 grid((uint32_t)(DEV ? std::min<uint64_t>(l.units, resident) : l.units));
  if (l.threads == 64) hipLaunchKernelGGL((fused_wave_kernel<DEV>), grid, dim3(64), 0, st, l.a);
  else if (l.threads == 128) hipLaunchKernelGGL((fused_pair_kernel<DEV>), grid, dim3(128), 0, st, l.a);
  else if (l.threads == 512) hipLaunchKernelGGL((fused_wide_kernel<DEV>), grid, dim3(512), 0, st, l.a);
  else if (longer) hipLaunchKernelGGL((fused_block_kernel<DEV, true>), grid, dim3(256), 0, st, l.a);
  else hipLaunchKernelGGL((fused_block_kernel<DEV, false>), grid, dim3(256), 0, st, l.a);
  if (l.a.nsec && l.a.sec[0].kind == SEC_SUM && l.a.ledgers_done)
    hipLaunchKernelGGL(fused_ledger_kernel, dim3(p.n_trows - l.a.trow0), dim3(64), 0, st, p.trows, l.a.trow0, p.tsum, DEV);
  SKY_HIP(hipGetLastError());
  return SKY_OK;
}
}  // namespace

bool fused_possible(const sky_graph* g) { return option(g, OPT_ROW_MERGE) != 0 && tiled_max_tiles(g) == (1u << 22); }

static int build_host_sized(sky_graph* g, uint32_t min_degree, CallDevice* call) {
  g->has_walk_index = false;
  const BuildPlan& p = *g->plan;
  FusedArgs base = common_args(g, p, p.t_all);
  const uint32_t n_tiles = p.n_tiles - base.tile0, n_trows = p.n_trows - base.trow0;
  base.list = p.rows;
  auto rows = [&](int c) { return class_min_degree(c) >= min_degree ? g->bin_counts[c] : 0u; };
  uint32_t past_wave = 0;  // rows of more than 509 entries: what a second launch would be for
  for (int c = CLS_COUNT - 1; c > CLS_LDS_W2; --c)
    if (class_min_degree(c) >= 510) past_wave += rows(c);
  // Vertices of a wavefront: enough wavefronts for every SIMD, but 128 rather than fewer where two wavefronts a SIMD remain, and up to 256 where
  // four do: the rows of a few vertices fill no batch of their class.  The last wavefronts of a sweep beside other launches are what is left of it behind
  // them: there a 12,288th of the vertices is the limit instead of an 8,192th.  (64 where there were fewer than 4,096 wavefronts of 128, 256 up
  // to 2 M vertices, an 8,192th above / now, us: 3 M entries in 478,000 rows 44 / 36, scale 20 with 6 edges a vertex 83 / 78, scale 22 with 3
  // 115 / 110, scale 23 with 4 232 / 219; scale 22 with 4 127 / 129, with 10 242 / 245; most others within 1 %.  29 M entries in rows of up to
  // 339, one launch, an 8,192th / a 12,288th 176 / 181.)
  base.split = g->V <= SPLIT_SWEEP;
  auto sweep = [&](bool beside) -> uint32_t {  // its wavefronts
    const uint32_t least = g->V > 1u << 20 ? 256u : std::min(192u, std::max(g->V / 4096u, std::min(128u, g->V / 2048u)));
    const uint32_t range = std::max(g->V / (beside ? 12288u : 8192u), least) / 64u * 64u;
    base.per_wave = base.split ? 64u : std::max(64u, std::min(SMALL_RANGE, range));
    const uint32_t ranges = (g->V + base.per_wave - 1) / base.per_wave;
    return base.split ? 4 * ranges : ranges;
  };
  if (past_wave && g->max_degree <= ALL_LONGEST) {
    const uint32_t sweeps = sweep(true);
    Launch all(base, 512);
    auto waves = [&](Section k, int c, uint32_t per) { all.add(k, rows(c), per * ALL_WAVES, p.start[c]); };
    all.add(SEC_STREAM, rows(CLS_STREAM_LAST), 1, p.start[CLS_STREAM_LAST]);
    all.add(SEC_STREAM, rows(CLS_HOLD), 1, p.start[CLS_HOLD]);
    auto range = [&](Section k, int c0, int c1) {  // classes whose lists lie back to back; min_degree may leave out the first ones
      uint32_t n = 0;
      int c = c0;
      for (int i = c1; i >= c0; --i)
        if (rows(i)) {
          n += rows(i);
          c = i;
        }
      all.add(k, n, 1, p.start[c]);
    };
    range(SEC_B10, CLS_MW2 + 5, CLS_MW2 + 8);
    range(SEC_B6, CLS_MW2, CLS_MW2 + 4);
    all.add(SEC_B6, rows(CLS_MW2_6), 1, p.start[CLS_MW2_6]);
    waves(SEC_W2, CLS_LDS_W2, 1);
    if (min_degree == 0) all.add(SEC_SWEEP, sweeps, ALL_WAVES, 0);
    waves(SEC_W6, CLS_LDS_W6, 1);
    waves(SEC_W1, CLS_LDS_W1, 1);
    waves(SEC_G32X, CLS_G32X, 64 / SHAPE_G32X.lanes);
    waves(SEC_G32S, CLS_G32S, 64 / SHAPE_G32S.lanes);
    waves(SEC_G32, CLS_G32, 64 / SHAPE_G32.lanes);
    waves(SEC_G16, CLS_G16, 64 / SHAPE_G16.lanes);
    if (all.units <= ALL_MOST) {
      all.a.call = call;
      if (all.units) hipLaunchKernelGGL(fused_all_kernel, dim3((uint32_t)all.units), dim3(512), 0, g->stream, all.a);
      SKY_HIP(hipGetLastError());
      return SKY_OK;
    }
  }
  uint32_t past_block = p.t_all > CLS_STREAM ? rows(CLS_STREAM) : 0u;  // rows of 2558 entries and more that are not made tile by tile
  if (p.t_all > CLS_STREAM_LAST) past_block += rows(CLS_STREAM_LAST);
  past_block += rows(CLS_HOLD);
  for (int c = CLS_MW2 + 4; c <= CLS_MW2 + MERGE_MAX_NW - 2; ++c) past_block += rows(c);
  auto entries = [&](uint32_t from, uint32_t to) {  // in rows of so many
    uint64_t n = 0;
    for (int c = CLS_TINY; c < CLS_COUNT; ++c)
      if (class_min_degree(c) >= from && class_min_degree(c) < to) n += g->bin_edges[c];
    return n;
  };
  Beside side;
  ForkMark mark{nullptr, 0};
  const bool two = min_degree == 0 && g->E >= MID_ALONE && past_block;
  if (min_degree == 0 ? past_wave && entries(510, 2558) < BESIDE_MERGED : g->E >= PART_BESIDE && past_block && entries(min_degree, 0xFFFFFFFFu) < PART_MOST) SKY_TRY(beside_begin(g, &side, &mark, two ? 2 : 1));
  // Without a fork four launches follow one another: the sweep rides along in the first, the long rows behind the scans.
  const bool fork = side.stream[0] != nullptr;
  const uint32_t sweeps = sweep(fork);
  Launch pair(base, 128), scan(base, 512), block(base, 256), rest(base, 64), wide(base, 512), alone(base, 512);
  Launch &longs = fork ? wide : scan, &mid = fork && min_degree == 0 && g->E >= MID_ALONE ? alone : longs;
  pair.add(SEC_TOTALS, n_tiles, 2, 0);
  pair.add(SEC_P8, rows(CLS_MW2), 1, p.start[CLS_MW2]);
  pair.add(SEC_P6, rows(CLS_MW2_6), 1, p.start[CLS_MW2_6]);
  scan.add(SEC_SCAN, n_trows, 1, 0);
  if (p.t_all > CLS_STREAM) longs.add(SEC_STREAM, rows(CLS_STREAM), 1, p.start[CLS_STREAM]);
  if (p.t_all > CLS_STREAM_LAST) longs.add(SEC_STREAM, rows(CLS_STREAM_LAST), 1, p.start[CLS_STREAM_LAST]);
  // Rows of 5118..8189 entries: streamed beside the others, where hold_row would spill, or, where they are enough for a launch,
  // HOLD_ALONE, by build_hold_kernel.
  const bool hold_alone = min_degree == 0 && rows(CLS_HOLD) >= HOLD_ALONE;  // last on the graph's stream; `first` stamps the call
  if (!hold_alone) longs.add(SEC_STREAM, rows(CLS_HOLD), 1, p.start[CLS_HOLD]);
  // two classes whose lists lie back to back; min_degree may leave out the first
  auto add_two = [&](Launch& l, Section k, int c) { l.add(k, rows(c) + rows(c + 1), 1, p.start[rows(c) ? c : c + 1]); };
  add_two(mid, SEC_B10, CLS_MW2 + 7);
  const bool longer = &mid != &alone && block_takes_longer(g, p.t_all);
  if (longer) {
    mid.add(SEC_B8, rows(CLS_MW2 + 6), 1, p.start[CLS_MW2 + 6]);
  } else {
    add_two(mid, SEC_B8, CLS_MW2 + 5);
    mid.add(SEC_B6, rows(CLS_MW2 + 4), 1, p.start[CLS_MW2 + 4]);
  }
  block.add(SEC_EMIT, n_tiles, 1, 0);
  if (longer) add_two(block, SEC_M14, CLS_MW2 + 4);
  block.add(SEC_M10, rows(CLS_MW2 + 3), 1, p.start[CLS_MW2 + 3]);
  block.add(SEC_M8, rows(CLS_MW2 + 2), 1, p.start[CLS_MW2 + 2]);
  block.add(SEC_M6, rows(CLS_MW2 + 1), 1, p.start[CLS_MW2 + 1]);
  // Rows of up to 509 entries alone are one launch; beside others the sweep goes to the side.
  const bool sides = fork && pair.units + scan.units + block.units + wide.units + alone.units > 0;
  Launch wave(base, 64);
  wave.add(SEC_SUM, n_tiles, 1, 0);
  wave.add(SEC_W2, rows(CLS_LDS_W2), 1, p.start[CLS_LDS_W2]);
  if (min_degree == 0) (sides ? rest : wave).add(SEC_SWEEP, sweeps, 1, 0);
  wave.add(SEC_W6, rows(CLS_LDS_W6), 1, p.start[CLS_LDS_W6]);
  wave.add(SEC_W1, rows(CLS_LDS_W1), 1, p.start[CLS_LDS_W1]);
  wave.add(SEC_G32X, rows(CLS_G32X), 64 / SHAPE_G32X.lanes, p.start[CLS_G32X]);
  wave.add(SEC_G32S, rows(CLS_G32S), 64 / SHAPE_G32S.lanes, p.start[CLS_G32S]);
  wave.add(SEC_G32, rows(CLS_G32), 64 / SHAPE_G32.lanes, p.start[CLS_G32]);
  wave.add(SEC_G16, rows(CLS_G16), 64 / SHAPE_G16.lanes, p.start[CLS_G16]);
  // The passes over tiles depend on one another, the last three launches on nothing; only a build without the others has one of them first.
  Launch* const order[] = {&wave, &pair, &scan, &block, &rest, &wide};
  Launch* first = nullptr;
  for (Launch* l : order)
    if (l->units && !first) first = l;
  if (first) {
    first->a.call = call;
    if (rest.units + wide.units + alone.units && first != &rest && first != &wide) first->a.fork = mark;
    else side = Beside{};
    SKY_TRY(enqueue<false>(p, *first, longer, g->stream));
  }
  auto others = [&]() -> int {
    hipStream_t on[2] = {g->stream, g->stream};
    for (int k = 0; k < 2; ++k)
      if (side.stream[k] && (k ? alone.units : rest.units + wide.units)) {
        SKY_TRY(beside_fork(&side, k));
        on[k] = side.stream[k];
      }
    for (Launch* l : {&rest, &wide})
      if (l != first) SKY_TRY(enqueue<false>(p, *l, longer, on[0]));
    if (alone.units) hipLaunchKernelGGL(fused_mid_kernel, dim3((uint32_t)alone.units), dim3(512), 0, on[1], alone.a);
    SKY_HIP(hipGetLastError());
    for (Launch* l : {&wave, &pair, &scan, &block})
      if (l != first) SKY_TRY(enqueue<false>(p, *l, longer, g->stream));
    if (hold_alone) SKY_TRY(build_rows_hold(g, p.rows + p.start[CLS_HOLD], rows(CLS_HOLD)));
    if (min_degree == 0) side.last = &g->call;  // build_all_fused: nothing but the call's end follows
    return beside_join(&side);
  };
  const int rc = others();
  if (rc != SKY_OK) beside_drop(&side);
  return rc;
}
int build_all_fused(sky_graph* g, CallDevice* call) { return build_host_sized(g, 0, call); }
int build_rows_from(sky_graph* g, uint32_t min_degree, CallDevice* call) { return build_host_sized(g, min_degree, call); }

// ---------------------------------------------------------------- rows of a frontier
int frontier_lists(sky_graph* g, const BuildPlan& p, uint32_t n_upper, sky_graph::PoolBuf* buf, FrontierLists* f) {
  // A workgroup needs 125 us to stream a row of 65,000 entries, which is as long as everything else that the build of a
  // small frontier does; the rows of a large one keep all workgroups streaming, and that is cheaper by the entry.
  f->few = n_upper <= SMALL_FRONTIER;
  f->tiled_from = f->few ? p.t_first : p.t_all;
  uint64_t at = 0;
  for (int c = 0; c < CLS_COUNT; ++c) {
    f->start[c] = (uint32_t)at;
    const bool tiled = c >= f->tiled_from && c <= CLS_HUGE;
    const uint64_t in_graph = c == CLS_TINY ? g->bin_edges[c] : g->bin_counts[c];  // a tiny row has an entry at least
    f->cap[c] = c == CLS_EMPTY || tiled ? 0u : (uint32_t)std::min<uint64_t>(n_upper, in_graph);
    at += f->cap[c];
  }
  SKY_TRY(buf_grow(buf, at * sizeof(RowRef)));
  f->list = (RowRef*)buf->p;
  return SKY_OK;
}

__global__ void clear_taken_kernel(uint32_t* taken) { *taken = 0; }

int build_frontier(sky_graph* g, const BuildPlan& p, const FrontierLists& f, uint32_t* counts, bool again, const uint32_t* bitmap,
                   uint32_t* built, uint32_t hop) {
  g->has_walk_index = false;
  FusedArgs base = common_args(g, p, f.tiled_from);
  const uint32_t n_tiles = p.n_tiles - base.tile0, n_trows = p.n_trows - base.trow0;
  base.list = f.list;
  base.counts = counts;
  base.bitmap = bitmap;
  base.bit_mask = frontier_mask(g->V);
  base.built = built;
  base.hop = hop + 1;
  Launch wave(base, 64), pair(base, 128), wide(base, 512), block(base, 256);
  Launch sum(base, 64), totals(base, 128), scan(base, 512), emit(base, 256);
  // The passes over tiles wait for one another, and where they look at many tiles for a frontier of few rows they are a good part: the rows then
  // go out beside them, the longest first.  (In the same four launches / beside, us: 40,000 seeds x 20 on the scale-22 graph with 30 edges a
  // vertex, 26,000 tiles, 125 / 115, 300 x 25 x 10 with 32 231 / 225, 40,000 x 25 x 10 676 / 669, 2,000 x 10 x 10 on the scale-21 graph with 40, 13,000
  // tiles, 338 / 329; with few tiles it costs more launches: 28,208 x 10 x 10 on the scale-19 graph with 5 140 / 149, 1,165 x 25 x 10, scale 16,
  // 125 / 139, 476 x 5 x 3 on the scale-22 graph with 5 75 / 79.)
  Beside side;
  ForkMark mark{nullptr, 0};
  if (f.few && n_tiles >= TILES_APART) SKY_TRY(beside_begin(g, &side, &mark, 1));
  const bool apart = side.stream[0] != nullptr;
  sum.a.fork = mark;
  auto add = [&](Launch& l, Section k, uint32_t per, int cls, int ncls = 1) {
    uint32_t upper = 0;
    for (int c = 0; c < ncls; ++c) upper += f.cap[cls + c];
    l.add_dev(k, upper, per, f.start[cls], cls, ncls, ncls > 1 ? f.start[cls + 1] - f.start[cls] : 0u);
  };
  (apart ? sum : wave).add(SEC_SUM, n_tiles, 1, 0);
  add(wave, SEC_W2, 1, CLS_LDS_W2);
  add(wave, SEC_W6, 1, CLS_LDS_W6);
  add(wave, SEC_W1, 1, CLS_LDS_W1);
  add(wave, SEC_G32X, 64 / SHAPE_G32X.lanes, CLS_G32X);
  add(wave, SEC_G32S, 64 / SHAPE_G32S.lanes, CLS_G32S);
  add(wave, SEC_G32, 64 / SHAPE_G32.lanes, CLS_G32);
  add(wave, SEC_G16, 64 / SHAPE_G16.lanes, CLS_G16);
  add(wave, SEC_G8, 64 / SHAPE_G8.lanes, CLS_G8);
  add(wave, SEC_G4, 64 / SHAPE_G4.lanes, CLS_G4);
  add(wave, SEC_G2, 64 / SHAPE_G2.lanes, CLS_G2);
  add(wave, SEC_TINY, 64, CLS_TINY);
  (apart ? totals : pair).add(SEC_TOTALS, n_tiles, 2, 0);
  add(pair, SEC_P8, 1, CLS_MW2);
  add(pair, SEC_P6, 1, CLS_MW2_6);
  (apart ? scan : wide).add(SEC_SCAN, n_trows, 1, 0);
  if (f.tiled_from > CLS_STREAM) add(wide, SEC_STREAM, 1, CLS_STREAM);
  if (f.tiled_from > CLS_STREAM_LAST) add(wide, SEC_STREAM, 1, CLS_STREAM_LAST);
  add(wide, SEC_STREAM, 1, CLS_HOLD);
  add(wide, SEC_B10, 1, CLS_MW2 + 7, 2);
  const bool longer = block_takes_longer(g, f.tiled_from);
  if (streams_by_queue(g, f.tiled_from, longer)) {
    wide.a.next = counts + CLS_COUNT;
    if (again) hipLaunchKernelGGL(clear_taken_kernel, dim3(1), dim3(1), 0, g->stream, wide.a.next);
  }
  if (longer) {
    add(wide, SEC_B8, 1, CLS_MW2 + 6);
  } else {
    add(wide, SEC_B8, 1, CLS_MW2 + 5, 2);
    add(wide, SEC_B6, 1, CLS_MW2 + 4);
  }
  (apart ? emit : block).add(SEC_EMIT, n_tiles, 1, 0);
  if (longer) add(block, SEC_M14, 1, CLS_MW2 + 4, 2);
  add(block, SEC_M10, 1, CLS_MW2 + 3);
  add(block, SEC_M8, 1, CLS_MW2 + 2);
  add(block, SEC_M6, 1, CLS_MW2 + 1);
  if (!apart) {
    for (const Launch* l : {&wave, &pair, &wide, &block}) SKY_TRY(enqueue<true>(p, *l, longer, g->stream));
    return SKY_OK;
  }
  SKY_TRY(enqueue<true>(p, sum, longer, g->stream));
  auto others = [&]() -> int {
    SKY_TRY(beside_fork(&side, 0));
    for (const Launch* l : {&wide, &block, &pair, &wave}) SKY_TRY(enqueue<true>(p, *l, longer, side.stream[0]));
    for (const Launch* l : {&totals, &scan, &emit}) SKY_TRY(enqueue<true>(p, *l, false, g->stream));
    return beside_join(&side);
  };
  const int rc = others();
  if (rc != SKY_OK) beside_drop(&side);
  return rc;
}

}  // namespace sky
