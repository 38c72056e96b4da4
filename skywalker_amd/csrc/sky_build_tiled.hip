// Alias tables of rows too long for one workgroup's LDS, built tile by tile by the whole GPU.
//
// A row is cut into tiles of 1024 slots counted from its 16-byte aligned start.  The table is the
// same pure function of the weights as everywhere else (see sky_build.hip); only the evaluation
// order changes:
//   tiled_sum_kernel      per tile   exact 128-bit partial sum of the weights
//   tiled_ledger_kernel   per row    total -> scale and fraction bits
//   tiled_totals_kernel   per tile   sum of deficits, sum of surpluses, first and last heavy
//   tiled_scan_kernel     per row    exclusive prefix of the tile totals (BL, BH), next heavy after each tile
//   tiled_emit_kernel     per tile   every entry of the tile
// In the last step a light with exclusive deficit prefix x needs the first slot whose surplus prefix
// exceeds x.  The tile holding that slot ("partner") follows from BH; its per-slot prefix is
// recomputed from the weights into LDS and searched there.  Heavies look up their retiring
// light the same way against BL.  Lights and heavies of a tile are monotone in their keys, so the
// partners of one tile are a contiguous run and the total number of (tile, partner) pairs of a row
// is at most twice its tile count: no per-slot scratch in global memory, O(1) passes over the weights.
#include <algorithm>

#include "sky_build_tile.h"

namespace sky {

// ---------------------------------------------------------------- row and tile bookkeeping
struct TiledCounters {
  unsigned long long next;  // low 32 bits: tiles handed out; high 32 bits: rows handed out
  uint32_t skipped;         // rows with more tiles than the path accepts (left to the streaming kernel)
  uint32_t pad;
};

// Geometry of every row; each block reserves a run of tile ids (and of prefix-array slots) for its
// rows with one atomic.  Tile numbering therefore depends on scheduling; no result does.
__global__ __launch_bounds__(256) void tiled_rows_kernel(const RowRef* __restrict__ vlist, uint32_t count,
                                                         const uint32_t* __restrict__ xadj, uint32_t max_tiles,
                                                         TiledRow* __restrict__ rows,
                                                         TiledCounters* __restrict__ ctr) {
  __shared__ uint32_t s_w[4];
  __shared__ unsigned long long s_base;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint32_t r = blockIdx.x * 256u + tid;
  TiledRow row = {};
  uint32_t nt = 0;
  bool skip = false;
  if (r < count) {
    row.v = vlist[r].v;
    row.off = xadj[row.v];
    row.d = xadj[row.v + 1] - row.off;
    row.base = row.off & ~3u;
    row.lead = row.off - row.base;
    row.span = row.lead + row.d;
    nt = (row.span + TILE - 1) / TILE;
    if (nt > max_tiles) {
      nt = 0;
      skip = true;
    }
    row.ntiles = nt;
  }
  const uint32_t inc = group_scan_u32<64>(nt);
  const uint32_t nskip = __popcll(__ballot(skip));
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  uint32_t before = 0, total = 0;
  for (int k = 0; k < 4; ++k) {
    if (k == wave) before = total;
    total += s_w[k];
  }
  if (tid == 0) s_base = atomicAdd(&ctr->next, ((unsigned long long)256u << 32) | total);
  if (lane == 0 && nskip) atomicAdd(&ctr->skipped, nskip);
  __syncthreads();
  if (r < count) {
    row.tile0 = (uint32_t)s_base + before + inc - nt;
    row.bofs = row.tile0 + (uint32_t)(s_base >> 32) + tid;  // every row owns ntiles + 1 prefix slots
    rows[r] = row;
  }
}

__global__ __launch_bounds__(256) void tiled_map_kernel(const TiledRow* __restrict__ rows, uint32_t count,
                                                        TileGeom* __restrict__ geom) {
  const uint32_t r = blockIdx.x;
  if (r >= count) return;
  const TiledRow row = rows[r];
  for (uint32_t t = threadIdx.x; t < row.ntiles; t += 256)
    geom[row.tile0 + t] = TileGeom{r, t, row.base, row.lead, row.span, {0, 0, 0}};
}

// ---------------------------------------------------------------- pass 1: exact sums
__global__ __launch_bounds__(TL_T) void tiled_sum_kernel(const TileGeom* __restrict__ geom,
                                                         const float* __restrict__ wgt, u128* __restrict__ tsum) {
  __shared__ WSum3 s_w[TL_T / 64];
  const uint32_t tile = blockIdx.x;
  const TileGeom tg = geom[tile];
  if (tg.span == 0) return;  // the grid may be larger than the number of tiles
  const TiledRow r = geom_row(tg, tile);
  const int tid = threadIdx.x;
  float w[TL_Q][4];
  load_tile(wgt, r, tg.T, tid, w);
  WSum3 sum{0.0, 0.0, 0.0};  // exact: a tile adds at most 1024 limbs below 2^32 + 1
#pragma unroll
  for (int q = 0; q < TL_Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) wsum3_add(sum, (double)w[q][k]);
  sum = group_sum_wsum3<64>(sum);
  if ((tid & 63) == 0) s_w[tid >> 6] = sum;
  __syncthreads();
  if (tid == 0) {
    WSum3 s = s_w[0];
    for (int i = 1; i < TL_T / 64; ++i) {
      s.top += s_w[i].top;
      s.mid += s_w[i].mid;
      s.low += s_w[i].low;
    }
    tsum[tile] = wsum3_to_u128(s);
  }
}

__global__ __launch_bounds__(64) void tiled_ledger_kernel(TiledRow* __restrict__ rows, uint32_t count,
                                                          const u128* __restrict__ tsum) {
  const uint32_t r = blockIdx.x;
  if (r >= count) return;
  const uint32_t t0 = rows[r].tile0, nt = rows[r].ntiles, d = rows[r].d;
  if (nt == 0) return;
  u128 sum{0, 0};
  for (uint32_t t = threadIdx.x; t < nt; t += 64) sum = add128(sum, tsum[t0 + t]);
  sum = group_sum_u128<64>(sum);
  if (threadIdx.x == 0) {
    const bool ok = (sum.lo | sum.hi) != 0;
    rows[r].ok = ok;
    if (ok) {
      const Ledger L = make_ledger(d, sum);
      rows[r].scale = L.scale;
      rows[r].fs = L.fs;
      rows[r].inv_fs = L.inv_fs;
      rows[r].one = L.one;
    }
  }
}

// ---------------------------------------------------------------- pass 2: tile totals
__global__ __launch_bounds__(TL_T) void tiled_totals_kernel(const TileGeom* __restrict__ geom,
                                                            const TiledRow* __restrict__ rows,
                                                            const float* __restrict__ wgt,
                                                            TileTotals* __restrict__ ttot) {
  __shared__ uint64_t s_d[TL_T / 64], s_u[TL_T / 64];
  __shared__ uint32_t s_f[TL_T / 64], s_l[TL_T / 64];
  const uint32_t tile = blockIdx.x;
  const TileGeom tg = geom[tile];
  if (tg.span == 0) return;
  const int tid = threadIdx.x;
  const uint32_t t = tg.T;
  float w[TL_Q][4];
  load_tile(wgt, geom_row(tg, tile), t, tid, w);  // requested before the row's ledger arrives
  const TiledRow r = rows[tg.row];
  if (!r.ok) return;
  const Ledger L = row_ledger(r);
  uint64_t sd = 0, su = 0;
  uint32_t fh = NONE32, lh = 0;  // lh holds idx + 1 so that 0 means none
  auto add_up = [&](auto may_wrap) {
    constexpr bool SAT = decltype(may_wrap)::value;
#pragma unroll
    for (int q = 0; q < TL_Q; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t idx = t * TILE + 4u * (q * TL_T + tid) + k;
        if (!in_row(r, idx)) continue;
        const Entry e = classify_fast((double)w[q][k], true, L);
        if (e.heavy) {
          su = add_sat<SAT>(su, e.amount);
          fh = min(fh, idx);
          lh = max(lh, idx + 1);
        } else {
          sd += e.amount;
        }
      }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      sd += shfl_xor_u64(sd, m);
      su = add_sat<SAT>(su, shfl_xor_u64(su, m));
      fh = min(fh, (uint32_t)__shfl_xor((int)fh, m, 64));
      lh = max(lh, (uint32_t)__shfl_xor((int)lh, m, 64));
    }
  };
  if (surpluses_may_wrap(L.scale)) add_up(std::true_type{});
  else add_up(std::false_type{});
  if ((tid & 63) == 0) {
    s_d[tid >> 6] = sd;
    s_u[tid >> 6] = su;
    s_f[tid >> 6] = fh;
    s_l[tid >> 6] = lh;
  }
  __syncthreads();
  if (tid == 0) {
    TileTotals o{0, 0, NONE32, 0};
    for (int i = 0; i < TL_T / 64; ++i) {
      o.d += s_d[i];
      o.u = add_sat(o.u, s_u[i]);
      o.first_heavy = min(o.first_heavy, s_f[i]);
      o.last_heavy = max(o.last_heavy, s_l[i]);
    }
    o.last_heavy = o.last_heavy ? o.last_heavy - 1 : NONE32;
    ttot[tile] = o;
  }
}

// ---------------------------------------------------------------- per row: bases and partner ranges of its tiles
constexpr int TS_T = 1024;
__global__ __launch_bounds__(TS_T) void tiled_scan_kernel(TiledRow* __restrict__ rows, uint32_t count,
                                                          const TileTotals* __restrict__ ttot,
                                                          uint64_t* __restrict__ BL, uint64_t* __restrict__ BH,
                                                          uint32_t* __restrict__ nfh, uint4* __restrict__ ranges) {
  __shared__ TileScanLds<TS_T> lds;
  if (blockIdx.x >= count) return;
  tile_scan_row<TS_T>(rows, blockIdx.x, ttot, BL, BH, nfh, ranges, lds);
}

// ---------------------------------------------------------------- pass 3: every entry of a tile
__global__ __launch_bounds__(TL_T) void tiled_emit_kernel(const TileGeom* __restrict__ geom,
                                                          const TiledRow* __restrict__ rows,
                                                          const float* __restrict__ wgt,
                                                          const uint64_t* __restrict__ gBL,
                                                          const uint64_t* __restrict__ gBH,
                                                          const uint32_t* __restrict__ nfh,
                                                          const uint4* __restrict__ ranges,
                                                          AliasEntry* __restrict__ table,
                                                          int8_t* __restrict__ valid) {
  __shared__ TileEmitLds lds;
  const uint32_t tile = blockIdx.x;
  const TileGeom tg = geom[tile];
  if (tg.span == 0) return;
  tile_emit(tg, tile, rows, wgt, gBL, gBH, nfh, ranges, table, valid, lds);
}

// ---------------------------------------------------------------- host driver
namespace {
struct TiledScratch {
  TiledRow* rows = nullptr;
  TiledCounters* totals = nullptr;
  TileGeom* geom = nullptr;
  u128* tsum = nullptr;
  TileTotals* ttot = nullptr;
  uint64_t *BL = nullptr, *BH = nullptr;
  uint32_t* nfh = nullptr;
  uint4* ranges = nullptr;
  uint32_t row_cap = 0, tile_cap = 0;
  size_t b_cap = 0;  // entries of BL and BH
};
TiledScratch& tiled_of(sky_graph* g) {
  if (!g->tiled_scratch) g->tiled_scratch = new TiledScratch();
  return *static_cast<TiledScratch*>(g->tiled_scratch);
}
}  // namespace

void free_tiled_scratch(sky_graph* g) {
  if (!g->tiled_scratch) return;
  TiledScratch* sc = static_cast<TiledScratch*>(g->tiled_scratch);
  void* ptrs[] = {sc->rows, sc->totals, sc->geom, sc->tsum, sc->ttot, sc->BL, sc->BH, sc->nfh, sc->ranges};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  delete sc;
  g->tiled_scratch = nullptr;
}

uint32_t tiled_max_tiles(const sky_graph* g) {
  const long long n = option(g, OPT_TILED_MAX_TILES);
  return (uint32_t)std::min<long long>(std::max<long long>(n, 1), TILED_MAX_TILES);
}

// Builds the rows of `rows_list` (device, n entries) that have at most the configured number of
// tiles; *skipped receives how many rows were left for the streaming kernel.  `edges` is the number of
// entries of the listed rows when the caller knows it (0 otherwise): the tile grids are then sized by
// the bound edges / TILE + 2 n, with empty records for the tiles that do not exist, and the host does
// not wait for the device to count them.
int build_rows_tiled(sky_graph* g, const RowRef* rows_list, uint32_t n, uint32_t* skipped, EventTimer* tm, uint64_t edges) {
  hipStream_t st = g->stream;
  TiledScratch& sc = tiled_of(g);
  const uint32_t max_tiles = tiled_max_tiles(g);
  *skipped = 0;
  if (n == 0) return SKY_OK;
  if (sc.row_cap < n) {
    if (sc.rows) SKY_HIP(hipFree(sc.rows));
    sc.rows = nullptr;
    sc.row_cap = 0;
    SKY_HIP(hipMalloc((void**)&sc.rows, (size_t)n * sizeof(TiledRow)));
    sc.row_cap = n;
  }
  if (!sc.totals) SKY_HIP(hipMalloc((void**)&sc.totals, sizeof(TiledCounters)));
  SKY_HIP(hipMemsetAsync(sc.totals, 0, sizeof(TiledCounters), st));
  hipLaunchKernelGGL(tiled_rows_kernel, dim3((n + 255) / 256), dim3(256), 0, st, rows_list, n, g->xadj,
                     max_tiles, sc.rows, sc.totals);
  const bool bounded = edges != 0 && max_tiles == TILED_MAX_TILES && edges / TILE + 2ull * n < (1ull << 31);
  uint32_t ntiles, nslots;
  if (bounded) {
    ntiles = (uint32_t)(edges / TILE + 2ull * n);
    nslots = 256u * ((n + 255) / 256);
  } else {
    TiledCounters totals = {};
    SKY_HIP(hipMemcpyAsync(&totals, sc.totals, sizeof(totals), hipMemcpyDeviceToHost, st));
    SKY_HIP(hipStreamSynchronize(st));
    ntiles = (uint32_t)totals.next;
    nslots = (uint32_t)(totals.next >> 32);  // 256 per block of rows
    *skipped = totals.skipped;
  }
  if (ntiles == 0) return SKY_OK;
  if (sc.tile_cap < ntiles) {
    void* olds[] = {sc.geom, sc.tsum, sc.ttot, sc.nfh, sc.ranges};
    for (void* p : olds)
      if (p) SKY_HIP(hipFree(p));
    sc.geom = nullptr; sc.tsum = nullptr; sc.ttot = nullptr; sc.nfh = nullptr; sc.ranges = nullptr;
    sc.tile_cap = 0;
    const size_t cap = (size_t)ntiles + ntiles / 4 + 1024;
    SKY_HIP(hipMalloc((void**)&sc.geom, cap * sizeof(TileGeom)));
    SKY_HIP(hipMalloc((void**)&sc.tsum, cap * sizeof(u128)));
    SKY_HIP(hipMalloc((void**)&sc.ttot, cap * sizeof(TileTotals)));
    SKY_HIP(hipMalloc((void**)&sc.nfh, cap * 4));
    SKY_HIP(hipMalloc((void**)&sc.ranges, cap * sizeof(uint4)));
    sc.tile_cap = (uint32_t)cap;
  }
  // prefix arrays hold ntiles + one extra entry per row
  const size_t b_need = (size_t)ntiles + nslots;
  if (sc.b_cap < b_need) {
    if (sc.BL) SKY_HIP(hipFree(sc.BL));
    if (sc.BH) SKY_HIP(hipFree(sc.BH));
    sc.BL = sc.BH = nullptr;
    sc.b_cap = 0;
    SKY_HIP(hipMalloc((void**)&sc.BL, (b_need + b_need / 4 + 1024) * 8));
    SKY_HIP(hipMalloc((void**)&sc.BH, (b_need + b_need / 4 + 1024) * 8));
    sc.b_cap = b_need + b_need / 4 + 1024;
  }
  if (bounded) SKY_HIP(hipMemsetAsync(sc.geom, 0, (size_t)ntiles * sizeof(TileGeom), st));  // span 0: no such tile
  hipLaunchKernelGGL(tiled_map_kernel, dim3(n), dim3(256), 0, st, sc.rows, n, sc.geom);
  if (tm) SKY_TRY(tm->mark("tiled_rows", 0));
  hipLaunchKernelGGL(tiled_sum_kernel, dim3(ntiles), dim3(TL_T), 0, st, sc.geom, g->adjwgt, sc.tsum);
  if (tm) SKY_TRY(tm->mark("tiled_sum", edges));
  hipLaunchKernelGGL(tiled_ledger_kernel, dim3(n), dim3(64), 0, st, sc.rows, n, sc.tsum);
  hipLaunchKernelGGL(tiled_totals_kernel, dim3(ntiles), dim3(TL_T), 0, st, sc.geom, sc.rows, g->adjwgt, sc.ttot);
  if (tm) SKY_TRY(tm->mark("tiled_totals", edges));
  hipLaunchKernelGGL(tiled_scan_kernel, dim3(n), dim3(TS_T), 0, st, sc.rows, n, sc.ttot, sc.BL, sc.BH, sc.nfh, sc.ranges);
  hipLaunchKernelGGL(tiled_emit_kernel, dim3(ntiles), dim3(TL_T), 0, st, sc.geom, sc.rows, g->adjwgt, sc.BL,
                     sc.BH, sc.nfh, sc.ranges, g->table, g->valid);
  if (tm) SKY_TRY(tm->mark("tiled_emit", edges));
  return SKY_OK;
}

}  // namespace sky
