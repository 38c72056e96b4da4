// Tiles of the rows that the whole GPU builds together (the passes are described in sky_build_tiled.hip): geometry, the
// scan over a row's tiles and the entries of a tile.
#pragma once
#include "sky_build_common.h"
#include "sky_graph.h"

namespace sky {

constexpr int TL_T = 256;                // threads per tile
constexpr int TL_Q = 1;                  // float4 quads per thread
constexpr int TILE = TL_T * 4 * TL_Q;    // slots per tile
static_assert(TILE == (int)TILED_TILE, "tile size is part of the dispatch contract");
constexpr uint32_t TILED_MAX_TILES = 1u << 22;  // rows of more tiles (4G entries) cannot exist with 32-bit offsets

struct TiledRow {
  uint32_t v, off, d, base, lead, span, ntiles, tile0, bofs;  // tile0: first tile id; bofs: first slot of the row's BL/BH
  double scale, fs, inv_fs;
  uint64_t one, total_h;
  uint32_t ok, last_heavy;  // last_heavy: span index
  uint32_t active;          // builds of a frontier: whether the row is among those that the build makes
};
struct TileTotals {
  uint64_t d, u;
  uint32_t first_heavy, last_heavy;  // span indices, NONE32 when the tile has no heavy
};

// Where a tile lies, one aligned record per tile: a tile's weights can be requested after one
// dependent load instead of two (tile -> row -> geometry).
struct __attribute__((aligned(32))) TileGeom {
  uint32_t row, T, base, lead, span, pad[3];  // row: index into the row array; T: tile number inside the row
};
__device__ __forceinline__ TiledRow geom_row(const TileGeom& tg, uint32_t tile) {
  TiledRow r = {};
  r.base = tg.base;
  r.lead = tg.lead;
  r.span = tg.span;
  r.tile0 = tile - tg.T;
  return r;
}

__device__ __forceinline__ Ledger row_ledger(const TiledRow& r) {
  Ledger L;
  L.scale = r.scale;
  L.fs = r.fs;
  L.inv_fs = r.inv_fs;
  L.one = r.one;
  return L;
}

// Weights of tile `t` of a row: quad q of thread tid covers span slots 4*(q*TL_T + tid) + t*TILE ...+3.
__device__ __forceinline__ void load_tile(const float* __restrict__ wgt, const TiledRow& r, uint32_t t, int tid,
                                          float (&w)[TL_Q][4]) {
#pragma unroll
  for (int q = 0; q < TL_Q; ++q) {
    const uint32_t pos = t * TILE + 4u * (q * TL_T + tid);
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pos < r.span) x = *reinterpret_cast<const float4*>(wgt + r.base + pos);
    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t idx = pos + k;
      w[q][k] = idx - r.lead < r.span - r.lead ? clamp_weight(xs[k]) : 0.0f;
    }
  }
}
__device__ __forceinline__ bool in_row(const TiledRow& r, uint32_t idx) { return idx - r.lead < r.span - r.lead; }

// first t in [0, nt) with B[t + 1] > key (nt if none)
__device__ __forceinline__ uint32_t first_tile_above(const uint64_t* B, uint32_t nt, uint64_t key) {
  return first_greater(B + 1, 0, nt, key);
}

// Per row: BL[t], BH[t] = deficits / surpluses before tile t (t = 0..ntiles, the last entry is the
// row total), stored at index tile0 + row + t; nfh[tile] = first heavy in any later tile.  One workgroup
// of T threads per row: a row of a million entries has a thousand tiles, and one wavefront walking
// them 64 at a time with dependent loads was a sixth of a millisecond on the critical path.
template <int T>
struct TileScanLds {
  uint64_t s_wl[T / 64], s_wh[T / 64];
  uint32_t s_wm[T / 64];
};
template <int TS_T, bool SAT>
__device__ __forceinline__ void tile_scan_row(TiledRow* __restrict__ rows, uint32_t r, const TileTotals* __restrict__ ttot,
                                              uint64_t* __restrict__ BL, uint64_t* __restrict__ BH,
                                              uint32_t* __restrict__ nfh, uint4* __restrict__ ranges,
                                              TileScanLds<TS_T>& lds) {
  constexpr int NW = TS_T / 64;
  auto& s_wl = lds.s_wl;
  auto& s_wh = lds.s_wh;
  auto& s_wm = lds.s_wm;
  const uint32_t t0 = rows[r].tile0, nt = rows[r].ntiles;
  if (nt == 0 || !rows[r].ok) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t b0 = rows[r].bofs;
  uint64_t cl = 0, ch = 0;
  uint32_t last = NONE32;
  for (uint32_t c = 0; c < nt; c += TS_T) {
    const uint32_t t = c + tid;
    uint64_t d = 0, u = 0;
    uint32_t lh = 0;
    if (t < nt) {
      const TileTotals x = ttot[t0 + t];
      d = x.d;
      u = x.u;
      lh = x.last_heavy == NONE32 ? 0 : x.last_heavy + 1;
    }
    const uint64_t il = group_scan_u64<64>(d), ih = group_scan_sat_u64<64, SAT>(u);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) lh = max(lh, (uint32_t)__shfl_xor((int)lh, m, 64));
    if (lane == 63) {
      s_wl[wave] = il;
      s_wh[wave] = ih;
      s_wm[wave] = lh;
    }
    __syncthreads();
    uint64_t bl = cl, bh = ch, tl = 0, th = 0;
    uint32_t lm = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (w == wave) {
        bl += tl;
        bh = add_sat<SAT>(bh, th);
      }
      tl += s_wl[w];
      th = add_sat<SAT>(th, s_wh[w]);
      lm = max(lm, s_wm[w]);
    }
    const uint64_t eh = before_own<SAT>(ih, u);  // all lanes together
    if (t < nt) {
      BL[b0 + t] = bl + il - d;
      BH[b0 + t] = add_sat<SAT>(bh, eh);
    }
    cl += tl;
    ch = add_sat<SAT>(ch, th);
    if (lm) last = lm - 1;
    __syncthreads();  // the wavefront totals are rewritten by the next round
  }
  // next first heavy: the tiles backwards, exclusive suffix minimum of first_heavy
  uint32_t carry = NONE32;
  for (int32_t c = (int32_t)((nt - 1) / TS_T * TS_T); c >= 0; c -= TS_T) {
    const uint32_t t = (uint32_t)c + tid;
    const uint32_t fh = t < nt ? ttot[t0 + t].first_heavy : NONE32;
    uint32_t suf = fh;  // inclusive suffix minimum over the lanes of the wavefront
#pragma unroll
    for (int dlt = 1; dlt < 64; dlt <<= 1) {
      const uint32_t o = (uint32_t)__shfl_down((int)suf, dlt, 64);
      if (lane + dlt < 64) suf = min(suf, o);
    }
    uint32_t excl = (uint32_t)__shfl_down((int)suf, 1, 64);
    if (lane == 63) excl = NONE32;
    if (lane == 0) s_wm[wave] = suf;  // minimum of the wavefront
    __syncthreads();
    uint32_t later = carry, all = carry;  // minimum over the later wavefronts of this round and the later rounds
#pragma unroll
    for (int w = NW - 1; w >= 0; --w) {
      if (w == wave) later = all;
      all = min(all, s_wm[w]);
    }
    if (t < nt) nfh[t0 + t] = min(excl, later);
    carry = all;
    __syncthreads();
  }
  if (tid == 0) {
    BL[b0 + nt] = cl;
    BH[b0 + nt] = ch;
    rows[r].total_h = ch;
    rows[r].last_heavy = last;
  }
  // partner tiles of every tile: lights of tile t (keys in [BL[t], BL[t+1]]) meet the tiles whose surplus
  // range holds those keys; heavies (y in (BH[t], BH[t+1]]) the tiles whose deficit range holds y
  __threadfence_block();
  __syncthreads();
  const uint64_t* rl = BL + b0;
  const uint64_t* rh = BH + b0;
  for (uint32_t t = tid; t < nt; t += TS_T) {
    uint4 g;
    g.x = first_tile_above(rh, nt, rl[t]);
    g.y = min(first_tile_above(rh, nt, rl[t + 1]), nt - 1);
    if (rh[t + 1] != rh[t]) {
      g.z = first_tile_above(rl, nt, rh[t]);
      g.w = min(first_tile_above(rl, nt, rh[t + 1] - 1), nt - 1);
    } else {
      g.z = 1;
      g.w = 0;
    }
    ranges[t0 + t] = g;
  }
}

template <int TS_T>
__device__ __forceinline__ void tile_scan_row(TiledRow* __restrict__ rows, uint32_t r, const TileTotals* __restrict__ ttot,
                                              uint64_t* __restrict__ BL, uint64_t* __restrict__ BH,
                                              uint32_t* __restrict__ nfh, uint4* __restrict__ ranges,
                                              TileScanLds<TS_T>& lds) {
  if (surpluses_may_wrap(rows[r].scale)) tile_scan_row<TS_T, true>(rows, r, ttot, BL, BH, nfh, ranges, lds);
  else tile_scan_row<TS_T, false>(rows, r, ttot, BL, BH, nfh, ranges, lds);
}

// ---------------------------------------------------------------- pass 3: every entry of a tile
// Resolves the own entries of one kind whose key lies in [lo, hi) against the per-slot prefix of tile
// `pt` held in smem[0..TILE).  OWN_HEAVY = false: lights, key = exclusive deficit prefix, prefix = surplus.
// OWN_HEAVY = true: heavies, key = y - 1, prefix = deficit.
template <bool OWN_HEAVY>
__device__ __forceinline__ void resolve_in_tile(const TiledRow& r, const Ledger& L, const uint64_t* smem, uint32_t pt,
                                                uint64_t lo, uint64_t hi, uint32_t heavy_mask, uint32_t live_mask,
                                                const uint32_t (&nh_after)[TL_Q], uint32_t T,
                                                const uint64_t (&key)[TL_Q][4], float (&op)[TL_Q][4],
                                                uint32_t (&oa)[TL_Q][4]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < TL_Q; ++q) {
    uint32_t mine = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int b = q * 4 + k;
      const bool kind = ((live_mask >> b) & 1) && (((heavy_mask >> b) & 1) != 0) == OWN_HEAVY;
      if (kind && key[q][k] >= lo && key[q][k] < hi) mine |= 1u << k;
    }
    if (!mine) continue;
    const uint32_t base[4] = {0, 0, 0, 0};
    uint32_t pos[4];
    search4(smem, base, key[q], (uint32_t)TILE, pos);
    if (OWN_HEAVY) {
      // next heavy after each slot of the quad; the row's last heavy never retires
      uint32_t nxt = nh_after[q];
#pragma unroll
      for (int k = 3; k >= 0; --k) {
        if (((mine >> k) & 1) && nxt != NONE32) {
          op[q][k] = residual_prob(L.one + key[q][k] + 1 - smem[pos[k]], L);
          oa[q][k] = nxt - r.lead;
        }
        if ((heavy_mask >> (q * 4 + k)) & 1) nxt = T * TILE + 4u * (q * TL_T + tid) + k;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if ((mine >> k) & 1) oa[q][k] = pt * TILE + pos[k] - r.lead;
    }
  }
}

// One pass over the partner tiles of one kind other than the own tile T: their per-slot prefix is
// recomputed from the weights into LDS.
template <bool OWN_HEAVY>
__device__ __forceinline__ void partner_pass(const TiledRow& r, const Ledger& L, const float* __restrict__ wgt,
                                             const uint64_t* __restrict__ B, uint32_t t_lo, uint32_t t_hi,
                                             uint64_t* smem,
                                             uint64_t* s_ex, uint32_t heavy_mask, uint32_t live_mask,
                                             const uint32_t (&nh_after)[TL_Q], uint32_t T,
                                             const uint64_t (&key)[TL_Q][4], float (&op)[TL_Q][4],
                                             uint32_t (&oa)[TL_Q][4]) {
  const int tid = threadIdx.x;
  const uint32_t nt = r.ntiles;
  for (uint32_t pt = t_lo; pt <= t_hi && pt < nt; ++pt) {
    const uint64_t lo = B[pt], hi = B[pt + 1];
    if (hi == lo || pt == T) continue;
    float pw[TL_Q][4];
    load_tile(wgt, r, pt, tid, pw);
    uint64_t pv[TL_Q][4], ps[TL_Q][4];
#pragma unroll
    for (int q = 0; q < TL_Q; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t idx = pt * TILE + 4u * (q * TL_T + tid) + k;
        const Entry e = classify_fast((double)pw[q][k], in_row(r, idx), L);
        pv[q][k] = e.heavy != OWN_HEAVY ? e.amount : 0;
      }
    __syncthreads();  // searches of the previous partner are done: s_ex and the prefix may be overwritten
    if (!OWN_HEAVY && surpluses_may_wrap(L.scale)) block_scan1<TL_T, TL_Q, true>(pv, s_ex, lo, ps);
    else block_scan1<TL_T, TL_Q, false>(pv, s_ex, lo, ps);
#pragma unroll
    for (int q = 0; q < TL_Q; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) smem[4u * (q * TL_T + tid) + k] = ps[q][k];
    __syncthreads();
    resolve_in_tile<OWN_HEAVY>(r, L, smem, pt, lo, hi, heavy_mask, live_mask, nh_after, T, key, op, oa);
  }
}

struct TileEmitLds {
  uint64_t smem[TILE];  // per-slot prefix of the current partner tile
  uint64_t s_ex[2 * TL_Q * (TL_T / 64)];
  uint32_t s_fh[TL_Q][TL_T / 64];
};
// Every entry of tile `tile` (tg.span not 0) by TL_T threads.
__device__ __forceinline__ void tile_emit(const TileGeom& tg, uint32_t tile, const TiledRow* __restrict__ rows,
                                          const float* __restrict__ wgt, const uint64_t* __restrict__ gBL,
                                          const uint64_t* __restrict__ gBH, const uint32_t* __restrict__ nfh,
                                          const uint4* __restrict__ ranges, AliasEntry* __restrict__ table,
                                          int8_t* __restrict__ valid, TileEmitLds& lds) {
  constexpr int NW = TL_T / 64;
  auto& smem = lds.smem;
  auto& s_ex = lds.s_ex;
  auto& s_fh = lds.s_fh;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint32_t T = tg.T;

  float w[TL_Q][4];
  load_tile(wgt, geom_row(tg, tile), T, tid, w);  // requested before the row record arrives
  const TiledRow r = rows[tg.row];
  if (!r.ok) {
#pragma unroll
    for (int q = 0; q < TL_Q; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t idx = T * TILE + 4u * (q * TL_T + tid) + k;
        if (in_row(r, idx)) {
          table[r.base + idx] = AliasEntry{0.0f, SKY_INVALID};
        }
      }
    if (T == 0 && tid == 0) valid[r.v] = 0;
    return;
  }
  if (T == 0 && tid == 0) valid[r.v] = 1;
  const Ledger L = row_ledger(r);
  const uint64_t* BL = gBL + r.bofs;  // tile prefixes of this row
  const uint64_t* BH = gBH + r.bofs;
  const uint64_t bl = BL[T], bl1 = BL[T + 1], bh = BH[T], bh1 = BH[T + 1];
  const uint4 rg = ranges[tile];

  // own tile: class and amount of every slot, both prefixes, search key of the own kind
  uint64_t key[TL_Q][4], sl[TL_Q][4], sh[TL_Q][4];
  float op[TL_Q][4];
  uint32_t oa[TL_Q][4];
  uint32_t heavy_mask = 0, live_mask = 0;
  uint64_t hb_mask[TL_Q];
  {
    uint64_t dl[TL_Q][4], dh[TL_Q][4];
#pragma unroll
    for (int q = 0; q < TL_Q; ++q) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t idx = T * TILE + 4u * (q * TL_T + tid) + k;
        const bool in = in_row(r, idx);
        const Entry e = classify_fast((double)w[q][k], in, L);
        dl[q][k] = e.heavy ? 0 : e.amount;
        dh[q][k] = e.heavy ? e.amount : 0;
        op[q][k] = e.heavy ? 1.0f : (float)e.p;
        if (in) live_mask |= 1u << (q * 4 + k);
        if (e.heavy) heavy_mask |= 1u << (q * 4 + k);
      }
      const uint32_t m = (heavy_mask >> (q * 4)) & 15u;
      const uint64_t bal = __ballot(m != 0);
      hb_mask[q] = bal;
      uint32_t fh = NONE32;
      if (bal) {
        const int l0 = __ffsll((unsigned long long)bal) - 1;
        const uint32_t m0 = (uint32_t)__builtin_amdgcn_readlane((int)m, l0);
        fh = T * TILE + 4u * (q * TL_T + wave * 64 + l0) + (uint32_t)(__ffs((int)m0) - 1);
      }
      if (lane == 0) s_fh[q][wave] = fh;
    }
    uint64_t tl, th;
    const bool may_wrap = surpluses_may_wrap(L.scale);
    block_scan2<TL_T, TL_Q>(may_wrap, dl, dh, s_ex, sl, sh, tl, th);  // its barrier also publishes s_fh
#pragma unroll
    for (int q = 0; q < TL_Q; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint64_t inside = sh[q][k];
        sl[q][k] += bl;
        sh[q][k] += bh;
        if (may_wrap) {
          asm volatile("");  // a branch, not a select in every row
          sh[q][k] = add_sat(inside, bh);
        }
        key[q][k] = ((heavy_mask >> (q * 4 + k)) & 1) ? sh[q][k] - 1 : sl[q][k] - dl[q][k];
      }
  }
  // next heavy after each quad (span index): later lanes, later waves, later sub-tiles, later tiles
  uint32_t nh_after[TL_Q];
  {
    const uint32_t later_tiles = nfh[tile];
#pragma unroll
    for (int q = 0; q < TL_Q; ++q) {
      const uint32_t m = (heavy_mask >> (q * 4)) & 15u;
      const uint64_t above = hb_mask[q] & ~((2ull << lane) - 1);
      const int ln = above ? __ffsll((unsigned long long)above) - 1 : lane;
      const uint32_t mn = (uint32_t)__shfl((int)m, ln, 64);
      uint32_t nx = above ? T * TILE + 4u * (q * TL_T + wave * 64 + ln) + (uint32_t)(__ffs((int)mn) - 1) : later_tiles;
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) {
        if (wv > wave) nx = min(nx, s_fh[q][wv]);
#pragma unroll
        for (int q2 = q + 1; q2 < TL_Q; ++q2) nx = min(nx, s_fh[q2][wv]);
      }
      nh_after[q] = nx;
    }
  }
  // defaults: a light without donor takes the last heavy (itself if the row has none);
  // a heavy that is last, or that no light retires, keeps {1, itself}
#pragma unroll
  for (int q = 0; q < TL_Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t idx = T * TILE + 4u * (q * TL_T + tid) + k;
      const bool heavy = (heavy_mask >> (q * 4 + k)) & 1;
      oa[q][k] = (!heavy && r.total_h) ? r.last_heavy - r.lead : idx - r.lead;
    }
  // the own tile is usually its own main partner, and its prefixes are already in registers
#pragma unroll
  for (int q = 0; q < TL_Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) smem[4u * (q * TL_T + tid) + k] = sh[q][k];
  __syncthreads();
  resolve_in_tile<false>(r, L, smem, T, bh, bh1, heavy_mask, live_mask, nh_after, T, key, op, oa);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < TL_Q; ++q)
#pragma unroll
    for (int k = 0; k < 4; ++k) smem[4u * (q * TL_T + tid) + k] = sl[q][k];
  __syncthreads();
  resolve_in_tile<true>(r, L, smem, T, bl, bl1, heavy_mask, live_mask, nh_after, T, key, op, oa);

  // the other partner tiles (ranges precomputed per tile by tiled_scan_kernel)
  partner_pass<false>(r, L, wgt, BH, rg.x, rg.y, smem, s_ex, heavy_mask, live_mask, nh_after, T, key, op, oa);
  partner_pass<true>(r, L, wgt, BL, rg.z, rg.w, smem, s_ex, heavy_mask, live_mask, nh_after, T, key, op, oa);

#pragma unroll
  for (int q = 0; q < TL_Q; ++q) {
    const uint32_t pos = T * TILE + 4u * (q * TL_T + tid);
    if (pos >= r.span) continue;
    if (pos >= r.lead && pos + 4 <= r.span) {
      store_entries4(table + r.base + pos, op[q], oa[q]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (in_row(r, pos + k)) {
          table[r.base + pos + k] = AliasEntry{op[q][k], oa[q][k]};
        }
    }
  }
}

}  // namespace sky
