// Alias tables of rows that fit a wavefront's lanes or a workgroup's LDS: the code that builds one row (or a wavefront's
// worth of rows) and that the kernels of sky_build.hip and sky_build_fused.hip launch.  The table is the pure function of
// the weights that sky_build.hip defines.
#pragma once
#include "sky_build_common.h"
#include "sky_graph.h"

namespace sky {

// Vectors that are only 4-byte aligned: global loads and stores of 8 and 16 bytes need no more on gfx950.
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(4)));

// ---------------------------------------------------------------- 2..32 lanes per row
// G lanes share one row of at most PER * G slots; every lane holds PER consecutive weights, so a
// wavefront carries 64 / G rows and the per-row steps that do not depend on the row length (exact
// sum, ledger, scans) are paid once per 64 / G rows.  Prefix sums run over the group by DPP; SL and
// SH of every slot go to a per-group LDS strip padded to PER * G slots (slots outside the row add
// nothing), which each entry then searches once with a fixed number of probes; the heavies' slots,
// compacted by rank, give "next heavy" and "last heavy".  The rank rides in bits 52..63 of the SH scan.
// Every lane of the wavefront must call this together (DPP); a group without a row passes d = 0.
// s_pre: [2 * BLOCK * PER] u64 ([0, BLK): SL of every slot of the block; [BLK, 2 * BLK): SH), s_hs: [BLOCK * PER]
// (per group: row-local slot of its h-th heavy).  Returns false for a row whose weights sum to zero.
constexpr uint64_t GROUP_CNT = 1ull << 52;

template <int G, int PER, int BLOCK = 256>
__device__ __forceinline__ bool group_build_row(uint32_t off, uint32_t d, const float* __restrict__ wgt,
                                                AliasEntry* __restrict__ table, uint64_t* __restrict__ s_pre,
                                                uint8_t* __restrict__ s_hs, uint32_t tid = threadIdx.x) {
  static_assert(PER >= 4 && PER <= 6, "a lane loads one float4 (and one float), or three float2");
  constexpr uint32_t SLOTS = PER * G;
  constexpr uint32_t HB = PER == 4 ? SLOTS : PER == 5 ? SLOTS / 5 * 4 : SLOTS / 3 * 2;  // largest power of two <= SLOTS
  static_assert((HB & (HB - 1)) == 0 && HB <= SLOTS && 2 * HB > SLOTS && SLOTS <= 256, "G is a power of two");
  constexpr uint32_t BLK = BLOCK * PER;                      // slots of one block's strips (BLOCK threads)
  const int gl = tid & (G - 1);
  const int lane = tid & 63;
  const uint32_t gbase = (uint32_t)PER * (tid - gl);  // first LDS slot of the group
  const uint32_t pos = (uint32_t)PER * gl;

  float xs[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) xs[k] = 0.0f;
  if (PER == 4 || PER == 5) {
    if (pos < d) {
      const float4u x = *reinterpret_cast<const float4u*>(wgt + off + pos);
      xs[0] = x.x; xs[1] = x.y; xs[2] = x.z; xs[3] = x.w;
    }
  } else {
#pragma unroll
    for (int h = 0; h < PER / 2; ++h)
      if (pos + 2 * h < d) {
        const float2u x = *reinterpret_cast<const float2u*>(wgt + off + pos + 2 * h);
        xs[2 * h] = x.x;
        xs[2 * h + 1] = x.y;
      }
  }
  if (PER % 2 == 1 && pos + PER - 1 < d) xs[PER - 1] = wgt[off + pos + PER - 1];
  double wd[PER];
  uint32_t live = 0;
  // the sum of the row as a plain fp64 sum where that is exact (plain_sum_is_exact); a wavefront in which some
  // group's is not falls back to the three-limb sum for all of its groups
  double Sd = 0.0;
  uint32_t mn = 0xFFFFFFFFu;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool in = pos + k < d;
    if (in) live |= 1u << k;
    const float cw = masked_weight(xs[k], in);
    wd[k] = (double)cw;
    Sd += wd[k];
    mn = min(mn, __float_as_uint(cw) - 1u);
  }
  Sd = group_sum_f64<G>(Sd);
  mn = group_min_u32<G>(mn);
  const bool plain = plain_sum_is_exact(Sd, mn);
  if (__any(!plain)) {
    WSum3 S{0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < PER; ++k) wsum3_add(S, wd[k]);
    S = group_sum_wsum3<G>(S);
    if (!plain) Sd = S.top + S.mid + S.low != 0.0 ? wsum3_to_double(S) : 0.0;
  }
  const bool row_ok = Sd != 0.0;
  Ledger L = make_ledger_small(d, Sd);
  if (!row_ok) L.scale = 0.0;
  const double neg_fs = -L.fs;

  uint64_t dl[PER], sl[PER], sh[PER];
  float op[PER];
  uint32_t heavy = 0;
  uint64_t ra = 0, rb = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const Entry e = classify_small_fma(wd[k], L, neg_fs);
    dl[k] = (e.heavy || !((live >> k) & 1)) ? 0 : e.amount;
    ra += dl[k];
    rb += e.heavy ? (e.amount | GROUP_CNT) : 0;
    sl[k] = ra;
    sh[k] = rb;
    op[k] = (float)e.p;
    if (e.heavy) heavy |= 1u << k;
  }
  const uint64_t ia = group_scan_u64<G>(ra), ib = group_scan_u64<G>(rb);
  const uint32_t nh = (uint32_t)(shfl_u64(ib, (lane - gl) + G - 1) >> 52);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    sl[k] += ia - ra;
    sh[k] += ib - rb;
    s_pre[gbase + pos + k] = sl[k];
    s_pre[BLK + gbase + pos + k] = sh[k] & (GROUP_CNT - 1);
    if ((heavy >> k) & 1) s_hs[gbase + (uint32_t)(sh[k] >> 52) - 1] = (uint8_t)(pos + k);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // light: first slot with SH > SL - D.  heavy: first slot with SL >= SH, i.e. SL > SH - 1.
  // The first probe narrows the answer to a window of HB slots that ends inside the strip.
  uint32_t arr[PER], at[PER];
  uint64_t key[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool hv = (heavy >> k) & 1;
    arr[k] = gbase + (hv ? 0u : BLK);
    key[k] = hv ? (sh[k] & (GROUP_CNT - 1)) - 1 : sl[k] - dl[k];
    at[k] = HB == SLOTS ? 0u : (s_pre[arr[k] + HB - 1] <= key[k] ? SLOTS - HB : 0u);
  }
#pragma unroll
  for (uint32_t step = HB / 2; step >= 1; step >>= 1) {
    uint64_t v[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = s_pre[arr[k] + at[k] + step - 1];
#pragma unroll
    for (int k = 0; k < PER; ++k) at[k] += v[k] <= key[k] ? step : 0u;
  }
  uint32_t oa[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint64_t v = s_pre[arr[k] + at[k]];
    const bool found = v > key[k];
    const uint32_t self = pos + k;
    if (!((heavy >> k) & 1)) {
      oa[k] = found ? at[k] : (nh ? (uint32_t)s_hs[gbase + nh - 1] : self);
    } else {
      const uint32_t hc = (uint32_t)(sh[k] >> 52);
      if (hc < nh && found) {
        op[k] = residual_prob(L.one + key[k] + 1 - v, L);
        oa[k] = s_hs[gbase + hc];
      } else {
        op[k] = 1.0f;
        oa[k] = self;
      }
    }
    if (!row_ok) {
      op[k] = 0.0f;
      oa[k] = SKY_INVALID;
    }
  }
  // the next row of this group reuses the strips: its writes must stay behind these reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int h = 0; h < PER / 2; ++h) {
    const uint32_t m = (live >> (2 * h)) & 3u;
    AliasEntry* t = table + off + pos + 2 * h;
    if (m == 3u) {
      uint4u o;
      o.x = __float_as_uint(op[2 * h]); o.y = oa[2 * h]; o.z = __float_as_uint(op[2 * h + 1]); o.w = oa[2 * h + 1];
      *reinterpret_cast<uint4u*>(t) = o;
    } else if (m == 1u) {
      t[0] = AliasEntry{op[2 * h], oa[2 * h]};
    }
  }
  if (PER % 2 == 1 && ((live >> (PER - 1)) & 1)) table[off + pos + PER - 1] = AliasEntry{op[PER - 1], oa[PER - 1]};
  return row_ok || d == 0;
}

// A row of one or two entries in closed form.
__device__ __forceinline__ bool tiny_row(uint32_t off, uint32_t d, const float* __restrict__ wgt,
                                         AliasEntry* __restrict__ table) {
  // a weight adds to the exact sum iff it is at least 2^-64
  constexpr float UNIT = 5.421010862427522170037e-20f;  // 2^-64
  const float w0 = clamp_weight(wgt[off]);
  if (d == 1) {
    const bool ok = w0 >= UNIT;
    table[off] = AliasEntry{ok ? 1.0f : 0.0f, ok ? 0u : SKY_INVALID};
    return ok;
  }
  const float w1 = clamp_weight(wgt[off + 1]);
  const bool ok = w0 >= UNIT || w1 >= UNIT;
  AliasEntry a{0.0f, SKY_INVALID}, b{0.0f, SKY_INVALID};
  if (ok) {
    WSum3 S{0.0, 0.0, 0.0};
    wsum3_add(S, (double)w0);
    wsum3_add(S, (double)w1);
    const Ledger L = make_ledger_small(2, wsum3_to_double(S));
    const Entry e0 = classify_small((double)w0, true, L), e1 = classify_small((double)w1, true, L);
    // a lone heavy is the last heavy: it keeps its bucket and tops up the light
    a = AliasEntry{e0.heavy ? 1.0f : (float)e0.p, (!e0.heavy && e1.heavy) ? 1u : 0u};
    b = AliasEntry{e1.heavy ? 1.0f : (float)e1.p, (!e1.heavy && e0.heavy) ? 0u : 1u};
  }
  uint4u o;
  o.x = __float_as_uint(a.prob); o.y = a.alias; o.z = __float_as_uint(b.prob); o.w = b.alias;
  *reinterpret_cast<uint4u*>(table + off) = o;
  return ok;
}

// ---------------------------------------------------------------- rows of at most 32 entries, where they lie
// One wavefront walks a contiguous range of vertices, 64 at a time, and builds every row of 1..32 entries it
// meets: the rows of a class queue up in LDS until they fill the wavefront (64 rows of 1..2 entries, 32 of 3..8 with
// 2 lanes each, 16 of 9..16 with 4, 8 of 17..32 with 8) and are then built by the same code as in the class kernels.
// Neighbouring rows of different classes share their cache lines, and here the same wavefront touches them within a
// few steps; no row list is written or read for these classes.  Also sets valid[] of the vertices it owns (rows of
// 0..32 entries).  Workgroups are single wavefronts: nothing in here waits for another wavefront.
// Queue capacities (128, 96, 80, 72): less than one batch left over plus the 64 vertices of a step
// (64 + 63, 64 + 31, 64 + 15, 64 + 7), rounded up.  A queue entry is the row's offset and, in 16 bits, its degree (6 bits) above the vertex's position in
// the wavefront's range (10 bits): the vertex id itself is only needed for a row without weight, whose flag is
// cleared.  6.5 KB of LDS per wavefront, so that six of them fit every SIMD (the kernel's registers allow six).
constexpr uint32_t SMALL_RANGE = 1024;  // most vertices per wavefront
constexpr uint32_t SMALL_QBASE[4] = {0, 128, 224, 304};
constexpr uint32_t SMALL_QTOTAL = 376;
constexpr size_t SMALL_LDS_BYTES = 2 * 64 * 4 * 8 + 64 * 4 + SMALL_QTOTAL * 6;
// Vertices [lo, lo + per_wave) of the n (src null: the vertices themselves) by one wavefront that is a workgroup.
__device__ __forceinline__ void small_rows_range(uint32_t lo, const uint32_t* __restrict__ xadj, const float* __restrict__ wgt,
                                                 const uint32_t* __restrict__ src, uint32_t n, uint32_t per_wave,
                                                 AliasEntry* __restrict__ table, int8_t* __restrict__ valid,
                                                 uint64_t* __restrict__ smem) {
  uint64_t* s_pre = smem;                                           // [2 * 64 * 4]
  uint32_t* q_off = reinterpret_cast<uint32_t*>(smem + 2 * 64 * 4);  // [SMALL_QTOTAL]
  uint16_t* q_it = reinterpret_cast<uint16_t*>(q_off + SMALL_QTOTAL);  // [SMALL_QTOTAL]
  uint8_t* s_hs = reinterpret_cast<uint8_t*>(q_it + SMALL_QTOTAL);   // [64 * 4]
  const uint32_t lane = threadIdx.x;
  const uint32_t hi = min(n, lo + per_wave);
  uint32_t cnt[4] = {0, 0, 0, 0};  // wave-uniform queue lengths: rows of 1..2, 3..8, 9..16, 17..32 entries

  // the last `rows` entries of queue q, one per group of G lanes; d = 0 for a group without a row.  `t` is the lane
  // number behind an empty asm statement: it keeps what depends on the lane number inside one batch (hoisted
  // out of the loop for all four row sizes at once, those values double the registers of the kernel).
  auto take = [&](int q, uint32_t rows, uint32_t G, uint32_t& t, uint32_t& off, uint32_t& it, uint32_t& d) {
    t = lane;
    asm volatile("" : "+v"(t));
    const uint32_t r = t / G;
    off = it = d = 0;
    if (r < rows) {
      const uint32_t k = SMALL_QBASE[q] + cnt[q] - rows + r;
      off = q_off[k];
      const uint32_t x = q_it[k];
      it = x & (SMALL_RANGE - 1);
      d = x >> 10;
    }
  };
  auto clear_valid = [&](uint32_t it) {  // a row whose weights sum to zero (rare)
    const uint32_t item = lo + it;
    valid[src ? src[item] : item] = 0;
  };
  auto build_tiny = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(0, rows, 1, t, off, it, d);
    if (d && !tiny_row(off, d, wgt, table)) clear_valid(it);
    cnt[0] -= rows;
  };
  auto build_g2 = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(1, rows, 2, t, off, it, d);
    const bool ok = group_build_row<2, 4, 64>(off, d, wgt, table, s_pre, s_hs, t);
    if ((t & 1) == 0 && !ok) clear_valid(it);
    cnt[1] -= rows;
  };
  auto build_g4 = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(2, rows, 4, t, off, it, d);
    const bool ok = group_build_row<4, 4, 64>(off, d, wgt, table, s_pre, s_hs, t);
    if ((t & 3) == 0 && !ok) clear_valid(it);
    cnt[2] -= rows;
  };
  auto build_g8 = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(3, rows, 8, t, off, it, d);
    const bool ok = group_build_row<8, 4, 64>(off, d, wgt, table, s_pre, s_hs, t);
    if ((t & 7) == 0 && !ok) clear_valid(it);
    cnt[3] -= rows;
  };

  // the row offsets of step i + 1 are requested before the batches of step i are built
  auto fetch = [&](uint32_t base, uint32_t& v, uint32_t& off, uint32_t& end) {
    const uint32_t item = base + lane;
    v = 0xFFFFFFFFu;
    off = end = 0;
    if (item < hi) {
      v = src ? src[item] : item;
      off = xadj[v];
      end = xadj[v + 1];
    }
  };
  uint32_t nv, noff, nend;
  fetch(lo, nv, noff, nend);
  for (uint32_t base = lo; base < hi; base += 64u) {
    const uint32_t v = nv, off = noff, d = nend - noff;
    if (base + 64u < hi) fetch(base + 64u, nv, noff, nend);
    int q = -1;
    if (v != 0xFFFFFFFFu && d <= 32u) {
      valid[v] = d != 0;  // a row without weight clears it when it is built
      q = d == 0 ? -1 : d <= 2 ? 0 : d <= 8 ? 1 : d <= 16 ? 2 : 3;
    }
    const uint32_t packed = (d << 10) | (base - lo + lane);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const unsigned long long m = __ballot(q == c);
      if (q == c) {
        const uint32_t p = SMALL_QBASE[c] + cnt[c] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        q_off[p] = off;
        q_it[p] = (uint16_t)packed;
      }
      cnt[c] += (uint32_t)__popcll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    while (cnt[0] >= 64u) build_tiny(64);
    while (cnt[1] >= 32u) build_g2(32);
    while (cnt[2] >= 16u) build_g4(16);
    while (cnt[3] >= 8u) build_g8(8);
    // the next step's queue entries stay behind this step's reads of the queues
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (cnt[0]) build_tiny(cnt[0]);
  if (cnt[1]) build_g2(cnt[1]);
  if (cnt[2]) build_g4(cnt[2]);
  if (cnt[3]) build_g8(cnt[3]);
}

// ---------------------------------------------------------------- one row per workgroup, pairing by merge
// Same table as build_lds_kernel, reached without a binary search per entry.  Lights and heavies
// are compacted by rank into one LDS array (inclusive SL of the lights from the front, inclusive
// SH of the heavies from the back, a sentinel after each).  In the order of the merged sequence,
// ties heavy first,
//   the alias of light r is the heavy rank reached when light r - 1 is taken (rank 0 for r = 0),
//   the light that finishes heavy h is the light rank reached when heavy h is taken,
// so each thread finds where its share of PER merged elements starts (one diagonal search) and
// walks it.  The heavy count rides in bits 52..63 of the SH scan: a row of at most 4093 entries
// keeps its sums below 2^52.
constexpr uint64_t MERGE_CNT = 1ull << 52;
constexpr uint32_t MERGE_SELF = 0x80000000u;  // "prob 1, alias self" in the per-heavy result word

// LDS of a row: 14 bytes a slot.
constexpr size_t merge_lds_bytes(int rowt, int per) { return ((size_t)rowt * per + 2) * 14; }

// The row `rr` by ROWT threads that share `smem` and, for the wavefronts' sums, s_aux[8 * ROWT / 64].  Returns false when its weights sum to zero.  All threads of the
// workgroup call it together; the arrays in LDS may be rewritten only after a barrier.
template <int ROWT, int PER>
__device__ __forceinline__ bool merge_row(const RowRef rr, uint64_t* smem, uint64_t* s_aux,
                                          const float* __restrict__ wgt, AliasEntry* __restrict__ table,
                                          const int tid = threadIdx.x) {
  // PER consecutive slots per thread, counted from the row's 16-byte aligned start; a thread moves them as
  // quads when PER is a multiple of 4, as pairs otherwise (its first slot is then only 8-byte aligned)
  constexpr int VEC = PER % 4 == 0 ? 4 : 2;
  static_assert(PER % VEC == 0 && PER <= 16, "whole vectors, and `live` has one bit per slot");
  constexpr int CAP = ROWT * PER;
  constexpr int NW = ROWT / 64;
  constexpr uint32_t TOP = CAP + 1;  // heavy h lives at index TOP - h of the value array and of the result array
  constexpr bool PACKED = CAP <= 4096;  // the heavy count rides in the SH scan; larger rows scan it separately
  static_assert(CAP <= 8192, "sums and shifts below assume rows of fewer than 2^13 entries");
  uint64_t* s_v = smem;                                             // [CAP + 2]
  uint32_t* s_res = reinterpret_cast<uint32_t*>(smem + CAP + 2);  // [CAP + 2]
  uint16_t* s_hs = reinterpret_cast<uint16_t*>(s_res + CAP + 2);   // [CAP + 2] row-local slot of heavy h
  WSum3* s_wsum = reinterpret_cast<WSum3*>(s_aux);      // [NW]
  double* s_fsum = reinterpret_cast<double*>(s_aux + 3 * NW);  // [NW]
  uint64_t* s_ex = s_aux + 4 * NW;                       // [3 * NW]
  uint32_t* s_mn = reinterpret_cast<uint32_t*>(s_aux + 7 * NW);  // [NW]

  const uint32_t off = rr.off, d = rr.d;
  const uint32_t base = off & ~3u, lead = off - base, span = lead + d;
  const int wave = tid >> 6, lane = tid & 63;
  const uint32_t pos0 = (uint32_t)PER * (uint32_t)tid;
  const bool wave_on = (uint32_t)(PER * 64 * wave) < span;

  double wd[PER];
  uint32_t live = 0;  // bit j: slot pos0 + j belongs to the row
  // the sum of the row as a plain fp64 sum where that is exact (plain_sum_is_exact), else as three limbs
  double rsum = 0.0;
  uint32_t mn = 0xFFFFFFFFu;
  if (wave_on) {
#pragma unroll
    for (int t = 0; t < PER / VEC; ++t) {
      const uint32_t pos = pos0 + (uint32_t)(VEC * t);
      float xs[4] = {0.f, 0.f, 0.f, 0.f};
      if (pos < span) {
        if constexpr (VEC == 4) {
          const float4 x = *reinterpret_cast<const float4*>(wgt + base + pos);
          xs[0] = x.x; xs[1] = x.y; xs[2] = x.z; xs[3] = x.w;
        } else {
          const float2 x = *reinterpret_cast<const float2*>(wgt + base + pos);
          xs[0] = x.x; xs[1] = x.y;
        }
      }
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const uint32_t idx = pos + k;
        const bool in = idx - lead < d;  // one unsigned compare: slots before the row wrap around
        if (in) live |= 1u << (t * VEC + k);
        const float cw = masked_weight(xs[k], in);
        wd[t * VEC + k] = (double)cw;
        rsum += wd[t * VEC + k];
        mn = min(mn, __float_as_uint(cw) - 1u);
      }
    }
    rsum = group_sum_f64<64>(rsum);
    mn = wave_min_u32(mn);
  } else {
#pragma unroll
    for (int j = 0; j < PER; ++j) wd[j] = 0.0;
  }
  if (NW > 1) {
    if (lane == 0) {
      s_fsum[wave] = rsum;
      s_mn[wave] = mn;
    }
    __syncthreads();
    rsum = s_fsum[0];
    mn = s_mn[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      rsum += s_fsum[i];
      mn = min(mn, s_mn[i]);
    }
  }
  if (!plain_sum_is_exact(rsum, (uint32_t)__builtin_amdgcn_readfirstlane((int)mn))) {  // uniform over the workgroup
    WSum3 sum{0.0, 0.0, 0.0};
    if (wave_on) {
#pragma unroll
      for (int j = 0; j < PER; ++j) wsum3_add(sum, wd[j]);
      sum = group_sum_wsum3<64>(sum);
    }
    if (NW > 1) {
      if (lane == 0) s_wsum[wave] = sum;
      __syncthreads();
      sum = s_wsum[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) {
        sum.top += s_wsum[i].top;
        sum.mid += s_wsum[i].mid;
        sum.low += s_wsum[i].low;
      }
    }
    rsum = sum.top + sum.mid + sum.low != 0.0 ? wsum3_to_double(sum) : 0.0;
  }
  if (rsum == 0.0) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if ((live >> j) & 1) table[base + pos0 + j] = AliasEntry{0.0f, SKY_INVALID};
    return false;
  }
  const Ledger L = make_ledger_small(d, rsum);
  const double neg_fs = -L.fs;

  float op[PER];
  uint32_t hcnt[PER];  // heavies up to and including this slot
  uint32_t heavy = 0;
  uint32_t nh, nl;
  {
    uint64_t dl[PER], dh[PER], sl[PER], sh[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const bool in = (live >> j) & 1;
      const Entry e = PACKED ? classify_small_fma(wd[j], L, neg_fs) : classify_fast(wd[j], in, L);
      dl[j] = (e.heavy || !in) ? 0 : e.amount;
      dh[j] = e.heavy ? (PACKED ? (e.amount | MERGE_CNT) : e.amount) : 0;
      op[j] = (float)e.p;
      if (e.heavy) heavy |= 1u << j;
    }
    uint64_t total_l, total_h;
    uint32_t ex_c = 0;
    if constexpr (PACKED) {
      block_scan2_flat<ROWT, PER>(dl, dh, s_ex, sl, sh, total_l, total_h, wave_on);
      nh = (uint32_t)(total_h >> 52);
    } else {
      block_scan2c_flat<ROWT, PER>(dl, dh, (uint32_t)__popc(heavy), s_ex, sl, sh, ex_c, total_l, total_h, nh, wave_on);
    }
    nl = d - nh;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t hc = PACKED ? (uint32_t)(sh[j] >> 52) : ex_c + (uint32_t)__popc(heavy & ((2u << j) - 1));
      hcnt[j] = hc;
      if (!((live >> j) & 1)) continue;
      const uint32_t li = pos0 + j - lead;
      const bool hv = (heavy >> j) & 1;
      s_v[hv ? TOP + 1 - hc : li - hc] = hv ? (PACKED ? (sh[j] & (MERGE_CNT - 1)) : sh[j]) : sl[j];
      if (hv) s_hs[hc - 1] = (uint16_t)li;
    }
  }
  if (tid == 0) {
    s_v[nl] = ~0ull;
    s_v[TOP - nh] = ~0ull;
  }
  __syncthreads();

  if (nh) {
    if (tid == 0) s_res[0] = s_hs[0];  // the first light starts in the first heavy
    // merged positions [k0, k0 + PER) belong to this thread; a lights and k0 - a heavies come before them
    const uint32_t k0 = pos0;
    if (k0 < d) {
      uint32_t lo = k0 > nh ? k0 - nh : 0u, hi = min(k0, nl);
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (s_v[mid - 1] < s_v[TOP - (k0 - mid)]) lo = mid; else hi = mid - 1;
      }
      uint32_t a = lo, b = k0 - lo;
      const uint32_t steps = min((uint32_t)PER, d - k0);
      uint64_t va = s_v[a], vb = s_v[TOP - b];  // heads of the two sequences: only the one taken is read again
#pragma unroll
      for (int s = 0; s < PER; ++s) {
        if ((uint32_t)s < steps) {
          if (vb <= va) {
            s_res[TOP - b] = a;
            ++b;
            vb = s_v[TOP - b];
          } else {
            ++a;
            if (a < nl) s_res[a] = s_hs[min(b, nh - 1)];
            va = s_v[a];
          }
        }
      }
    }
    __syncthreads();
    // heavies, densely by rank: residual probability from the light that finishes them
    for (uint32_t h = tid; h < nh; h += ROWT) {
      const uint32_t r = s_res[TOP - h];
      uint32_t out = MERGE_SELF;
      if (h + 1 < nh && r < nl) out = __float_as_uint(residual_prob(L.one + s_v[TOP - h] - s_v[r], L));
      s_res[TOP - h] = out;
    }
    __syncthreads();
  }

  if (pos0 < span) {
    uint32_t oa[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t li = pos0 + j - lead;
      const uint32_t hc = hcnt[j];
      oa[j] = li;
      if (nh && ((live >> j) & 1)) {
        if ((heavy >> j) & 1) {
          const uint32_t x = s_res[TOP - (hc - 1)];
          op[j] = x == MERGE_SELF ? 1.0f : __uint_as_float(x);
          if (x != MERGE_SELF) oa[j] = s_hs[hc];
        } else {
          oa[j] = s_res[li - hc];
        }
      }
    }
#pragma unroll
    for (int t = 0; t < PER / VEC; ++t) {
      const uint32_t pos = pos0 + (uint32_t)(VEC * t);
      if (pos >= lead && pos + VEC <= span) {
        if constexpr (VEC == 4) {
          const float p4[4] = {op[4 * t], op[4 * t + 1], op[4 * t + 2], op[4 * t + 3]};
          const uint32_t a4[4] = {oa[4 * t], oa[4 * t + 1], oa[4 * t + 2], oa[4 * t + 3]};
          store_entries4(table + base + pos, p4, a4);
        } else {
          *reinterpret_cast<uint4*>(table + base + pos) =
              make_uint4(__float_as_uint(op[2 * t]), oa[2 * t], __float_as_uint(op[2 * t + 1]), oa[2 * t + 1]);
        }
      } else {
#pragma unroll
        for (int k = 0; k < VEC; ++k)
          if ((live >> (t * VEC + k)) & 1) table[base + pos + k] = AliasEntry{op[VEC * t + k], oa[VEC * t + k]};
      }
    }
  }
  return true;
}

}  // namespace sky
