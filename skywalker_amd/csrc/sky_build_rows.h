// Alias tables of rows that fit a wavefront's lanes or a workgroup's LDS: the code that builds one row (or a wavefront's
// worth of rows) and that the kernels of sky_build.hip and sky_build_fused.hip launch.  The table is the pure function of
// the weights that sky_build.hip defines.
#pragma once
#include <type_traits>

#include "sky_build_common.h"
#include "sky_graph.h"

namespace sky {

// Vectors that are only 4-byte aligned: global loads and stores of 8 and 16 bytes need no more on gfx950.
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(4)));

// ---------------------------------------------------------------- slots of a wavefront
// A thread works on PER consecutive slots, so that prefixes and pairing stay in registers, but memory wants the lanes of an
// instruction side by side: 4 bytes read and 8 written per entry run at 3.1 TB/s when every lane moves its own 8 slots as
// 16-byte pieces, at 1.8 with 16 slots, at 5.5 to 6.0 when the lanes' pieces are consecutive (4 GiB tables, one MI355X).  So
// the wavefront's weights and entries change hands in LDS, in room of its own: 12 or 24 instructions of 16 bytes per lane
// for 8 or 16 slots.
// Pieces of 16 bytes lie where no two of eight lanes that follow one another meet in a bank: P pieces per lane.
template <int P>
__device__ __forceinline__ uint32_t piece_at(uint32_t c) {
  return P % 8 == 0 ? c ^ ((c >> 3) & 7u) : P % 4 == 0 ? c ^ ((c >> 3) & 3u) : P % 2 == 0 ? c ^ ((c >> 3) & 1u) : c;
}
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Values of the slots first + PER * lane + k of an array, 0 from `end` on (16 bytes behind that may be read).
// `stage`: 64 * PER * 4 bytes of LDS for this wavefront, 16-byte aligned.
template <int PER>
__device__ __forceinline__ void wave_load(const float* __restrict__ src, uint32_t first, uint32_t end, void* stage,
                                          uint32_t lane, float (&x)[PER]) {
  static_assert(PER % 2 == 0, "whole pairs");
  float4* const s4 = reinterpret_cast<float4*>(stage);
  constexpr int Q = PER / 4, PIECES = 16 * PER;  // whole instructions; pieces of the wavefront
  constexpr int N = (PIECES + 63) / 64;
  float4 v[N];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const uint32_t c = 64u * t + lane, pos = first + 4 * c;
    v[t] = make_float4(0.f, 0.f, 0.f, 0.f);
    if ((PIECES % 64 == 0 || c < PIECES) && pos < end) {
      const float4u y = *reinterpret_cast<const float4u*>(src + pos);
      v[t] = make_float4(y.x, y.y, y.z, y.w);
    }
    if (pos < end && pos + 4 > end) {  // one lane of a row
      if (pos + 1 >= end) v[t].y = 0.f;
      if (pos + 2 >= end) v[t].z = 0.f;
      v[t].w = 0.f;
    }
  }
  if constexpr (PER == 4) {
    x[0] = v[0].x; x[1] = v[0].y; x[2] = v[0].z; x[3] = v[0].w;
  } else {
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const uint32_t c = 64u * t + lane;
      if (PIECES % 64 == 0 || c < PIECES) s4[PER % 4 == 0 ? piece_at<Q>(c) : c] = v[t];
    }
    wave_lds_sync();
    if constexpr (PER % 4 == 0) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const float4 y = s4[piece_at<Q>(Q * lane + q)];
        x[4 * q] = y.x; x[4 * q + 1] = y.y; x[4 * q + 2] = y.z; x[4 * q + 3] = y.w;
      }
    } else {
      const float2* const s2 = reinterpret_cast<const float2*>(stage);
#pragma unroll
      for (int h = 0; h < PER / 2; ++h) {
        const float2 y = s2[PER / 2 * lane + h];
        x[2 * h] = y.x; x[2 * h + 1] = y.y;
      }
    }
  }
}
// Entries of the slots first + PER * lane + k that lie below `end`.
// `stage`: 64 * PER * 8 bytes of LDS for this wavefront, 16-byte aligned.
template <int PER>
__device__ __forceinline__ void wave_store(AliasEntry* __restrict__ dst, uint32_t first, uint32_t end,
                                           void* stage, uint32_t lane, const float (&p)[PER], const uint32_t (&a)[PER]) {
  constexpr int P = PER / 2;
  uint4* const s4 = reinterpret_cast<uint4*>(stage);
  auto put = [&](uint32_t pos, const uint4u& y) {
    if (pos + 2 <= end) *reinterpret_cast<uint4u*>(dst + pos) = y;
    else if (pos < end) dst[pos] = AliasEntry{__uint_as_float(y.x), y.y};
  };
  if constexpr (PER == 4) {  // side by side enough
#pragma unroll
    for (int h = 0; h < 2; ++h)
      put(first + 4 * lane + 2 * h, uint4u{__float_as_uint(p[2 * h]), a[2 * h], __float_as_uint(p[2 * h + 1]), a[2 * h + 1]});
    return;
  }
#pragma unroll
  for (int h = 0; h < P; ++h)
    s4[piece_at<P>(P * lane + h)] = make_uint4(__float_as_uint(p[2 * h]), a[2 * h], __float_as_uint(p[2 * h + 1]), a[2 * h + 1]);
  wave_lds_sync();
#pragma unroll
  for (int t = 0; t < P; ++t) {
    const uint32_t c = 64u * t + lane;
    const uint4 y = s4[piece_at<P>(c)];
    put(first + 2 * c, uint4u{y.x, y.y, y.z, y.w});
  }
}

// ---------------------------------------------------------------- slots of a quad of lanes
template <int PERM>
__device__ __forceinline__ uint32_t quad_get(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, PERM, 0xF, 0xF, true);
}
constexpr int quad_perm(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }
// The lanes of a quad exchange the entries of their 8 consecutive slots each: v[l] becomes pair tid & 3 of those of the quad's lane
// l, so that one 16-byte store a lane moves 64 bytes in a row.  All lanes of the wavefront call it together.
__device__ __forceinline__ void quad_exchange(uint32_t tid, const float (&p)[8], const uint32_t (&a)[8], uint32_t (&v)[4][4]) {
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    v[h][0] = __float_as_uint(p[2 * h]);
    v[h][1] = a[2 * h];
    v[h][2] = __float_as_uint(p[2 * h + 1]);
    v[h][3] = a[2 * h + 1];
  }
  const bool b0 = tid & 1, b1 = tid & 2;
  auto swap = [&](auto perm, bool odd, uint32_t& lo, uint32_t& hi) {  // a 2 x 2 transpose between partner lanes
    constexpr int P = decltype(perm)::value;
    const uint32_t from_lo = quad_get<P>(lo), from_hi = quad_get<P>(hi);
    lo = odd ? from_hi : lo;
    hi = odd ? hi : from_lo;
  };
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    using X1 = std::integral_constant<int, quad_perm(1, 0, 3, 2)>;
    using X2 = std::integral_constant<int, quad_perm(2, 3, 0, 1)>;
    swap(X1{}, b0, v[0][w], v[1][w]);
    swap(X1{}, b0, v[2][w], v[3][w]);
    swap(X2{}, b1, v[0][w], v[2][w]);
    swap(X2{}, b1, v[1][w], v[3][w]);
  }
}

// ---------------------------------------------------------------- sums as doubles
// An amount is one rounding instead of an addition and a mask, a residual one fused multiply-add instead of a conversion.
// Deficits and surpluses are summed apart.  A light, and a slot behind the row, has a deficit of at most 2^40: in fewer than 2^13
// slots every sum of deficits is a whole number below 2^53, which a double holds.  The surpluses add up to as much where every
// weight counts, so that both together pass 2^53; where weights below 2^-64, which add nothing to the row's sum, have shares
// all the same they add up to more by themselves.  A sum of surpluses below 2^53 is exact in whatever order it was added, and
// one that was rounded is at least 2^53 (rounding is monotone): above every deficit prefix, which is all that is asked of it.
template <int G>
__device__ __forceinline__ double group_scan_f64(double v) {
  const int gl = lane_id() & (G - 1);
  auto from = [&](int dist, auto get) {
    const double o = __longlong_as_double((long long)get((uint64_t)__double_as_longlong(v)));
    v += G >= 16 || gl >= dist ? o : 0.0;
  };
  from(1, [](uint64_t b) { return dpp0_u64<DPP_ROW_SHR1, 0xF>(b); });
  if (G >= 4) from(2, [](uint64_t b) { return dpp0_u64<DPP_ROW_SHR2, 0xF>(b); });
  if (G >= 8) from(4, [](uint64_t b) { return dpp0_u64<DPP_ROW_SHR4, 0xF>(b); });
  if (G >= 16) from(8, [](uint64_t b) { return dpp0_u64<DPP_ROW_SHR8, 0xF>(b); });
  if (G >= 32) from(16, [](uint64_t b) { return dpp0_u64<DPP_ROW_BCAST15, 0xA>(b); });
  if (G >= 64) from(32, [](uint64_t b) { return dpp0_u64<DPP_ROW_BCAST31, 0xC>(b); });
  return v;
}
__device__ __forceinline__ double wave_scan_f64(double v) { return group_scan_f64<64>(v); }
__device__ __forceinline__ double lane_before_f64(double v) {
  return __longlong_as_double((long long)lane_before_u64((uint64_t)__double_as_longlong(v)));
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ double lane_shfl_f64(double v, int lane) {
  return __longlong_as_double((long long)shfl_u64((uint64_t)__double_as_longlong(v), lane));
}
// max(|t|, m) in one instruction (fmax would quieten its operands first; neither is a NaN here).
__device__ __forceinline__ double max_abs_f64(double t, double m) {
  double x;
  asm("v_max_f64 %0, |%1|, %2" : "=v"(x) : "v"(t), "v"(m));
  return x;
}

// ---------------------------------------------------------------- 2..32 lanes per row
// G lanes share one row of at most PER * G slots; every lane holds PER consecutive weights, so a
// wavefront carries 64 / G rows and the per-row steps that do not depend on the row length (exact
// sum, ledger, scans) are paid once per 64 / G rows.  The rows are paired by a merge, as merge_row below does it: lights' prefix
// sums from the front of the row's strip in LDS, heavies' from its back, a sentinel after each; a lane finds by a search along the
// diagonal where its PER merged elements start and walks them.  A step leaves, for the light it takes, which heavy is the
// next light's alias, and for the heavy it takes the residual that its light leaves.
// Slots behind the row have weight 0 and so come out as lights of a whole bucket's deficit that rank after the row's own;
// a heavy that only they reach has a prefix sum above the deficits of the row's own lights.
// Instruction issue bounds it (94 % of the vector units' cycles for rows of 50 that lie side by side; scattered rows of a power-law
// graph wait for lines that they use in part).
// Every lane of the wavefront must call this together (DPP); a group without a row passes d = 0.
// `smem`: group_lds_bytes(G, PER, BLOCK) of LDS for the BLOCK threads that call it.  Returns false for a row whose
// weights sum to zero.
//
// A strip has PER * G + 2 entries: light r at index r, heavy h at index TOP - h.  Every offset that a step needs is the offset of
// the light or the heavy at hand, or of the next one:
//   val   prefix sum of the light or heavy; once every lane has walked its share,
//   word  of light r: the offset of its alias' heavy.  Of index TOP - h - 1: the residual of heavy h, below its own index because
//         the entry there also holds
//   slot  of index TOP - h: the slot of heavy h, which is the alias of heavy h - 1 (a byte, behind the sums)
// (16-byte entries of all three save a shift a slot and lose more to bank conflicts; words of their own cost a
// wavefront in six its place.)
constexpr uint32_t group_entries(int G, int PER, int BLOCK) {
  return ((uint32_t)(BLOCK / G) * (G * PER + 2) + 2 + 7) / 8 * 8;  // one more at either end is read
}
constexpr size_t group_lds_bytes(int G, int PER, int BLOCK) { return (size_t)group_entries(G, PER, BLOCK) * 9; }

// Lanes and slots of a lane by class.  8 slots a lane where 4 would do for twice the lanes: what a lane does once for its row
// (sum, division, scans, search) is half of its instructions with 4.  Rows that lie side by side, 200 M entries in rows of
// 100 (32 lanes of 4 / 16 of 8) 739 / 630 us, of 50 (16 of 4 / 8 of 8) 720 / 640.  Rows of 33..64 that lie scattered in a graph
// built by class wait for their lines, of which half as many lanes ask for fewer at a time: they lose some 5 and 2 % (the scale-26
// graph 0.615 / 0.650 ms, rows of every length in random order 0.261 / 0.267, five processes a side that differ by as much), 0.4 % of
// such a build; rows of 65..128 gain there too (scale 25 with 56 edges a vertex 0.255 / 0.22 ms).
// Not for the rows of up to 32: 200 M entries in rows of 24 835 / 680, but where they lie among others half as many lanes
// means batches that are half as full (scale 20 with 16 edges a vertex 140 / 150, scale 22 with 10 316 / 333).
struct GroupShape {
  int lanes, per;
};
constexpr GroupShape SHAPE_G2{2, 4}, SHAPE_G4{4, 4}, SHAPE_G8{8, 4}, SHAPE_G16{8, 8}, SHAPE_G32{16, 8}, SHAPE_G32S{32, 5}, SHAPE_G32X{32, 6};

template <int G, int PER, int BLOCK = 256>
__device__ __forceinline__ bool group_build_row(uint32_t off, uint32_t d, const float* __restrict__ wgt,
                                                AliasEntry* __restrict__ table, void* __restrict__ smem, uint32_t tid = threadIdx.x) {
  static_assert((PER >= 4 && PER <= 6) || PER == 8, "a lane loads one float4 (and one float), two, or three float2");
  constexpr uint32_t SLOTS = PER * G, STRIDE = SLOTS + 2, TOP = SLOTS + 1;
  static_assert(SLOTS <= 256, "slots in 8 bits");
  // A lane's surpluses are at most (PER + 2) d shares of 2^40 (a weight that counts in part has up to 2 d shares, all of them
  // together): where the prefix up to them was rounded, the one before them lies above every deficit prefix too, and so does
  // their difference.
  static_assert((PER + 3) * SLOTS < 8192, "the surpluses before a lane may be got by subtraction");
  constexpr uint32_t SZ = 8, N = group_entries(G, PER, BLOCK);
  char* const s_v = reinterpret_cast<char*>(smem);
  auto val = [&](uint32_t at) -> double& { return *reinterpret_cast<double*>(s_v + at); };
  auto word = [&](uint32_t at) -> uint32_t& { return *reinterpret_cast<uint32_t*>(s_v + at); };
  auto slot_of = [&](uint32_t at) -> uint8_t& { return *reinterpret_cast<uint8_t*>(s_v + N * 8 + (at >> 3)); };
  const uint32_t gl = tid & (G - 1), lane = tid & 63;
  const uint32_t strip = SZ * (STRIDE * (tid / G) + 1);  // its offset
  const uint32_t pos = (uint32_t)PER * gl;
  const uint32_t last_lane = lane - gl + G - 1;

  float xs[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) xs[k] = 0.0f;
  if (PER != 6) {
#pragma unroll
    for (int h = 0; h < PER / 4; ++h)
      if (pos + 4 * h < d) {
        const float4u x = *reinterpret_cast<const float4u*>(wgt + off + pos + 4 * h);
        xs[4 * h] = x.x; xs[4 * h + 1] = x.y; xs[4 * h + 2] = x.z; xs[4 * h + 3] = x.w;
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
  double wd[PER];  // clamped weights, then the amounts
  // the sum of the row as a plain fp64 sum where that is exact (plain_sum_is_exact); a wavefront in which some
  // group's is not falls back to the three-limb sum for all of its groups
  double Sd = 0.0;
  uint32_t mn = 0xFFFFFFFFu;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const float cw = masked_weight(xs[k], pos + k < d);
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
  const double scale = row_ok ? (double)d / Sd : 0.0;
  double fs = 1099511627776.0, neg_fs = -1099511627776.0;  // 2^40
  asm("" : "+v"(fs), "+v"(neg_fs));  // in registers: as literals they would be moved into every sum's place

  float op[PER];
  bool hv[PER];
  double run_d = 0.0, run_u = 0.0;  // deficits and surpluses of this lane's slots
  uint32_t cnt = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const double p = wd[k] * scale, t = fma(p, fs, neg_fs);  // = (p - 1) * 2^F rounded once: the product is exact
    hv[k] = t >= 0.5;
    const double heavy = hv[k] ? 1.0 : 0.0, light = hv[k] ? 0.0 : 1.0;
    wd[k] = rint(max_abs_f64(t, heavy));  // |t| < 0.5 for a light with t > 0: rounds to the deficit 0
    op[k] = (float)p;
    run_d = fma(wd[k], light, run_d);
    run_u = fma(wd[k], heavy, run_u);
    cnt += hv[k] ? 1u : 0u;
  }
  const double id = group_scan_f64<G>(run_d), iu = group_scan_f64<G>(run_u);
  const uint32_t ic = group_scan_u32<G>(cnt);
  const uint32_t nh = (uint32_t)__shfl((int)ic, (int)last_lane, 64), nl = SLOTS - nh;
  // A heavy keeps itself when its prefix lies above the deficits of the row's own lights (a slot behind the row counts 2^40), or
  // when it is the last, the only one whose prefix is all the surplus.
  const double most = lane_shfl_f64(fmin(fma((double)(SLOTS - d), neg_fs, id), iu - 1.0), (int)last_lane);
  uint32_t at[PER];  // of a light's entry, of the one below a heavy's
  bool self[PER];
  {
    const uint32_t ex_c = ic - cnt;
    uint32_t la = strip + SZ * (pos - ex_c), below = strip + SZ * (TOP - 1 - ex_c);
    double sh = iu - run_u, sl = id - run_d;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      at[k] = hv[k] ? below : la;
      self[k] = false;
      if (hv[k]) {
        sh += wd[k];
        val(below + SZ) = sh;
        slot_of(below + SZ) = (uint8_t)(pos + k);
        self[k] = sh > most;
        below -= SZ;
      } else {
        sl += wd[k];
        val(la) = sl;
        la += SZ;
      }
    }
    if (gl == G - 1) {
      val(strip + SZ * nl) = __builtin_huge_val();
      val(strip + SZ * (nl + 1)) = __builtin_huge_val();
    }
  }
  wave_lds_sync();
  if (gl == 0) slot_of(strip + SZ * (nl + 1)) = slot_of(strip + SZ * (nl + 2));  // a light beyond every heavy takes the last

  // merged positions [pos, pos + PER) belong to this lane; some lights, the next of which is at a, and pos less so many
  // heavies, the next of which is at q, come before them
  uint32_t a = strip + SZ * (pos > nh ? pos - nh : 0u);
  const uint32_t dq = SZ * (TOP - pos);
  {
    const uint32_t hi = strip + SZ * min(pos, nl);
#pragma unroll
    for (uint32_t step = 1u << (31 - __builtin_clz(SLOTS / 2)); step >= 1; step >>= 1) {
      if (step >= SLOTS / 8 && step > 1 && !__any(min(nh, nl) >= step)) continue;  // few heavies, or few lights: never so far apart
      const uint32_t to = min(a + SZ * step, hi);
      a = val(to - SZ) < val(to + dq) ? to : a;
    }
  }
  uint32_t q = a + dq;
  uint32_t to[PER], x[PER];
#pragma unroll
  for (int s = 0; s < PER; ++s) {
    const double vl = val(a), vh = val(q);
    const bool take = vh <= vl;  // the heavy
    const float p = (float)fma(vl - vh, -1.0 / 1099511627776.0, 1.0);
    const uint32_t an = a + SZ, qn = q - SZ;
    to[s] = take ? qn : an;
    x[s] = take ? __float_as_uint(p) : q;
    a = take ? a : an;
    q = take ? qn : q;
  }
  wave_lds_sync();
#pragma unroll
  for (int s = 0; s < PER; ++s) word(to[s]) = x[s];
  if (gl == 0) word(strip) = strip + SZ * TOP;  // the first light starts in the first heavy
  wave_lds_sync();

  uint32_t oa[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint32_t w = word(at[k]), m = slot_of(hv[k] ? at[k] : w);
    oa[k] = self[k] ? pos + k : m;
    if (hv[k]) op[k] = self[k] ? 1.0f : __uint_as_float(w);
  }
  if (__any(nh == 0)) {  // all weights alike, none that counts, or no row
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      if (nh == 0) oa[k] = row_ok ? pos + k : SKY_INVALID;
      if (!row_ok) op[k] = 0.0f;
    }
  }
  // the next row of this group reuses the strips: its writes must stay behind these reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  auto put = [&](uint32_t k, const uint4u& o) {  // slots k and k + 1
    if (k + 1 < d) *reinterpret_cast<uint4u*>(table + off + k) = o;
    else if (k < d) table[off + k] = AliasEntry{__uint_as_float(o.x), o.y};
  };
  if constexpr (PER == 8 && G >= 4) {  // a quad of lanes moves its 256 bytes as whole 64-byte pieces
    uint32_t v[4][4];
    quad_exchange(tid, op, oa, v);
#pragma unroll
    for (int h = 0; h < 4; ++h) put(PER * (gl & ~3u) + 8 * h + 2 * (gl & 3u), uint4u{v[h][0], v[h][1], v[h][2], v[h][3]});
  } else {
#pragma unroll
    for (int h = 0; h < PER / 2; ++h)
      put(pos + 2 * h, uint4u{__float_as_uint(op[2 * h]), oa[2 * h], __float_as_uint(op[2 * h + 1]), oa[2 * h + 1]});
    if (PER % 2 == 1 && pos + PER - 1 < d) table[off + pos + PER - 1] = AliasEntry{op[PER - 1], oa[PER - 1]};
  }
  return row_ok || d == 0;
}

// A row of one or two entries in closed form.  (The second weight loaded only where there is one, 40 M entries in rows of 1..100: 263 us, now 253.)
__device__ __forceinline__ bool tiny_row(uint32_t off, uint32_t d, const float* __restrict__ wgt,
                                         AliasEntry* __restrict__ table) {
  // a weight adds to the exact sum iff it is at least 2^-64
  constexpr float UNIT = 5.421010862427522170037e-20f;  // 2^-64
  const float2u pair = *reinterpret_cast<const float2u*>(wgt + off);  // both at once; the array has room behind its last entry
  const float w0 = clamp_weight(pair.x);
  if (d == 1) {
    const bool ok = w0 >= UNIT;
    table[off] = AliasEntry{ok ? 1.0f : 0.0f, ok ? 0u : SKY_INVALID};
    return ok;
  }
  const float w1 = clamp_weight(pair.y);
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
// 0..32 entries).  Nothing in here waits for another wavefront.
// Queue capacities: less than one batch left over plus the 64 vertices of a step, rounded up.  A queue entry is the row's
// offset and, in 16 bits, its degree (6 bits) above the vertex's position in the wavefront's range (10 bits): the vertex
// id itself is only needed for a row without weight, whose flag is cleared.  5 KB of LDS per wavefront: the kernel's
// registers decide how many fit a SIMD.
constexpr uint32_t SMALL_RANGE = 1024;  // most vertices per wavefront
constexpr uint32_t SMALL_BATCH[4] = {64, 64 / SHAPE_G2.lanes, 64 / SHAPE_G4.lanes, 64 / SHAPE_G8.lanes};
constexpr uint32_t small_cap(int q) { return (SMALL_BATCH[q] + 63 + 7) / 8 * 8; }
constexpr uint32_t SMALL_QBASE[4] = {0, small_cap(0), small_cap(0) + small_cap(1), small_cap(0) + small_cap(1) + small_cap(2)};
constexpr uint32_t SMALL_QTOTAL = SMALL_QBASE[3] + small_cap(3);
constexpr size_t smax(size_t a, size_t b) { return a > b ? a : b; }
// strips of the groups, the largest of three
constexpr size_t SMALL_STRIPS = smax(group_lds_bytes(SHAPE_G2.lanes, SHAPE_G2.per, 64),
                                     smax(group_lds_bytes(SHAPE_G4.lanes, SHAPE_G4.per, 64), group_lds_bytes(SHAPE_G8.lanes, SHAPE_G8.per, 64)));
static_assert(SMALL_STRIPS % 8 == 0);
constexpr size_t SMALL_LDS_BYTES = SMALL_STRIPS + SMALL_QTOTAL * 6;
// Vertices [lo, lo + per_wave) of the n (src null: the vertices themselves) by one wavefront.  `queues`: bit q set for the rows of queue q,
// rows of no entries with those of 1..2; the others are left to other wavefronts.
__device__ __forceinline__ void small_rows_range(uint32_t lo, const uint32_t* __restrict__ xadj, const float* __restrict__ wgt,
                                                 const uint32_t* __restrict__ src, uint32_t n, uint32_t per_wave,
                                                 AliasEntry* __restrict__ table, int8_t* __restrict__ valid,
                                                 uint64_t* __restrict__ smem, uint32_t queues = 15u) {
  uint32_t* q_off = reinterpret_cast<uint32_t*>(smem + SMALL_STRIPS / 8);  // [SMALL_QTOTAL]
  uint16_t* q_it = reinterpret_cast<uint16_t*>(q_off + SMALL_QTOTAL);  // [SMALL_QTOTAL]
  const uint32_t lane = threadIdx.x & 63;
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
    take(1, rows, SHAPE_G2.lanes, t, off, it, d);
    const bool ok = group_build_row<SHAPE_G2.lanes, SHAPE_G2.per, 64>(off, d, wgt, table, smem, t);
    if ((t & (SHAPE_G2.lanes - 1)) == 0 && !ok) clear_valid(it);
    cnt[1] -= rows;
  };
  auto build_g4 = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(2, rows, SHAPE_G4.lanes, t, off, it, d);
    const bool ok = group_build_row<SHAPE_G4.lanes, SHAPE_G4.per, 64>(off, d, wgt, table, smem, t);
    if ((t & (SHAPE_G4.lanes - 1)) == 0 && !ok) clear_valid(it);
    cnt[2] -= rows;
  };
  auto build_g8 = [&](uint32_t rows) {
    uint32_t t, off, it, d;
    take(3, rows, SHAPE_G8.lanes, t, off, it, d);
    const bool ok = group_build_row<SHAPE_G8.lanes, SHAPE_G8.per, 64>(off, d, wgt, table, smem, t);
    if ((t & (SHAPE_G8.lanes - 1)) == 0 && !ok) clear_valid(it);
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
      q = d <= 2 ? 0 : d <= 8 ? 1 : d <= 16 ? 2 : 3;
      if ((queues >> q) & 1) valid[v] = d != 0;  // a row without weight clears it when it is built
      else q = -1;
      if (d == 0) q = -1;
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
    while (cnt[1] >= SMALL_BATCH[1]) build_g2(SMALL_BATCH[1]);
    while (cnt[2] >= SMALL_BATCH[2]) build_g4(SMALL_BATCH[2]);
    while (cnt[3] >= SMALL_BATCH[3]) build_g8(SMALL_BATCH[3]);
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
// walks it.
//
// What bounds it is vector instructions, so
// - prefix sums are doubles (above);
// - slots behind the row's end in its last wavefront have weight 0 and go along as lights of deficit 2^40.  They come
//   after every light of the row, in rank and in the merged order, so nothing of the row depends on them, and no step
//   needs a mask; a heavy that only one of them reaches is one that nobody finishes;
// - a slot takes part in the compaction on the side of its kind alone;
// - the offsets of a step are those of the strips of group_build_row above: of the light and the heavy at hand and of the next ones,
//   and a step leaves the residual of the heavy that it takes: no pass over the heavies follows.
//
// LDS of a row: 10 bytes a slot (sum, slot of a heavy): the words take the place of the sums once every thread has walked its
// share.  That costs two barriers, and words apart (14 bytes) cost rows that reside on a CU.  200 M entries, before (a pass
// over the heavies, 12 or 14 bytes) / with 10 / with 14 bytes: rows of 230 692 / 730 / 690 us, 350 605 / 596 / 640, 500 585 / 573
// / -, 700 651 / 668 / 680, 1,400 637 / 680 / 650, 2,500 610 / 572 / -, 3,000 752 / 727 / 750, 3,500 758 / 635 / -, 4,800 750 / 675 / -.
constexpr bool merge_words(int rowt, int per) { return rowt * per == 256 || rowt * per == 1536; }
constexpr size_t merge_lds_bytes(int rowt, int per) { return (((size_t)rowt * per + 4) * (merge_words(rowt, per) ? 14 : 10) + 15) / 16 * 16; }

// The row `rr` by ROWT threads that share `smem` and, for the wavefronts' sums, s_aux[8 * ROWT / 64].  Returns false when its
// weights sum to zero.  All threads of the workgroup (the wavefront, for ROWT = 64) call it together; the arrays in LDS may
// be rewritten only after a barrier.
template <int ROWT, int PER>
__device__ __forceinline__ bool merge_row(const RowRef rr, uint64_t* smem, uint64_t* s_aux,
                                          const float* __restrict__ wgt, AliasEntry* __restrict__ table,
                                          const int tid = threadIdx.x) {
  constexpr int CAP = ROWT * PER;
  auto row_sync = [] {  // a row of one wavefront waits for no other: its workgroup may have more
    if (ROWT > 64) __syncthreads();
    else wave_lds_sync();
  };
  constexpr int NW = ROWT / 64;
  constexpr uint32_t TOP = CAP + 1, SZ = 8, B0 = SZ;  // light r at B0 + SZ * r, heavy h at B0 + SZ * (TOP - h)
  static_assert(CAP < 8000 && PER % 2 == 0, "sums of deficits below 2^53, offsets in 16 bits, whole pairs");
  char* const s_v = reinterpret_cast<char*>(smem);  // one more at either end is read
  constexpr bool WORDS = merge_words(ROWT, PER);
  char* const s_w = s_v + (CAP + 4) * SZ;
  char* const s_hs = WORDS ? s_w + (CAP + 4) * 4 : s_w;
  auto val = [&](uint32_t at) -> double& { return *reinterpret_cast<double*>(s_v + at); };
  auto word = [&](uint32_t at) -> uint32_t& { return *reinterpret_cast<uint32_t*>(WORDS ? s_w + (at >> 1) : s_v + at); };
  auto slot_of = [&](uint32_t at) -> uint16_t& { return *reinterpret_cast<uint16_t*>(s_hs + (at >> 2)); };

  const uint32_t off = rr.off, d = rr.d;
  const int wave = tid >> 6, lane = tid & 63;
  const uint32_t k0 = (uint32_t)PER * (uint32_t)tid, wfirst = PER * 64u * (uint32_t)wave;
  const bool wave_on = wfirst < d;
  const uint32_t slots = min((uint32_t)CAP, (d + PER * 64u - 1) / (PER * 64u) * (PER * 64u));  // of the wavefronts that are on

  double wd[PER];  // clamped weights, then the amounts
  // the sum of the row as a plain fp64 sum where that is exact (plain_sum_is_exact), else as three limbs
  double rsum = 0.0;
  uint32_t mn = 0xFFFFFFFFu;
  if (wave_on) {
    float xs[PER];
    wave_load<PER>(wgt + off, wfirst, d, s_v + PER * 256 * wave, lane, xs);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const float cw = clamp_weight(xs[j]);
      wd[j] = (double)cw;
      rsum += wd[j];
      mn = min(mn, __float_as_uint(cw) - 1u);
    }
    rsum = lane_f64(wave_scan_f64(rsum), 63);
    mn = wave_min_u32(mn);
  }
  if (NW > 1) {
    double* const s_sum = reinterpret_cast<double*>(s_aux);
    uint32_t* const s_mn = reinterpret_cast<uint32_t*>(s_aux + NW);
    if (lane == 0) {
      s_sum[wave] = rsum;
      s_mn[wave] = mn;
    }
    row_sync();
    rsum = s_sum[0];
    mn = s_mn[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      rsum += s_sum[i];
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
      WSum3* const s_w = reinterpret_cast<WSum3*>(s_aux + 2 * NW);
      if (lane == 0) s_w[wave] = sum;
      row_sync();
      sum = s_w[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) {
        sum.top += s_w[i].top;
        sum.mid += s_w[i].mid;
        sum.low += s_w[i].low;
      }
    }
    rsum = sum.top + sum.mid + sum.low != 0.0 ? wsum3_to_double(sum) : 0.0;
  }
  if (rsum == 0.0) {
    for (uint32_t k = tid; k < d; k += ROWT) table[off + k] = AliasEntry{0.0f, SKY_INVALID};
    return false;
  }

  float op[PER];
  bool hv[PER];
  double run_d = 0.0, run_u = 0.0;  // deficits and surpluses of this thread's slots
  uint32_t cnt = 0;
  if (wave_on) {
    const double scale = (double)d / rsum;
    double fs = 1099511627776.0, neg_fs = -1099511627776.0;  // 2^40
    asm("" : "+v"(fs), "+v"(neg_fs));  // in registers: as literals they would be moved into every sum's place
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const double p = wd[j] * scale, t = fma(p, fs, neg_fs);  // = (p - 1) * 2^F rounded once: the product is exact
      hv[j] = t >= 0.5;
      const double heavy = hv[j] ? 1.0 : 0.0, light = hv[j] ? 0.0 : 1.0;
      wd[j] = rint(max_abs_f64(t, heavy));  // |t| < 0.5 for a light with t > 0: rounds to the deficit 0
      op[j] = (float)p;
      run_d = fma(wd[j], light, run_d);
      run_u = fma(wd[j], heavy, run_u);
      cnt += hv[j] ? 1u : 0u;
    }
  }
  // what lies before this thread's slots, and in the whole row: deficits, surpluses, heavies
  double ex_d, ex_u, all_d, all_u;
  uint32_t ex_c, nh;
  {
    double* const s_p = reinterpret_cast<double*>(s_aux + 5 * NW);   // [2 * NW]
    uint32_t* const s_c = reinterpret_cast<uint32_t*>(s_aux + 7 * NW);  // [NW]
    const double id = wave_scan_f64(run_d), iu = wave_scan_f64(run_u);
    const uint32_t ic = group_scan_u32<64>(cnt);
    ex_d = id - run_d;
    ex_u = lane_before_f64(iu);  // not iu - run_u: a thread's own surpluses may take the prefix past 2^53
    ex_c = ic - cnt;
    if (NW == 1) {
      nh = (uint32_t)__builtin_amdgcn_readlane((int)ic, 63);
      all_d = lane_f64(id, 63);
      all_u = lane_f64(iu, 63);
    } else {
      if (lane == 63) {
        s_p[2 * wave] = id;
        s_p[2 * wave + 1] = iu;
        s_c[wave] = ic;
      }
      __syncthreads();
      nh = 0;
      all_d = all_u = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        if (w == wave) {
          ex_d += all_d;
          ex_u += all_u;
          ex_c += nh;
        }
        all_d += s_p[2 * w];
        all_u += s_p[2 * w + 1];
        nh += s_c[w];
      }
      nh = (uint32_t)__builtin_amdgcn_readfirstlane((int)nh);
    }
  }
  const uint32_t nl = slots - nh;  // the row's own come first: d - nh of them
  const uint32_t end_l = B0 + SZ * nl, end_h = B0 + SZ * (TOP - nh);
  // A heavy keeps itself when its prefix lies above the deficits of the row's own lights (a slot behind the row counts 2^40), or
  // when it is the last, the only one whose prefix is all the surplus.
  const double most = fmin(fma((double)(slots - d), -1099511627776.0, all_d), all_u - 1.0);
  uint32_t at[PER];  // of a light's entry, of the one below a heavy's
  bool self[PER];
  if (wave_on) {
    uint32_t la = B0 + SZ * (k0 - ex_c), below = B0 + SZ * (TOP - 1 - ex_c);
    double sl = ex_d, sh = ex_u;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      at[j] = hv[j] ? below : la;
      self[j] = false;
      if (hv[j]) {
        sh += wd[j];
        val(below + SZ) = sh;
        slot_of(below + SZ) = (uint16_t)(k0 + j);
        self[j] = sh > most;
        below -= SZ;
      } else {
        sl += wd[j];
        val(la) = sl;
        la += SZ;
      }
    }
    if (lane == 63 && k0 + PER == slots) {
      val(end_l) = __builtin_huge_val();
      val(end_h) = __builtin_huge_val();
    }
  }
  row_sync();

  uint32_t oa[PER];
  if (nh) {
    uint32_t to[PER], x[PER];
    if (wave_on) {
      // merged positions [k0, k0 + PER) belong to this thread; some lights, the next of which is at a, and k0 less so many
      // heavies, the next of which is at q, come before them
      const uint32_t hi = B0 + SZ * min(k0, nl), dq = SZ * (TOP - k0), fewer = min(nh, nl);
      uint32_t a = B0 + SZ * (k0 > nh ? k0 - nh : 0u);
#pragma unroll
      for (uint32_t step = 1u << (31 - __builtin_clz(CAP / 2)); step >= 1; step >>= 1) {
        if (step <= fewer) {  // uniform
          const uint32_t up = min(a + SZ * step, hi);
          a = val(up - SZ) < val(up + dq) ? up : a;
        }
      }
      uint32_t q = a + dq;
#pragma unroll
      for (int s = 0; s < PER; ++s) {
        const double vl = val(a), vh = val(q);
        const bool take = vh <= vl;  // the heavy
        const float p = (float)fma(vl - vh, -1.0 / 1099511627776.0, 1.0);
        const uint32_t an = a + SZ, qn = q - SZ;
        to[s] = take ? qn : an;
        x[s] = take ? __float_as_uint(p) : q;
        if (WORDS) word(to[s]) = x[s];
        a = take ? a : an;
        q = take ? qn : q;
      }
    }
    if (tid == 0) slot_of(end_h) = slot_of(end_h + SZ);  // a light beyond every heavy takes the last
    if (!WORDS) {
      row_sync();
      if (wave_on) {
#pragma unroll
        for (int s = 0; s < PER; ++s) word(to[s]) = x[s];
      }
    }
    if (tid == 0) word(B0) = B0 + SZ * TOP;  // the first light starts in the first heavy
    row_sync();
    if (wave_on) {
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const uint32_t w = word(at[j]), m = slot_of(hv[j] ? at[j] : w);
        oa[j] = self[j] ? k0 + j : m;
        if (hv[j]) op[j] = self[j] ? 1.0f : __uint_as_float(w);
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < PER; ++j) oa[j] = k0 + j;
  }
  if (!WORDS || NW == 1) row_sync();  // the entries take the place of the sums
  if (wave_on) wave_store<PER>(table + off, wfirst, d, s_v + PER * 512 * wave, lane, op, oa);
  return true;
}

}  // namespace sky
