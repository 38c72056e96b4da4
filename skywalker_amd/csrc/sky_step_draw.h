// The draw of one (walker, step) from a table that is never built: only entry `col` of the step's table is ever read, so
// the threads of a workgroup evaluate that entry alone, from the same prefix-sum definition the offline build uses:
//   pass 1  exact sum of the row's weights -> ledger, class of entry col
//           (a light col whose own share accepts the draw needs nothing more)
// in rows of up to 256 entries all of it by one wavefront, in registers (draw_wave), where the row type says so (Row::WAVE); in rows of up to 4 or
// 16 slots a thread (Row::HELD) and 4,095 entries
//   scan    of deficits and surpluses over the workgroup, whose prefixes each thread has for its own slots (draw_held)
// and in longer ones
//   pass 2  deficits and surpluses of every chunk of the row; their prefixes over the chunks
//   then    the one chunk that holds col gives the prefix up to col, and the one chunk in which the other kind's
//           prefix crosses it gives the slot (and the chunk with the next or last heavy that heavy)
// The result is bit for bit the draw from the fully built table.  The row's weights come from an object, so the
// same code serves node2vec's second-order weights, a graph's own weights and those of a bias operator linked in.
//
// What bounds it is latency: a walker's step is this chain, one after another.  Two sweeps of the row without a barrier
// inside and a constant number of steps after them replaced sweeps that synchronised the workgroup six times per 256
// slots (a row of 35,000 entries: 137 rounds).
#pragma once
#include "sky_common.h"

namespace sky {

// Vectors that are only 4-byte aligned: global loads of 16 bytes need no more on gfx950.
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int N2V_T = 256;
constexpr uint32_t NONE_SLOT = 0xFFFFFFFFu;
constexpr uint32_t DRAW_CHUNK = 256;  // slots a wavefront takes at a time: 4 consecutive ones per lane
constexpr int DRAW_CHUNKS = 256;      // most chunks of a row; longer rows have longer chunks (a power of two times 256)

template <int T>
struct DrawLds {
  uint64_t d[DRAW_CHUNKS], u[DRAW_CHUNKS];  // deficits and surpluses of every chunk, then their inclusive prefixes
  double fsum[T / 64];
  u128 sum[T / 64];
  uint32_t mn[T / 64];
  uint64_t key;
  uint32_t heavy[T / 64];
  uint32_t result;
};

__device__ __forceinline__ bool row_contains(const uint32_t* __restrict__ row, uint32_t n, uint32_t key) {
  uint32_t lo = 0, len = n;
  while (len > 0) {
    const uint32_t half = len >> 1;
    const uint32_t x = row[lo + half];
    if (x == key) return true;
    if (x < key) {
      lo += half + 1;
      len -= half + 1;
    } else {
      len = half;
    }
  }
  return false;
}

// Weights of the U times 256 slots from `base` on, four consecutive ones of each 256 per lane, zeros from `end` on.
template <int U, class Row>
__device__ __forceinline__ void row_weights(Row& row, uint32_t base, uint32_t end, bool again, float (&w)[U][4]) {
  const uint32_t k = base + 4 * (threadIdx.x & 63);
  if constexpr (U > 1) {
    row.many(k, end, again, w);
  } else {
    if (again) row.again(k, w[0]);
    else row.first(k, w[0]);
  }
}

// Rest of the draw below: column `col` of class `ec` with the acceptance number u.  SAT: the row's surpluses may wrap.
template <bool SAT, int T, class Row>
__device__ __forceinline__ uint32_t draw_entry(Row& row, const uint32_t d, const Ledger& L, const uint32_t col, const Entry& ec,
                                               const float u, const uint32_t csz, const uint32_t nc, const uint32_t k0,
                                               const uint32_t k1, DrawLds<T>& lds) {
  constexpr int NW = T / 64;
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // what depends on the lane number stays inside this form's code
  const uint32_t wave = tid >> 6, lane = tid & 63;
  // the four slots of this lane in the 256 from `base` on: amounts of the two kinds
  auto amounts = [&](uint32_t base, uint64_t (&dd)[4], uint64_t (&uu)[4]) {
    float w[4];
    row.again(base + 4 * lane, w);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool in = base + 4 * lane + k < d;
      const Entry e = classify_fast((double)w[k], in, L);
      dd[k] = in && !e.heavy ? e.amount : 0;
      uu[k] = e.heavy ? e.amount : 0;
    }
  };

  // pass 2: totals of the chunks
  {
    constexpr int U = Row::U;
    uint64_t sd = 0, su = 0;
    for (uint32_t base = k0; base < k1; base += DRAW_CHUNK * U) {
      float w[U][4];
      row_weights<U>(row, base, k1, true, w);
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint32_t at = base + DRAW_CHUNK * j;
        if (at >= k1) continue;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool in = at + 4 * lane + k < d;
          const Entry e = classify_fast((double)w[j][k], in, L);
          sd += in && !e.heavy ? e.amount : 0;
          su = add_sat<SAT>(su, e.heavy ? e.amount : 0);
        }
        if (((at + DRAW_CHUNK) & (csz - 1)) && at + DRAW_CHUNK < k1) continue;  // the chunk goes on
        sd = group_scan_u64<64>(sd);
        su = group_scan_sat_u64<64, SAT>(su);
        if (lane == 63) {
          const uint32_t c = at / csz;
          lds.d[c] = sd;
          lds.u[c] = su;
        }
        sd = su = 0;
      }
    }
  }
  __syncthreads();

  if (wave == 0) {
    {  // prefixes over the chunks: 4 consecutive ones per lane
      constexpr int PER = DRAW_CHUNKS / 64;
      uint64_t pd[PER], pu[PER], rd = 0, ru = 0;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const uint32_t c = lane * PER + j;
        rd += c < nc ? lds.d[c] : 0;
        ru = add_sat<SAT>(ru, c < nc ? lds.u[c] : 0);
        pd[j] = rd;
        pu[j] = ru;
      }
      const uint64_t bd = group_scan_u64<64>(rd) - rd, bu = before_own<SAT>(group_scan_sat_u64<64, SAT>(ru), ru);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        lds.d[lane * PER + j] = bd + pd[j];
        lds.u[lane * PER + j] = add_sat<SAT>(bu, pu[j]);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // first chunk of the row whose inclusive prefix in p exceeds key, nc if none
    auto chunk_above = [&](const uint64_t* p, uint64_t key) -> uint32_t {
#pragma unroll
      for (int j = 0; j < DRAW_CHUNKS / 64; ++j) {
        const uint32_t c = 64 * j + lane;
        const unsigned long long m = __ballot(c < nc && p[c] > key);
        if (m) return 64 * j + (uint32_t)__ffsll((long long)m) - 1;
      }
      return nc;
    };
    // first slot of chunk c whose inclusive prefix (of surpluses or deficits) exceeds key, and that prefix
    auto slot_above = [&](uint32_t c, bool surplus, uint64_t key, uint64_t& at) -> uint32_t {
      const uint64_t* p = surplus ? lds.u : lds.d;
      const uint32_t end = c + 1 == nc ? d : (c + 1) * csz;
      uint64_t before = c ? p[c - 1] : 0;
      for (uint32_t base = c * csz; base < end; base += DRAW_CHUNK) {
        uint64_t dd[4], uu[4], run[4];
        amounts(base, dd, uu);
        uint64_t t = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          t = add_sat<SAT>(t, surplus ? uu[k] : dd[k]);
          run[k] = t;
        }
        const uint64_t inc = group_scan_sat_u64<64, SAT>(t), mine = add_sat<SAT>(before, before_own<SAT>(inc, t));
        const unsigned long long m = __ballot(add_sat<SAT>(before, inc) > key);
        if (m) {
          const int l = __ffsll((long long)m) - 1;
          uint32_t k = 3;
          uint64_t x = add_sat<SAT>(mine, run[3]);
#pragma unroll
          for (int j = 2; j >= 0; --j)
            if (add_sat<SAT>(mine, run[j]) > key) {
              k = j;
              x = add_sat<SAT>(mine, run[j]);
            }
          at = shfl_u64(x, l);
          return (uint32_t)__shfl((int)(base + 4 * lane + k), l, 64);
        }
        before = add_sat<SAT>(before, shfl_u64(inc, 63));
      }
      // not reached while the weights stay what they were in pass 2; a bias operator that answers differently each
      // time must not keep the wavefront here
      at = key + 1;
      return end - 1;
    };
    // first (last) heavy slot of [from, end), both inside chunk c; NONE_SLOT if there is none
    auto heavy_in = [&](uint32_t c, uint32_t from, bool last) -> uint32_t {
      const uint32_t end = c + 1 == nc ? d : (c + 1) * csz;
      uint32_t got = NONE_SLOT;
      for (uint32_t base = c * csz; base < end; base += DRAW_CHUNK) {
        if (base + DRAW_CHUNK <= from) continue;
        uint64_t dd[4], uu[4];
        amounts(base, dd, uu);
        uint32_t mine = NONE_SLOT;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t slot = base + 4 * lane + k;
          if (uu[k] && slot >= from && (last || mine == NONE_SLOT)) mine = slot;
        }
        const unsigned long long m = __ballot(mine != NONE_SLOT);
        if (m) {
          const int l = last ? 63 - __clzll((long long)m) : __ffsll((long long)m) - 1;
          got = (uint32_t)__shfl((int)mine, l, 64);
          if (!last) break;
        }
      }
      return got;
    };

    // key: deficits before a light col, surpluses up to and with a heavy col
    const uint32_t cc = col / csz;
    uint64_t key = ec.heavy ? (cc ? lds.u[cc - 1] : 0) : (cc ? lds.d[cc - 1] : 0), part = 0;
    for (uint32_t base = cc * csz; base <= col; base += DRAW_CHUNK) {
      uint64_t dd[4], uu[4];
      amounts(base, dd, uu);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t slot = base + 4 * lane + k;
        part = add_sat<SAT>(part, ec.heavy ? (slot <= col ? uu[k] : 0) : (slot < col ? dd[k] : 0));
      }
    }
    key = add_sat<SAT>(key, shfl_u64(group_scan_sat_u64<64, SAT>(part), 63));

    uint32_t cand = col;
    const uint64_t total_u = lds.u[nc - 1];
    if (!ec.heavy) {
      // first heavy whose surplus prefix exceeds the key; the last heavy if there is none; col itself without any heavy
      const uint32_t cm = chunk_above(lds.u, key);
      if (cm < nc) {
        uint64_t at;
        cand = slot_above(cm, true, key, at);
      } else if (total_u) {
        cand = heavy_in(chunk_above(lds.u, total_u - 1), 0, true);
      }
    } else {
      // next heavy after col (none: col is the last heavy and keeps the draw), then the first light l with
      // SL(l) >= y: prob = (one + y - SL(l)) / one
      uint32_t nxt = col + 1 < d ? heavy_in(cc, col + 1, false) : NONE_SLOT;
      if (nxt == NONE_SLOT) {
        const uint32_t cn = chunk_above(lds.u, lds.u[cc]);
        if (cn < nc) nxt = heavy_in(cn, 0, false);
      }
      const uint32_t cl = nxt != NONE_SLOT ? chunk_above(lds.d, key - 1) : nc;
      if (cl < nc) {
        uint64_t sl = 0;
        (void)slot_above(cl, false, key - 1, sl);
        cand = u < residual_prob(L.one + key - sl, L) ? col : nxt;
      }
    }
    if (NW == 1) return cand;
    if (lane == 0) lds.result = cand;
  }
  __syncthreads();
  return lds.result;  // the next draw starts with a barrier
}

// The same for a row of at most 4 Q T slots, Q quads of consecutive ones a thread: one scan over the workgroup gives every prefix,
// the thread of col the key, and the thread whose prefixes it falls between the slot.  Three barriers and some 3,000 cycles, where the
// sweep over chunks and the chain on one wavefront behind it take 9,000 (counted in the table-per-step walk, rows of 800 entries on
// average).  The amounts of four quads held in registers would make them 147, three wavefronts to a SIMD: they are computed again.
// Up to HELD_MOST entries, whose surpluses add up to less than 2^64 whatever the weights (d times d, in shares of 2^40): a second form that saturates
// cost a walker of one wavefront 9 registers, which is the sixth wavefront to a SIMD (20,000 walkers x 4 without tables, scale 16, 78.5 -> 76.2 us).
// Longer rows have nothing to gain by it: where all rows have 4,097..8,191 entries, 200 walkers x 40 of 512 threads take 668 us with four quads a
// thread and 501 with the two sweeps (700 x 20 672 / 517; with windows 891 / 777 and, 500 x 20, 568 / 500), 1,500 x 20 of 256 threads through
// rows of 4,096 698 / 553.  Rows of 2,049..4,095 with two quads a thread of 512 instead of four: 200 x 40 365 -> 280, with windows 568 -> 478.
constexpr uint32_t HELD_MOST = 4095;
template <int Q, int T, class Row>
__device__ __forceinline__ uint32_t draw_held(Row& row, const uint32_t d, const Ledger& L, const uint32_t col, const Entry& ec,
                                              const float u, DrawLds<T>& lds) {
  constexpr int NW = T / 64, S = 4 * Q;
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // what depends on the lane number stays inside this form's code
  const uint32_t wave = tid >> 6, lane = tid & 63, k0 = S * tid, owner = col / S, own = col % S;
  // f(slot within the thread's, heavy, amount)
  uint64_t a[4];
  uint32_t ah = 0;
  auto each = [&](bool again, auto&& f) {
#pragma unroll 1
    for (int q = 0; q < Q; ++q) {
      if (Q > 1 || !again) {
        float w[4];
        row.again(k0 + 4 * q, w);
        ah = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const Entry e = classify_fast((double)w[k], k0 + 4 * q + k < d, L);
          a[k] = e.amount;
          ah |= (e.heavy ? 1u : 0u) << k;
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) f(4 * q + k, (ah >> k) & 1, a[k]);
    }
  };
  uint64_t sd = 0, su = 0;
  uint32_t heavy = 0;  // bit k: slot k0 + k
  each(false, [&](int k, bool h, uint64_t x) {
    heavy |= (h ? 1u : 0u) << k;
    sd += h ? 0 : x;
    su += h ? x : 0;
  });
  const uint64_t id = group_scan_u64<64>(sd), iu = group_scan_u64<64>(su);
  uint64_t bd = id - sd, bu = iu - su;  // before the thread's slots
  uint64_t tu = 0;                                      // surpluses of the row
  if (lane == 63) {
    lds.d[wave] = id;
    lds.u[wave] = iu;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const uint64_t x = lds.d[i], y = lds.u[i];
    tu += y;
    if (i < (int)wave) {
      bd += x;
      bu += y;
    }
  }
  if (tid == owner) {  // deficits before a light col, surpluses up to and with a heavy col
    uint64_t key = ec.heavy ? bu : bd;
    each(true, [&](int k, bool h, uint64_t x) {
      key += ec.heavy ? (h && k <= (int)own ? x : 0) : (!h && k < (int)own ? x : 0);
    });
    lds.key = key;
    lds.result = col;
  }
  // first (last) heavy slot of each wavefront among those in `mask`
  auto heavies = [&](uint32_t mask, bool last) {
    const unsigned long long m = __ballot(mask != 0);
    const int l = last ? 63 - __clzll((long long)(m | 1)) : __ffsll((long long)(m | 1ull << 63)) - 1;
    const uint32_t slot = (uint32_t)__shfl((int)(k0 + (last ? 31 - __clz((int)(mask | 1)) : __ffs((int)(mask | 1u << 31)) - 1)), l, 64);
    if (lane == 0) lds.heavy[wave] = m ? slot : NONE_SLOT;
  };
  if (ec.heavy) heavies(tid < owner ? 0u : tid == owner ? heavy & ~((2u << own) - 1u) : heavy, false);
  __syncthreads();
  const uint64_t key = lds.key;
  if (!ec.heavy) {
    // first heavy whose surplus prefix exceeds the key; the last heavy if there is none; col itself without any heavy
    if (key < tu) {
      if (bu <= key && key < bu + su) {
        uint32_t at = S;
        each(true, [&](int k, bool h, uint64_t x) {
          if (h) bu += x;
          at = at == S && bu > key ? k : at;
        });
        lds.result = min(k0 + at, d - 1);  // a bias operator may answer differently each time
      }
    } else if (tu) {
      heavies(heavy, true);
      __syncthreads();
      if (tid == 0) {
        uint32_t slot = NONE_SLOT;
#pragma unroll
        for (int i = 0; i < NW; ++i)
          if (lds.heavy[i] != NONE_SLOT) slot = lds.heavy[i];
        lds.result = slot;
      }
    }
  } else {
    // next heavy after col (none: col is the last heavy and keeps the draw), then the first light l with
    // SL(l) >= y: prob = (one + y - SL(l)) / one
    uint32_t nxt = NONE_SLOT;
#pragma unroll
    for (int i = 0; i < NW; ++i) nxt = min(nxt, lds.heavy[i]);
    if (nxt != NONE_SLOT && bd < key && key <= bd + sd) {
      uint64_t sl = 0;
      each(true, [&](int k, bool h, uint64_t x) {
        if (!h) bd += x;
        sl = sl == 0 && bd >= key ? bd : sl;  // the key of a heavy is at least 1
      });
      lds.result = u < residual_prob(L.one + key - sl, L) ? col : nxt;
    }
  }
  __syncthreads();
  return lds.result;
}

// Ledger of the row of d >= 1 entries by a workgroup of T, of which this wavefront has slots [k0, k1); false when the weights sum to
// zero.
template <int T, class Row, class Lds>
__device__ __forceinline__ bool row_ledger(Row& row, const uint32_t d, const uint32_t k0, const uint32_t k1, Lds& lds, Ledger& L) {
  constexpr int NW = T / 64, U = Row::U;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // pass 1: the sum as a plain fp64 sum where that is exact (plain_sum_is_exact), else in 128 bits
  double fsum = 0.0;
  uint32_t mn = 0xFFFFFFFFu;
  for (uint32_t base = k0; base < k1; base += DRAW_CHUNK * U) {
    float w[U][4];
    row_weights<U>(row, base, k1, false, w);
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (base + DRAW_CHUNK * j < k1)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          fsum += (double)w[j][k];
          mn = min(mn, __float_as_uint(w[j][k]) - 1u);
        }
  }
  fsum = group_sum_f64<64>(fsum);
  mn = wave_min_u32(mn);
  if (NW > 1) {
    if (lane == 0) {
      lds.fsum[wave] = fsum;
      lds.mn[wave] = mn;
    }
    __syncthreads();
    fsum = lds.fsum[0];
    mn = lds.mn[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      fsum += lds.fsum[i];
      mn = min(mn, lds.mn[i]);
    }
  } else {  // what first() has left in LDS
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (plain_sum_is_exact(fsum, mn)) {
    if (fsum == 0.0) return false;
    L = make_ledger_small(d, fsum);
    if (d >= (1u << 22)) {
      const int F = 62 - (31 - __clz((int)d));
      L.one = 1ull << F;
      L.fs = (double)L.one;
      L.inv_fs = 1.0 / L.fs;
    }
  } else {
    u128 sum{0, 0};
    for (uint32_t base = k0; base < k1; base += DRAW_CHUNK) {
      float w[4];
      row.again(base + 4 * lane, w);
#pragma unroll
      for (int k = 0; k < 4; ++k) sum = add128(sum, weight_fixed(w[k]));
    }
    sum = group_sum_u128<64>(sum);
    if (NW > 1) {
      if (lane == 0) lds.sum[wave] = sum;
      __syncthreads();
      sum = lds.sum[0];
#pragma unroll
      for (int i = 1; i < NW; ++i) sum = add128(sum, lds.sum[i]);
    }
    if ((sum.lo | sum.hi) == 0) return false;
    L = make_ledger(d, sum);
  }
  return true;
}

// The draw from a row of at most 64 S entries by one wavefront, S consecutive slots a lane: no barrier, no LDS, no sweep twice.  S is 4 for rows
// of up to WAVE_MOST entries, and 1 for those of up to 64 (table-per-step walks: 2,000 x 40 on the scale-18 graph 525 -> 507 us, on the scale-17
// graph 412 -> 392, 1,500 x 20 on the scale-14 graph with 5 edges a vertex 88 -> 80).
// In the table-per-step walk with a bit a vertex one wavefront of the workgroup draws for all (WAVE_ONE), from weights that it has tested bits for; the
// others wait for it and leave the SIMDs to the walkers beside.  A step from a row of 256 entries and fewer, half of all, takes 8,300 cycles instead of 11,000 (2,000 x
// 40 on the scale-18 graph 549 -> 518 us, on the scale-17 graph 449 -> 410, 200 x 40 there 254 -> 217).  With eight slots a lane a row of 300
// takes as long as by the workgroup, with sixteen a row of 950 takes longer (518 / 520 / 803 us).
// In the walk without tables every wavefront of the workgroup draws for itself, all the same slot, and no barrier is met (WAVE_EACH).  A workgroup
// of one wavefront has eight slots a lane for rows of 257 to 512 entries too (10,000 x 8 on the scale-22 graph 183.9 -> 180.3 us, while the 80
// registers of six wavefronts to a SIMD suffice: with what the compiler keeps of the sum for the amounts it spills, 181.5).  Sixteen for rows
// of up to 1,024 spill (217, and 183.5 with the slots in four strips and the amounts computed again).
// Not for rows whose weights only come in slot order, as a window in LDS moves along (N2vRow), or from an operator (FunctionRow): WAVE_NONE, untried.
// All lanes call it together.
constexpr uint32_t WAVE_MOST = 256;
enum WaveRows { WAVE_NONE, WAVE_ONE, WAVE_EACH };
__device__ __forceinline__ uint64_t lane_u64(uint64_t v, int lane) {
  return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane) << 32 |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}
// Ledger of a row of d >= 1 entries that the lanes of one wavefront hold, S each, zeros past the row; false when the weights sum to zero.
template <int S>
__device__ __forceinline__ bool wave_ledger(float (&w)[S], const uint32_t d, Ledger& L) {
  double fsum = 0.0;
  uint32_t most = 0;  // the complement of the least (weight bits - 1): what lanes without a source add to a scan, 0, changes nothing
#pragma unroll
  for (int k = 0; k < S; ++k) {
    fsum += (double)w[k];
    most = max(most, 0u - __float_as_uint(w[k]));
  }
  auto scan = [&](auto step) {
    step(std::integral_constant<int, DPP_ROW_SHR1>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, DPP_ROW_SHR2>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, DPP_ROW_SHR4>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, DPP_ROW_SHR8>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, DPP_ROW_BCAST15>{}, std::integral_constant<int, 0xA>{});
    step(std::integral_constant<int, DPP_ROW_BCAST31>{}, std::integral_constant<int, 0xC>{});
  };
  scan([&](auto ctrl, auto rows) {
    constexpr int C = decltype(ctrl)::value, R = decltype(rows)::value;
    fsum += __longlong_as_double((long long)dpp0_u64<C, R>((uint64_t)__double_as_longlong(fsum)));
    most = max(most, dpp0<C, R>(most));
  });
  fsum = __longlong_as_double((long long)lane_u64((uint64_t)__double_as_longlong(fsum), 63));
  most = (uint32_t)__builtin_amdgcn_readlane((int)most, 63);
  if (plain_sum_is_exact(fsum, ~most)) {
    if (fsum == 0.0) return false;
    L = make_ledger_small(d, fsum);
  } else {
    u128 sum{0, 0};
#pragma unroll
    for (int k = 0; k < S; ++k) {
      sum = add128(sum, weight_fixed(w[k]));
      if (S > 4 && k + 1 < S) asm volatile("" : "+v"(w[k + 1]), "+v"(sum.lo));  // one after another
    }
    sum = group_sum_u128<64>(sum);
    if ((sum.lo | sum.hi) == 0) return false;
    L = make_ledger(d, sum);
  }
  return true;
}
template <int S = 4, class Row>
__device__ __forceinline__ uint32_t draw_wave(Row& row, const uint32_t d, const uint32_t rx, const float u) {
  const uint32_t lane = threadIdx.x & 63, k0 = S * lane;
  float w[S];
  row.load(k0, w);
  Ledger L;
  if (!wave_ledger(w, d, L)) return NONE_SLOT;
  if (S > 4) {  // the doubles of the sum are not kept for the amounts
#pragma unroll
    for (int k = 0; k < S; ++k) asm volatile("" : "+v"(w[k]));
  }
  const uint32_t col = __umulhi(rx, d), j = col % S;
  float wc = w[0];
#pragma unroll
  for (int k = 1; k < S; ++k) wc = j == (uint32_t)k ? w[k] : wc;
  const Entry ec = classify_fast((double)__uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(wc), (int)(col / S))), true, L);
  const bool heavy = __builtin_amdgcn_readfirstlane(ec.heavy ? 1 : 0);
  if (!heavy && u < (float)ec.p) return col;  // the light keeps the draw: its alias is never read
  uint64_t a[S];
  uint32_t h = 0;  // bit k: slot k0 + k is heavy
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const Entry e = classify_fast((double)w[k], k0 + k < d, L);
    a[k] = e.amount;
    h |= (e.heavy ? 1u : 0u) << k;
  }
  // deficits before a light col, surpluses up to and with a heavy col
  uint64_t key = 0;
#pragma unroll
  for (int k = 0; k < S; ++k) key += ((h >> k) & 1) == (heavy ? 1u : 0u) && (heavy ? k0 + k <= col : k0 + k < col) ? a[k] : 0;
  key = lane_u64(group_scan_u64<64>(key), 63);
  // first slot of a kind whose inclusive prefix exceeds `past`, and that prefix; NONE_SLOT if there is none
  uint64_t at = 0;
  auto above = [&](uint32_t kind, uint64_t past) -> uint32_t {
    uint64_t run[S], t = 0;
#pragma unroll
    for (int k = 0; k < S; ++k) {
      t += ((h >> k) & 1) == kind ? a[k] : 0;
      run[k] = t;
    }
    const uint64_t inc = group_scan_u64<64>(t), before = inc - t;
    const unsigned long long m = __ballot(inc > past);
    if (!m) return NONE_SLOT;
    const int l = __ffsll((long long)m) - 1;
    uint32_t k = S - 1;
    uint64_t x = inc;
#pragma unroll
    for (int i = S - 2; i >= 0; --i)
      if (before + run[i] > past) {
        k = i;
        x = before + run[i];
      }
    at = lane_u64(x, l);
    return S * (uint32_t)l + (uint32_t)__builtin_amdgcn_readlane((int)k, l);
  };
  if (!heavy) {
    // first heavy whose surplus prefix exceeds the key; the last heavy if there is none; col itself without any heavy
    const uint32_t s = above(1, key);
    if (s != NONE_SLOT) return s;
    const unsigned long long m = __ballot(h != 0);
    if (!m) return col;
    const int l = 63 - __clzll((long long)m);
    return S * (uint32_t)l + 31u - (uint32_t)__clz(__builtin_amdgcn_readlane((int)h, l));
  }
  // next heavy after col (none: col is the last heavy and keeps the draw), then the first light l with SL(l) >= key:
  // prob = (one + key - SL(l)) / one
  const uint32_t after = k0 > col ? h : k0 + S - 1 <= col ? 0u : h & ~((2u << j) - 1u);
  const unsigned long long m = __ballot(after != 0);
  if (!m || above(0, key - 1) == NONE_SLOT) return col;
  const int l = __ffsll((long long)m) - 1;
  return u < residual_prob(L.one + key - at, L) ? col : S * (uint32_t)l + (uint32_t)__ffs(__builtin_amdgcn_readlane((int)after, l)) - 1u;
}

// Row-local slot that (walker, step) with random numbers r draws from the row of d >= 1 entries, or NONE_SLOT when
// their weights sum to zero.  Called by every thread of a workgroup of T.  `row`:
//   row.first(k, w)   clamped weights of slots k .. k + 3 (k a multiple of 4; zeros past the row).  A wavefront goes
//                     through its part of the row in slot order, once, all lanes together (k advances by 4 per lane)
//   row.again(k, w)   the same, afterwards, for any slots and by any wavefront
//   Row::U            how many times 256 slots are in flight at once; if that is more than one, instead of first():
//   row.many(k, end, again, w)  slots k + 256 j .. k + 256 j + 3 for j < U, zeros from slot `end` on, in both sweeps
//   Row::WAVE         whether rows of up to WAVE_MOST entries (twice that for WAVE_EACH and T = 64) go to draw_wave, and then instead of all these:
//   row.load(k, w)    clamped weights of slots k, k + 1, .. of one lane (zeros past the row), as many as w holds: 1, 4 or 8
//   Row::HELD         0, 4 or 16: rows of up to so many slots a thread (HELD_MOST entries at most, 8 slots a thread of 512) by draw_held
template <int T, class Row>
__device__ __forceinline__ uint32_t draw_slot(Row& row, const uint32_t d, const u32x4& r, DrawLds<T>& lds) {
  constexpr int NW = T / 64;
  const uint32_t wave = threadIdx.x >> 6;
  if constexpr (Row::WAVE == WAVE_EACH) {
    if (d <= WAVE_MOST) return draw_wave<4>(row, d, r.x, u24(r.y));
    if constexpr (NW == 1) {
      if (d <= 2 * WAVE_MOST) return draw_wave<8>(row, d, r.x, u24(r.y));
    }
  }
  uint32_t csz = DRAW_CHUNK;
  while ((uint64_t)csz * DRAW_CHUNKS < d) csz *= 2;
  const uint32_t nc = (uint32_t)(((uint64_t)d + csz - 1) / csz), cpw = (nc + NW - 1) / NW;
  const uint32_t c0 = wave * cpw, c1 = min(nc, c0 + cpw);
  __syncthreads();  // the draw before has been read by everyone
  if constexpr (Row::WAVE == WAVE_ONE) {
    if (d <= WAVE_MOST) {
      static_assert(NW > 1, "a wavefront alone goes on as it is");
      if (wave == (blockIdx.x & (NW - 1))) {  // not always on the same SIMD
        const uint32_t cand = d <= 64 ? draw_wave<1>(row, d, r.x, u24(r.y)) : draw_wave<4>(row, d, r.x, u24(r.y));
        if ((threadIdx.x & 63) == 0) lds.result = cand;
      }
      __syncthreads();
      return lds.result;
    }
  }
  const uint32_t k0 = c0 < nc ? c0 * csz : d, k1 = c0 < nc ? (c1 == nc ? d : c1 * csz) : d;  // this wavefront's slots

  Ledger L;
  if (!row_ledger<T>(row, d, k0, k1, lds, L)) return NONE_SLOT;
  const uint32_t col = __umulhi(r.x, d);
  const float u = u24(r.y);
  Entry ec;
  {
    float w[4];
    row.again(col & ~3u, w);
    const uint32_t j = col & 3u;
    ec = classify_fast((double)(j == 0 ? w[0] : j == 1 ? w[1] : j == 2 ? w[2] : w[3]), true, L);
  }
  if (!ec.heavy && u < (float)ec.p) return col;  // the light keeps the draw: its alias is never read

  if constexpr (Row::HELD == 0) {
    return surpluses_may_wrap(L.scale) ? draw_entry<true, T>(row, d, L, col, ec, u, csz, nc, k0, k1, lds)
                                       : draw_entry<false, T>(row, d, L, col, ec, u, csz, nc, k0, k1, lds);
  }
  if constexpr (Row::WAVE == WAVE_NONE || 4 * T > WAVE_MOST) {
    if (d <= std::min(4u * T, HELD_MOST)) return draw_held<1, T>(row, d, L, col, ec, u, lds);
  }
  if constexpr (Row::HELD == 16) {
    constexpr uint32_t Q = T >= 512 ? 2 : 4;
    if (d <= std::min(4 * Q * T, HELD_MOST)) return draw_held<Q, T>(row, d, L, col, ec, u, lds);
  }
  if (surpluses_may_wrap(L.scale)) return draw_entry<true, T>(row, d, L, col, ec, u, csz, nc, k0, k1, lds);
  return draw_entry<false, T>(row, d, L, col, ec, u, csz, nc, k0, k1, lds);
}

// The graph's own weights of a row (the weight array has 16 spare bytes, so four slots can be read from any).
struct PlainRow {
  static constexpr int U = 4;
  static constexpr WaveRows WAVE = WAVE_EACH;
  static constexpr int HELD = 4;
  const float* w;
  uint32_t d;
  __device__ __forceinline__ void load(uint32_t k, float (&x)[4]) const { again(k, x); }
  __device__ __forceinline__ void load(uint32_t k, float (&x)[8]) const {
    float a[4], b[4];
    again(k, a);
    again(k + 4, b);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      x[t] = a[t];
      x[4 + t] = b[t];
    }
  }
  __device__ __forceinline__ void load(uint32_t k, float (&x)[1]) const { x[0] = masked_weight(w[min(k, d - 1)], k < d); }
  // Branches that a wavefront takes as one: all loads are on their way before the first is waited for.
  __device__ __forceinline__ void many(uint32_t k, uint32_t end, bool, float (&x)[U][4]) const {
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
    float4u q[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      q[j] = float4u{0, 0, 0, 0};
      if (first + 256u * j < end) q[j] = *reinterpret_cast<const float4u*>(w + min(k + 256u * j, (d - 1) & ~3u));
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) x[j][t] = masked_weight(q[j][t], k + 256u * j + t < end);
  }
  __device__ __forceinline__ void again(uint32_t k, float (&x)[4]) const {
    const float4u q = *reinterpret_cast<const float4u*>(w + min(k, (d - 1) & ~3u));
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = masked_weight(q[t], k + t < d);
  }
};

// A row whose weights are computed by a function of the slot (row(k): clamped weight of slot k < d): those of a row of up
// to CAP entries stay in LDS after the first pass, those of a longer one are computed again.
constexpr uint32_t FN_CACHE = 4096;
template <class Fn>
struct FunctionRow {
  static constexpr int U = 1;
  static constexpr WaveRows WAVE = WAVE_NONE;
  static constexpr int HELD = 0;  // the operator is called where it is linked in: node2vec's, 8,000 walkers x 20, scale 16, 5.5 ms, 6.0 with
  Fn fn;
  uint32_t d;
  float* cache;  // [FN_CACHE]
  __device__ __forceinline__ void first(uint32_t k, float (&w)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w[j] = k + j < d ? fn(k + j) : 0.0f;
      if (d <= FN_CACHE && k + j < d) cache[k + j] = w[j];
    }
  }
  __device__ __forceinline__ void again(uint32_t k, float (&w)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = k + j < d ? (d <= FN_CACHE ? cache[k + j] : fn(k + j)) : 0.0f;
  }
};

}  // namespace sky
