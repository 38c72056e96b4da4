// k-hop neighbour sampling (replaces the fused sample_kernel and OfflineSample of
// src/offline_sample.cu:72-141,443-513, and sample_kernel / OnlineGBSampleNew of
// src/online_sample_new.cu:191-270,459-547).
//
// Output layout (include/sampler_result.cuh:226-260,421-426): per seed, hop h occupies
// width[h] = prod fanout[0..h] slots starting at offsets[h]; the children of slot s of hop h are
// slots s*fanout[h+1].. of hop h+1; sample_lengths holds one count per parent slot of every hop
// but the last.  A parent of degree deg with fanout k contributes all its neighbours when
// k >= deg, else k alias draws with replacement; draw i of slot s uses
// Philox(seed; seed index, s*k + i, h, DOM_SAMPLE).  One workgroup per start vertex takes it through all
// hops (or through one, when the rows of the next hop are built in between): no device-side queues, and the
// result does not depend on scheduling.
//
// Online mode builds the table of every distinct frontier vertex, once, through the same
// kernels as the offline build (into the graph's table storage), then samples the hop; or, where that takes less (choose_direct),
// evaluates the draws of a hop from the weights.
#include <algorithm>
#include <functional>
#include <memory>
#include <vector>

#include "sky_build_fused.h"
#include "sky_graph.h"
#include "sky_step_draw.h"

namespace sky {

struct HopGeom {
  uint32_t h, k, fan_h;          // hop index, fanout of the next hop, fanout of this hop
  uint64_t width, off, off_next; // slots of hop h, where they start, where hop h+1 starts
  uint64_t loff, loff_prev;      // sample_lengths offsets of hop h and h-1
  uint64_t lps, slen;            // per-seed strides of data and sample_lengths
};

__device__ __forceinline__ bool slot_filled(const HopGeom& g, const uint32_t* sl, uint64_t si, uint64_t s) {
  if (g.h == 0) return true;
  // slots of a hop fit 32 bits (sky_sample_layout checks the fanout product)
  const uint32_t s32 = (uint32_t)s;
  return sl[si * g.slen + g.loff_prev + s32 / g.fan_h] > s32 % g.fan_h;
}

constexpr uint32_t SAMPLE_HOPS = 7;  // sky_sample_layout takes at most 8 levels
struct SampleArgs {
  const uint32_t *xadj, *adjncy;
  const AliasEntry* table;
  const int8_t* valid;
  const uint32_t* seeds;  // read at hop 0, whose slots this kernel then writes; null: they are in place
  uint32_t *data, *sl;
  uint32_t* totals;  // children of a start vertex over all hops so far (null: not wanted)
  uint32_t V, h0, h1;  // hops [h0, h1)
  uint32_t parts;      // workgroups per start vertex (1 unless h1 == h0 + 1)
  uint32_t lanes;      // lanes per start vertex (a power of two; 64 when parts > 1)
  uint64_t first, N;   // start vertices [first, N)
  CallDevice* call;    // stamped by the call's first kernel (null: another kernel was)
  CallDevice* words;   // without tables: where a hop is refused (null: none is)
  uint64_t seed;
  HopGeom hop[SAMPLE_HOPS];
};

// The parent in slot s of hop g.h, V when the slot is not filled.
__device__ __forceinline__ uint32_t parent_of(const SampleArgs& a, const HopGeom& g, uint64_t si, uint32_t s) {
  if (g.h == 0 && a.seeds) return a.seeds[si];
  const uint32_t v = a.data[si * g.lps + g.off + s];  // beside the count that says whether it is one
  return slot_filled(g, a.sl, si, s) ? v : 0xFFFFFFFFu;
}

// Children with replacement: one lane per (slot, draw), U of them at a time so that their chains of four dependent
// loads overlap.  What bounds a hop is that chain, not its bytes; a wavefront for itself is the cheapest unit that
// waits for it: no barrier between hops, and the hops of one start vertex follow one another without the rest of the
// batch (one launch per hop over all slots, filled or not, took 117 us for the 40,000 x 25 x 10 batch on the scale-22
// graph, most of its 10 M lanes idle).
constexpr int SAMPLE_T = 64, SAMPLE_U = 4;
__global__ __launch_bounds__(SAMPLE_T) void sample_draw_kernel(SampleArgs a) {
  constexpr int U = SAMPLE_U;
  if (a.h0 == 0) call_stamp(a.call);
  // start vertices with few draws share the wavefront, a.lanes lanes each
  const uint32_t T = a.lanes, tid = threadIdx.x & (T - 1), part = blockIdx.x % a.parts;
  const uint64_t si = a.first + (uint64_t)(blockIdx.x / a.parts) * (SAMPLE_T / T) + threadIdx.x / T;
  const bool own = si < a.N;
  uint32_t mine = 0;
  for (uint32_t h = a.h0; h < a.h1; ++h) {
    const HopGeom& g = a.hop[h];
    const uint64_t total = g.width * g.k;  // at most 2^32
    if (h == 0 && a.seeds && part == 0 && tid == 0 && own) a.data[si * g.lps] = a.seeds[si];
    for (uint64_t j0 = (uint64_t)part * (T * U); j0 < total; j0 += (uint64_t)a.parts * (T * U)) {
      uint32_t s[U], i[U], v[U], o[U], deg[U], cand[U], child[U];
      bool in[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t j = j0 + u * T + tid;
        in[u] = own && j < total;
        s[u] = (uint32_t)j / g.k;
        i[u] = (uint32_t)j - s[u] * g.k;
        v[u] = in[u] ? parent_of(a, g, si, s[u]) : 0xFFFFFFFFu;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        o[u] = deg[u] = 0;
        if (v[u] < a.V) {
          o[u] = a.xadj[v[u]];
          deg[u] = a.xadj[v[u] + 1] - o[u];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // a row without weight has no children: its entries say so where one is drawn, its flag where all are copied
        cand[u] = SKY_INVALID;
        if (deg[u] > g.k) {
          const u32x4 r = philox(a.seed, (uint32_t)si, s[u] * g.k + i[u], g.h, DOM_SAMPLE);
          const uint32_t col = __umulhi(r.x, deg[u]);
          const AliasEntry e = a.table[o[u] + col];
          cand[u] = u24(r.y) < e.prob ? col : e.alias;
        } else if (deg[u]) {
          if (!a.valid[v[u]]) deg[u] = 0;
          if (i[u] < deg[u]) cand[u] = i[u];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        child[u] = 0;
        if (cand[u] != SKY_INVALID) child[u] = a.adjncy[o[u] + cand[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (!in[u]) continue;
        if (cand[u] != SKY_INVALID) a.data[si * g.lps + g.off_next + (uint64_t)s[u] * g.k + i[u]] = child[u];
        if (i[u] == 0) {
          const uint32_t cnt = cand[u] != SKY_INVALID ? min(deg[u], g.k) : 0u;
          a.sl[si * g.slen + g.loff + s[u]] = cnt;
          mine += cnt;
        }
      }
    }
    if (h + 1 < a.h1) {  // the next hop reads what this wavefront has just written
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  }
  if (a.totals) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const uint32_t o = (uint32_t)__shfl_xor((int)mine, m, 64);
      if ((uint32_t)m < T) mine += o;
    }
    if (tid == 0 && own) a.totals[si] = (a.h0 ? a.totals[si] : 0u) + mine;
  }
}

// Online, without a table: the children of a slot from the weights of its row, by T threads that have S consecutive slots of it each.
// With the deficits and surpluses up to the last of them in LDS every lane evaluates a draw of its own, by searches over the threads'
// prefixes and the slots of the one they end at.
template <int T>
struct DirectLds {
  uint64_t d[T], u[T];  // inclusive prefixes by thread
  u128 sum[T / 64];
  double fsum[T / 64];
  uint64_t wd[T / 64], wu[T / 64];
  uint32_t mn[T / 64], any;
};
// Children that the row of d > 0 entries yields: g.k, d if it has no more, none if they weigh nothing.  tid: of the T threads, a
// workgroup or one of its wavefronts.
template <int T>
__device__ __forceinline__ uint32_t direct_children(const SampleArgs& a, const HopGeom& g, const float* __restrict__ wgt, uint64_t si,
                                                    uint32_t s, uint32_t off, uint32_t d, uint32_t tid, DirectLds<T>& lds) {
  constexpr int NW = T / 64;
  const uint32_t wave = tid >> 6, lane = tid & 63;
  const uint32_t* const nbr = a.adjncy + off;
  uint32_t* const out = a.data + si * g.lps + g.off_next + (uint64_t)s * g.k;
  PlainRow row{wgt + off, d};
  auto sync = [] {
    if constexpr (NW > 1) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  };
  sync();  // the row before has been drawn from
  if (d <= g.k) {
    // all of them, of a row that weighs something: 2^-64 is the least a weight counts for
    bool any = false;
    for (uint32_t k = tid; k < d; k += T) any = any || clamp_weight(row.w[k]) >= 5.421010862427522e-20f;
    if (NW > 1) {
      if (tid == 0) lds.any = 0;
      __syncthreads();
      if (any) lds.any = 1;
      __syncthreads();
      any = lds.any;
    } else {
      any = __any(any);
    }
    if (!any) return 0;
    for (uint32_t k = tid; k < d; k += T) out[k] = nbr[k];
    return d;
  }
  // A slot a lane: what a draw reads is there already, and its only chain is one search in LDS (30,000 seeds x 20 on the scale-22 graph with 20
  // edges a vertex 77.4 -> 72.0 us, 8,000 x 20 on the scale-16 graph 40.8 -> 39.2, 8,000 x 15,10,5 on the scale-21 graph 292.7 -> 287.8).
  if (NW == 1 && d <= 64) {
    float w[1];
    row.load(tid, w);
    const uint32_t next = nbr[min(tid, d - 1)];
    Ledger L;
    if (!wave_ledger(w, d, L)) return 0;
    const Entry e = classify_fast((double)w[0], tid < d, L);
    const unsigned long long heavies = __ballot(e.heavy);
    const float p = (float)e.p;
    lds.d[tid] = group_scan_u64<64>(e.heavy ? 0 : e.amount);
    lds.u[tid] = group_scan_u64<64>(e.heavy ? e.amount : 0);
    sync();
    const uint64_t total_u = lds.u[63], total_d = lds.d[63];
    // fewer draws than entries, so one a lane; all lanes together: they have the row
    const u32x4 r = philox(a.seed, (uint32_t)si, s * g.k + tid, g.h, DOM_SAMPLE);
    const uint32_t col = __umulhi(r.x, d);
    const float u = u24(r.y);
    const bool heavy = heavies >> col & 1, kept = u < __shfl(p, (int)col, 64);
    uint32_t cand = col;
    if (!heavy && !kept) {
      // first heavy whose surplus prefix exceeds the deficits before col; the last heavy if there is none; col itself without any heavy
      if (total_u) cand = first_greater(lds.u, 0, 64, min(col ? lds.d[col - 1] : 0, total_u - 1));
    } else if (heavy) {
      // the first light l with SL(l) >= the key, and the next heavy: prob = (one + key - SL(l)) / one
      const uint64_t key = lds.u[col];
      if (key < total_u && key <= total_d && !(u < residual_prob(L.one + key - lds.d[first_greater(lds.d, 0, 64, key - 1)], L)))
        cand = col + (uint32_t)__ffsll((long long)(heavies >> (col + 1)));
    }
    const uint32_t child = (uint32_t)__shfl((int)next, (int)cand, 64);
    if (tid < g.k) out[tid] = child;
    return g.k;
  }
  uint32_t csz = DRAW_CHUNK;
  while ((uint64_t)csz * NW < d) csz *= 2;
  const uint32_t k0 = (uint32_t)min((uint64_t)d, (uint64_t)wave * csz), k1 = (uint32_t)min((uint64_t)d, (uint64_t)(wave + 1) * csz);
  Ledger L;
  if (!row_ledger<T>(row, d, k0, k1, lds, L)) return 0;
  const uint32_t S = ((d - 1) / T + 4) & ~3u;
  // f(slot, heavy, amount) of the slots [from, to), `from` a multiple of 4, until it says true
  auto slots = [&](uint32_t from, uint32_t to, auto&& f) {
    auto go = [&](auto quads) {  // that are requested together
      constexpr int Q = decltype(quads)::value;
      for (uint32_t k = from; k < to; k += 4 * Q) {
        float w[Q][4];
#pragma unroll
        for (int q = 0; q < Q; ++q) row.again(k + 4 * q, w[q]);
#pragma unroll
        for (int j = 0; j < 4 * Q; ++j) {
          const Entry e = classify_fast((double)w[j / 4][j % 4], k + j < d, L);
          if (k + j < to && f(k + j, e.heavy, e.amount)) return;
        }
      }
    };
    if (S > 4) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 1>{});
  };
  uint64_t sd = 0, su = 0;
  const uint32_t own = (uint32_t)min((uint64_t)d, (uint64_t)tid * S), end = (uint32_t)min((uint64_t)d, (uint64_t)(tid + 1) * S);
  slots(own, end, [&](uint32_t, bool heavy, uint64_t x) {
    sd += heavy ? 0 : x;
    su = add_sat<true>(su, heavy ? x : 0);
    return false;
  });
  sd = group_scan_u64<64>(sd);
  su = group_scan_sat_u64<64, true>(su);
  if (NW > 1) {
    if (lane == 63) {
      lds.wd[wave] = sd;
      lds.wu[wave] = su;
    }
    sync();
#pragma unroll
    for (int i = 0; i + 1 < NW; ++i)
      if (i < (int)wave) {
        sd += lds.wd[i];
        su = add_sat<true>(su, lds.wu[i]);
      }
  }
  lds.d[tid] = sd;
  lds.u[tid] = su;
  sync();
  const uint64_t total_u = lds.u[T - 1], total_d = lds.d[T - 1];
  // first slot of the kind whose inclusive prefix exceeds the key, which the kind's total does, and that prefix
  auto above = [&](bool surplus, uint64_t key, uint64_t& at) -> uint32_t {
    const uint64_t* p = surplus ? lds.u : lds.d;
    const uint32_t t = first_greater(p, 0, T, key);
    uint64_t run = t ? p[t - 1] : 0;
    uint32_t got = d - 1;
    slots(t * S, (uint32_t)min((uint64_t)d, (uint64_t)(t + 1) * S), [&](uint32_t k, bool heavy, uint64_t x) {
      if (heavy == surplus) run = add_sat<true>(run, x);
      if (run > key) got = k;
      return run > key;
    });
    at = run;
    return got;
  };
  for (uint32_t i = tid; i < g.k; i += T) {
    const u32x4 r = philox(a.seed, (uint32_t)si, s * g.k + i, g.h, DOM_SAMPLE);
    const uint32_t col = __umulhi(r.x, d), t = col / S;
    const float u = u24(r.y);
    // deficits before a light col, surpluses up to and with a heavy col
    uint64_t key_d = t ? lds.d[t - 1] : 0, key_u = t ? lds.u[t - 1] : 0;
    bool heavy = false;
    float p = 0.0f;
    {
      float w[4];
      row.again(col & ~3u, w);
      const uint32_t j = col & 3u;
      const Entry e = classify_fast((double)(j == 0 ? w[0] : j == 1 ? w[1] : j == 2 ? w[2] : w[3]), true, L);
      heavy = e.heavy;
      p = (float)e.p;
    }
    uint32_t cand = col;
    if (heavy || !(u < p)) {
      slots(t * S, col + 1, [&](uint32_t k, bool h, uint64_t x) {
        if (h) key_u = add_sat<true>(key_u, x);
        else if (k < col) key_d += x;
        return false;
      });
      uint64_t at;
      if (!heavy) {
        // first heavy whose surplus prefix exceeds the key; the last heavy if there is none; col itself without any heavy
        if (total_u) cand = above(true, min(key_d, total_u - 1), at);
      } else if (key_u < total_u && key_u <= total_d) {
        // the first light l with SL(l) >= the key, and the next heavy: prob = (one + key - SL(l)) / one
        (void)above(false, key_u - 1, at);
        if (!(u < residual_prob(L.one + key_u - at, L))) cand = above(true, key_u, at);
      }
    }
    out[i] = nbr[cand];
  }
  return g.k;
}

constexpr int DIRECT_T = 512;
constexpr uint32_t DIRECT_LONG = 1024;

// Whether a hop is drawn from the weights after all.  Its parents are the caller's: well connected vertices, or one of them again and
// again, whose rows are swept for every slot where a build makes each once, and long ones with the whole GPU.  Refused
// is a hop with a workgroup of more than `most_chain` entries in long rows, counting DIRECT_PER_ROW more for each (they follow one another,
// 1.1 ns each), or with more than `budget` entries altogether (18 ps each).  The answer reaches the host while the draws run, which are
// 4 to 8 us later for it.  (All hops from tables / from the weights whatever they meet / by this rule, us.  8,192 seeds x 20, the scale-16
// graph, any vertices 55 / 38 / 44, the first 8,192 64 / 106 / 73, ends of edges 67 / 127 / 78, one vertex of 12,938 entries 138 / 432 / 147;
// the scale-22 graph with 32 edges a vertex 91 / 46 / 53, 221 / 989 / 231, 406 / 846 / 399, one of 319,795 161 / 7,192 / 184.  1,024 x 10 x
// 10 there 360 / 332 / 323, 537 / 1,255 / 522, 564 / 835 / 539, 508 / 3,626 / 495.)
constexpr int CHECK_T = 256, CHECK_U = 4;
constexpr uint32_t DIRECT_CHAIN = 32768, DIRECT_PER_ROW = 4096;
// Above any sum of entries (40,960 slots of less than 2^32, or 2 M of up to DIRECT_ROW), and 2,000 workgroups may add it.
constexpr unsigned long long DIRECT_TOO_LONG = 1ull << 50;
__global__ __launch_bounds__(CHECK_T) void sample_check_kernel(SampleArgs a, uint64_t budget, uint32_t most_chain,
                                                               CallHost* __restrict__ host, unsigned long long number) {
  __shared__ unsigned long long s_sum[CHECK_T / 64];
  __shared__ uint32_t s_chain[CHECK_T / 64];
  call_stamp(a.call);
  const HopGeom& g = a.hop[a.h0];
  const uint64_t slots = a.N * g.width;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t v[CHECK_U], d[CHECK_U];
#pragma unroll
  for (int u = 0; u < CHECK_U; ++u) {
    const uint64_t slot = ((uint64_t)blockIdx.x * CHECK_U + u) * CHECK_T + threadIdx.x, si = slot / g.width;
    v[u] = slot < slots ? parent_of(a, g, si, (uint32_t)(slot - si * g.width)) : 0xFFFFFFFFu;
  }
#pragma unroll
  for (int u = 0; u < CHECK_U; ++u) d[u] = v[u] < a.V ? a.xadj[v[u] + 1] - a.xadj[v[u]] : 0u;
  unsigned long long sum = 0;
  uint32_t chain = 0;  // of the longest of the workgroups whose slots these are
#pragma unroll
  for (int u = 0; u < CHECK_U; ++u) {
    sum += d[u];
    uint32_t c = d[u] > DIRECT_LONG ? min(d[u], most_chain) + DIRECT_PER_ROW : 0u;
#pragma unroll
    for (int m = 1; m < DIRECT_T / 64; m *= 2) c += (uint32_t)__shfl_xor((int)c, m, 64);
    chain = max(chain, c);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    sum += shfl_xor_u64(sum, m);
    chain = max(chain, (uint32_t)__shfl_xor((int)chain, m, 64));
  }
  if (lane == 0) {
    s_sum[wave] = sum;
    s_chain[wave] = chain;
  }
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < CHECK_T / 64; ++w) {
    sum += s_sum[w];
    chain = max(chain, s_chain[w]);
  }
  if (chain > most_chain) sum += DIRECT_TOO_LONG;
  if (gridDim.x > 1) {
    atomicAdd(&a.words->entries, sum);
    __threadfence();
    if (atomicAdd(&a.words->arrived, 1ull) != gridDim.x - 1) return;
    sum = atomicExch(&a.words->entries, 0ull);
    a.words->arrived = 0;
  }
  a.words->refused = sum > budget;
  call_answer(host, number, 0, sum > budget);
}

// A wavefront a slot; the slots of a workgroup whose rows are too long for one are left to all eight together.  What bounds it is the chain
// of some six dependent loads of a slot and the longest row (1,676 seeds x 20 on the scale-22 graph, the longest row met of 100,000 entries:
// 382 us with a wavefront a slot throughout, 106 with four, 77 like this).
__global__ __launch_bounds__(DIRECT_T) void sample_direct_kernel(SampleArgs a, const float* __restrict__ wgt) {
  constexpr int NW = DIRECT_T / 64;
  __shared__ __align__(16) unsigned char smem[std::max(sizeof(DirectLds<DIRECT_T>), NW * sizeof(DirectLds<64>))];
  __shared__ uint32_t s_off[NW], s_d[NW];
  call_stamp(a.call);
  const bool refused = a.words && a.words->refused;
  const HopGeom& g = a.hop[a.h0];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto done = [&](uint64_t si, uint32_t s, uint32_t cnt) {
    a.sl[si * g.slen + g.loff + s] = cnt;
    if (!a.totals) return;
    if (g.h == 0) a.totals[si] = cnt;
    else atomicAdd(&a.totals[si], cnt);
  };
  const uint64_t first = a.first + (uint64_t)blockIdx.x * NW, slots = a.N * g.width;
  {
    const uint64_t slot = first + wave, si = slot / g.width;
    const uint32_t s = (uint32_t)(slot - si * g.width);
    uint32_t off = 0, d = 0;
    if (slot < slots) {
      const uint32_t v = parent_of(a, g, si, s);
      if (g.h == 0 && a.seeds && lane == 0) a.data[si * g.lps] = v;
      if (v < a.V) {
        off = a.xadj[v];
        d = a.xadj[v + 1] - off;
      }
      off = (uint32_t)__builtin_amdgcn_readfirstlane((int)off);
      d = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
      if (refused) return;  // the whole workgroup, here or below
      if (d <= DIRECT_LONG) {
        const uint32_t cnt = d ? direct_children<64>(a, g, wgt, si, s, off, d, lane, reinterpret_cast<DirectLds<64>*>(smem)[wave]) : 0u;
        if (lane == 0) done(si, s, cnt);
      }
    }
    if (lane == 0) {
      s_off[wave] = off;
      s_d[wave] = d > DIRECT_LONG ? d : 0u;
    }
  }
  if (refused) return;
  __syncthreads();
  for (uint32_t w = 0; w < NW; ++w) {
    const uint32_t d = s_d[w];
    if (d == 0) continue;
    const uint64_t slot = first + w, si = slot / g.width;
    const uint32_t s = (uint32_t)(slot - si * g.width);
    const uint32_t cnt = direct_children<DIRECT_T>(a, g, wgt, si, s, s_off[w], d, threadIdx.x, *reinterpret_cast<DirectLds<DIRECT_T>*>(smem));
    if (threadIdx.x == 0) done(si, s, cnt);
  }
}

// Distinct children (the rule of the reference's online sampler, roll_atomic / roll_once of
// src/online_sample_new.cu:72-105: up to 11 rounds, a candidate whose slot of the row is already selected is
// dropped, a parent may end with fewer than k children), made sequential so that the result does not depend on
// scheduling: draw i of slot s tries Philox(seed; seed index, s*k + i, h + 256 t, DOM_SAMPLE) for t = 0..10 and
// keeps the first candidate slot that no earlier draw of this parent kept; the children are written densely in
// the order of i.
// A group of G lanes (the power of two that holds k) shares a parent, one draw per lane.  All draws take their first
// candidate at once.  Let f be the first draw whose candidate equals that of an earlier one: the draws before it are
// final, and every draw from f on whose candidate one of those has kept goes on to its next try, again all at once,
// until no two candidates are equal.  The sequential rule comes out of this exactly, in as many rounds of dependent
// loads as candidates collide in a row, where one lane per parent took one per try: hop 1 of a 1024-seed batch with
// fanout 25 197 -> 17 us.
// What bounds a batch is the start vertex with the most rounds, and rounds are many where a row is hardly longer than k (25
// draws from 29 entries took 47, with 1.8 the mean of 1,024 start vertices).  Such a row, of up to 64 entries, is therefore held in
// LDS, entries and neighbours both, which also makes one dependent load of two.  A bit for every entry then says what is taken:
// a prefix over the draws of their candidates' bits finds f, the bits before f are final, and a draw that meets one of
// them goes on until it meets none, in the same round.  No more than k rounds, none of which leaves the CU: 1,024 seeds, 25 x 10 on the
// scale-20 graph 50 -> 36 us.  The first draw that needs its next try takes that one and the one behind it for all draws of the
// wavefront, which keep the candidates: a lane's random numbers take a wavefront as long as those of all, and ten tries are then drawn
// five times, not as often as draws need them (1,024 seeds x 25 27.3 -> 24.2 us, 25 x 10 34.7 -> 33.5, 300 x 32 x 7 on the scale-21 graph 31.9 -> 28.6,
// 5,000 x 15 x 10 x 5 154.5 -> 147; one at a time or five 1 to 2 % behind two.  Draw after draw instead of rounds: 34.4; tries taken
// by the idle groups of a hop with one parent: 25.2).
constexpr uint32_t DISTINCT_MAX_K = 64;  // largest fanout of this rule
constexpr uint32_t DISTINCT_ROUNDS = 11;
constexpr uint32_t DISTINCT_AHEAD = 2;  // tries that are taken together in a row in LDS
static_assert((DISTINCT_ROUNDS - 1) % DISTINCT_AHEAD == 0 && 6 * (DISTINCT_ROUNDS - 1) <= 64, "the candidates of all tries fit 64 bits");
// Entries a lane of a row that its group holds in LDS: 24 KB for 512 threads, four workgroups of which are all wavefronts that a CU takes.
constexpr uint32_t DISTINCT_ROW = 4;
__host__ __device__ inline uint32_t distinct_lanes(uint32_t k) {
  uint32_t g = 4;
  while (g < k) g *= 2;
  return g;
}

// T spreads the parents of one start vertex over several wavefronts, for batches of a few start vertices.
template <int T>
__global__ __launch_bounds__(T) void sample_distinct_kernel(SampleArgs a) {
  __shared__ __align__(16) uint32_t s_c[T];
  __shared__ AliasEntry s_row[T * DISTINCT_ROW];
  __shared__ uint32_t s_adj[T * DISTINCT_ROW];
  __shared__ uint32_t s_n[T / 64];
  if (a.h0 == 0) call_stamp(a.call);
  const uint64_t si = a.first + blockIdx.x / a.parts;
  const uint32_t part = blockIdx.x % a.parts, tid = threadIdx.x, lane = tid & 63;
  uint32_t mine = 0;
  for (uint32_t h = a.h0; h < a.h1; ++h) {
    const HopGeom& g = a.hop[h];
    const uint32_t k = g.k, G = distinct_lanes(k), i = tid & (G - 1), gbase = tid - i;
    const unsigned long long gm = G == 64 ? ~0ull : ((1ull << G) - 1ull);
    auto group_mask = [&](bool p) { return (__ballot(p) >> (lane & ~(G - 1))) & gm; };
    if (h == 0 && a.seeds && part == 0 && tid == 0) a.data[si * g.lps] = a.seeds[si];
    const uint32_t groups = T / G;
    for (uint64_t s0 = (uint64_t)part * groups; s0 < g.width; s0 += (uint64_t)a.parts * groups) {
      const uint64_t slot = s0 + tid / G;
      const uint32_t s = (uint32_t)slot;
      const bool in = slot < g.width;
      const uint32_t v = in ? parent_of(a, g, si, s) : 0xFFFFFFFFu;
      uint32_t o = 0, deg = 0;
      if (v < a.V) {
        const int8_t ok = a.valid[v];  // beside the bounds
        o = a.xadj[v];
        deg = a.xadj[v + 1] - o;
        if (!ok) deg = 0;
      }
      // Five draws and fewer collide so seldom that only a start vertex with several wavefronts, which wait for the slowest of
      // them, gains (3,000 seeds, 5 x 3 on the scale-18 graph 27 -> 25 us; one wavefront each, 5,000 seeds, 15 x 10 x 5 217 -> 223).
      const bool held = G >= (T > 64 ? 8u : 16u) && deg > k && deg <= min(64u, DISTINCT_ROW * G);
      const uint32_t rbase = DISTINCT_ROW * gbase;
      if (held) {
        AliasEntry x[DISTINCT_ROW];
        uint32_t y[DISTINCT_ROW];
#pragma unroll
        for (uint32_t m = 0; m < DISTINCT_ROW; ++m) {  // all on their way before the first is waited for
          const uint32_t j = min(m * G + i, deg - 1);
          x[m] = a.table[o + j];
          y[m] = a.adjncy[o + j];
        }
#pragma unroll
        for (uint32_t m = 0; m < DISTINCT_ROW; ++m) {
          const uint32_t j = m * G + i;
          if (j < deg) {
            s_row[rbase + j] = x[m];
            s_adj[rbase + j] = y[m];
          }
        }
      }
      uint32_t cand = 0, child = 0, t = 0;
      bool live = i < min(deg, k);  // a draw that keeps something, as far as is known
      const bool direct = deg > k && !held;
      uint32_t col = 0;
      float u = 0.0f;
      auto numbers = [&](uint32_t round) {
        const u32x4 r = philox(a.seed, (uint32_t)si, s * k + i, g.h + 256u * round, DOM_SAMPLE);
        col = __umulhi(r.x, deg);
        u = u24(r.y);
      };
      if (live && deg > k) numbers(0);
      AliasEntry e{0.0f, 0};
      if (live && !held) {  // on its way meanwhile
        if (direct) e = a.table[o + col];
        else child = a.adjncy[o + (cand = i)];  // all neighbours
      }
      if (__any(held)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        auto drawn = [&] {
          const AliasEntry x = s_row[rbase + col];
          return u < x.prob ? col : x.alias;
        };
        if (held && live) cand = drawn();
        uint64_t next = 0;  // candidates of the tries behind the first, 6 bits each, `filled` of them
        uint32_t filled = 0;
        auto fill = [&] {
          if (held && live) {
#pragma unroll
            for (uint32_t m = 0; m < DISTINCT_AHEAD; ++m) {
              numbers(filled + 1 + m);
              next |= (uint64_t)drawn() << (6 * (filled + m));
            }
          }
          filled += DISTINCT_AHEAD;
        };
        for (;;) {
          const uint64_t bit = held && live ? 1ull << cand : 0ull;
          uint64_t before = bit;  // candidates of this draw and the earlier ones of its group, then of the earlier ones
          auto from = [&](uint32_t dist, uint64_t x) { before |= i >= dist ? x : 0ull; };
          from(1, dpp0_u64<DPP_ROW_SHR1, 0xF>(before));
          from(2, dpp0_u64<DPP_ROW_SHR2, 0xF>(before));
          from(4, dpp0_u64<DPP_ROW_SHR4, 0xF>(before));
          from(8, dpp0_u64<DPP_ROW_SHR8, 0xF>(before));
          if (G >= 32) before |= dpp0_u64<DPP_ROW_BCAST15, 0xA>(before);
          if (G >= 64) before |= dpp0_u64<DPP_ROW_BCAST31, 0xC>(before);
          before = lane_before_u64(before);
          if (i == 0) before = 0;
          const unsigned long long bad = group_mask((before & bit) != 0);
          if (!__any(bad != 0)) break;
          const uint32_t f = bad ? (uint32_t)__ffsll((long long)bad) - 1 : 0u;
          const uint64_t final = bad ? shfl_u64(before, (int)((lane & ~(G - 1)) + f)) : 0ull;
          bool taken = i >= f && (bit & final);
          while (__any(taken)) {
            if (taken && ++t == DISTINCT_ROUNDS) live = taken = false;
            if (__any(taken && t > filled)) fill();
            if (taken) {
              cand = (uint32_t)(next >> (6 * (t - 1))) & 63u;
              taken = (final >> cand) & 1;
            }
          }
        }
        if (held && live) child = s_adj[rbase + cand];
      }
      if (__any(live && !held)) {
        // The entry of the next try is requested when this one's candidate is taken (1,024 seeds, 25 x 10 on the scale-20 graph 60 -> 58 us,
        // 806 with 4 edges a vertex 43 -> 38; several tries at once cost more in random numbers than they save: 65).
        auto take = [&] {
          cand = u < e.prob ? col : e.alias;
          child = a.adjncy[o + cand];
          if (t + 1 < DISTINCT_ROUNDS) {
            numbers(t + 1);
            e = a.table[o + col];
          }
        };
        if (live && direct) take();
        for (;;) {
          s_c[tid] = cand;
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          unsigned long long same = 0;  // earlier draws of the group with this draw's candidate
          for (uint32_t j = 0; j < k; j += 4) {
            const uint4 c = *reinterpret_cast<const uint4*>(s_c + gbase + j);
            const uint32_t m = (c.x == cand ? 1u : 0u) | (c.y == cand ? 2u : 0u) | (c.z == cand ? 4u : 0u) | (c.w == cand ? 8u : 0u);
            same |= (unsigned long long)m << j;
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the next round's candidates stay behind these reads
          __builtin_amdgcn_wave_barrier();
          const unsigned long long alive = group_mask(live);
          same &= alive & ((1ull << i) - 1ull);
          const unsigned long long bad = group_mask(live && direct && same != 0);
          if (!__any(bad != 0)) break;
          if (bad) {
            const uint32_t f = (uint32_t)__ffsll((long long)bad) - 1;
            if (live && i >= f && (same & ((1ull << f) - 1ull))) {  // a final draw holds the candidate
              if (++t == DISTINCT_ROUNDS) live = false;
              else take();
            }
          }
        }
      }
      const unsigned long long kept = group_mask(live);
      if (live) a.data[si * g.lps + g.off_next + slot * k + (uint32_t)__popcll(kept & ((1ull << i) - 1ull))] = child;
      if (in && i == 0) {
        a.sl[si * g.slen + g.loff + s] = (uint32_t)__popcll(kept);
        mine += (uint32_t)__popcll(kept);
      }
    }
    if (h + 1 < a.h1) __syncthreads();  // the next hop reads what this workgroup has just written
  }
  if (a.totals) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) mine += (uint32_t)__shfl_xor((int)mine, m, 64);
    if (lane == 0) s_n[tid >> 6] = mine;
    __syncthreads();
    if (tid == 0) {
      mine = a.h0 ? a.totals[si] : 0u;
#pragma unroll
      for (int w = 0; w < T / 64; ++w) mine += s_n[w];
      a.totals[si] = mine;
    }
  }
}

// Collects the distinct vertices of the filled slots of hop h whose table has not been built
// during this call: the first setter of the vertex's bit appends it, to the segments of the degree classes (sky_build_fused.h), to
// a plain list, or to both (a null pointer leaves one out).  One update per workgroup of 1024 lanes and counter: a word
// serves its atomics one after another.
// Of the lanes of a workgroup that want the same vertex one asks for its bit: each writes its number to the vertex's place in LDS, and who
// finds a lane with its own vertex there leaves the bit to that one.  (8,192 times one start vertex: a word serves an atomic in 5 ns,
// 44 us.)
constexpr int COLLECT_T = 1024;
constexpr uint32_t COLLECT_SEEN = 4096;
__global__ __launch_bounds__(COLLECT_T) void frontier_collect_kernel(const uint32_t* __restrict__ data,
                                                                     const uint32_t* __restrict__ sl, uint64_t total,
                                                                     uint32_t V, HopGeom g, uint32_t* bitmap, uint32_t bit_mask,
                                                                     const uint32_t* __restrict__ xadj,
                                                                     int8_t* __restrict__ valid, FrontierLists f,
                                                                     uint32_t* __restrict__ counts,
                                                                     uint32_t* __restrict__ list,
                                                                     uint32_t* __restrict__ count) {
  __shared__ uint32_t s_cnt[CLS_COUNT], s_base[CLS_COUNT];
  __shared__ uint32_t s_n[COLLECT_T / 64 + 1];
  __shared__ uint32_t s_v[COLLECT_T];
  __shared__ uint16_t s_owner[COLLECT_SEEN];
  const uint64_t tid = (uint64_t)blockIdx.x * COLLECT_T + threadIdx.x;
  bool fresh = false, live = false;
  uint32_t v = 0;
  if (tid < total) {
    uint64_t si, s;
    if (total <= 0xFFFFFFFFull) {
      const uint32_t si32 = (uint32_t)tid / (uint32_t)g.width;
      si = si32;
      s = (uint32_t)tid - si32 * (uint32_t)g.width;
    } else {
      si = tid / g.width;
      s = tid % g.width;
    }
    if (slot_filled(g, sl, si, s)) {
      v = data[si * g.lps + g.off + s];
      live = v < V;
    }
  }
  // The draws of a hop land on a few well-connected vertices again and again.  A bit that reads as set needs no
  // atomic: bits are never cleared during a call, and one that another XCD has just set and that still reads as clear
  // is decided by the atomic.
  const uint32_t b = frontier_bit(v, bit_mask), bit = 1u << (b & 31);
  const bool want = live && !(bitmap[b >> 5] & bit);
  const uint32_t seen = b & (COLLECT_SEEN - 1u);
  s_v[threadIdx.x] = v;
  if (want) s_owner[seen] = (uint16_t)threadIdx.x;
  __syncthreads();
  if (want) {
    const uint32_t other = s_owner[seen];
    if (other == threadIdx.x || s_v[other] != v) fresh = !(atomicOr(&bitmap[b >> 5], bit) & bit);
  }
  if (counts) append_rows(fresh, v, xadj, valid, f, counts, s_cnt, s_base);
  if (list) append_list(fresh, v, list, count, s_n);
}

// Start of an online call: start vertices in place, the bitmap of built rows and the counters cleared.  A call that runs
// through all hops writes every length and total; one that is handed out hop by hop may end before, so those are cleared
// for it (`sl`, nsl words, and `totals`, N; null: left alone).
__global__ __launch_bounds__(256) void sample_init_kernel(const uint32_t* __restrict__ seeds, uint32_t N, uint64_t lps,
                                                          uint32_t* __restrict__ data, uint32_t* __restrict__ bitmap,
                                                          uint32_t words, uint32_t* __restrict__ counts, uint32_t ncounts,
                                                          uint32_t* __restrict__ sl, uint64_t nsl, uint32_t* __restrict__ totals,
                                                          CallDevice* __restrict__ call) {
  call_stamp(call);
  const uint64_t i0 = (uint64_t)blockIdx.x * 256u + threadIdx.x, step = (uint64_t)gridDim.x * 256u;
  for (uint64_t i = i0; i < ncounts; i += step) counts[i] = 0;
  for (uint64_t i = i0; i < words; i += step) bitmap[i] = 0;
  for (uint64_t i = i0; i < N; i += step) data[i * lps] = seeds[i];
  if (sl)
    for (uint64_t i = i0; i < nsl; i += step) sl[i] = 0;
  if (totals)
    for (uint64_t i = i0; i < N; i += step) totals[i] = 0;
}

// One call of the k-hop sampler, taken apart hop by hop: begin (start vertices in place), then for
// every hop frontier (online: the distinct parents whose rows are not built yet), build (online: their rows) and
// draw, then end (count, time).  sample_khop runs the steps in turn; sky_sample_session_* hands them to callers that
// supply the weights of a frontier's rows themselves.
struct SampleSession {
  sky_graph* g = nullptr;
  bool online = false, dev_sized = false, distinct = false;
  std::vector<char> direct;  // by hop: drawn from the weights, without tables
  const uint32_t* seeds = nullptr;
  uint32_t N = 0, hops = 0;
  uint64_t seed = 0;
  uint32_t *data = nullptr, *sample_lengths = nullptr;
  std::vector<uint32_t> fanout;
  std::vector<uint64_t> width, off, loff;
  uint64_t lps = 0, slen = 0;
  CallDevice* call = nullptr;
  CallWords own_words;  // of a session whose steps are calls of their own
  uint32_t *bitmap = nullptr, *list = nullptr, *d_count = nullptr;
  // Counters of the frontiers, a hop's own each, cleared when the call begins: the length of its list, then FRONTIER_WORDS
  // with the rows of every degree class (dev_sized).  Behind them a word for every row that can be made tile by tile, for the hop
  // of this call that has built it: kept with the graph's rows instead, another call's build between two hops of a session made the
  // session build the row again, from weights that its caller had not supplied.
  uint32_t *list_counts = nullptr, *front_counts = nullptr, *built = nullptr;
  FrontierLists front;
  std::vector<char> made;  // by hop: its rows have been built (a session's caller may have a hop built and drawn once more)
  // The plan of the graph when the call began.  Another call between the steps of a session may make the graph a new one, when
  // a knob that decides how long rows are built has changed.
  std::shared_ptr<BuildPlan> plan;
  std::vector<uint64_t> budget;  // by hop without tables: entries beyond which it is refused (0: never)
  bool stamped = false;          // the call's first kernel is on its way
  std::function<void()> init;    // enqueues sample_init_kernel, for an online call that is not direct throughout
  bool want_list = false;        // the caller is to see the frontier as a list of vertices
  uint32_t* totals = nullptr;    // children of each start vertex, when the kernels add them up
  uint32_t frontier_upper = 0;   // most rows the last frontier can hold
  uint32_t frontier_count = 0;   // its size, when the host has read it (dev_sized false)
  // A session keeps its buffers while other calls, other sessions among them, use the same graph: the first to come holds
  // those of the graph, the others have their own.
  bool holds_pool = false;
  sky_graph::PoolBuf own[sky_graph::POOL_SLOTS];
  explicit SampleSession(sky_graph* g_) : g(g_) {
    holds_pool = !g->sampler_busy;
    g->sampler_busy = true;
  }
  SampleSession(const SampleSession&) = delete;
  ~SampleSession() {
    if (holds_pool) g->sampler_busy = false;
    call_release(&own_words);
    for (auto& b : own)
      if (b.p) (void)hipFree(b.p);
  }
  sky_graph::PoolBuf* buffer(int slot) { return holds_pool ? &g->pool[slot] : &own[slot]; }
  CallWords* words() { return want_list ? &own_words : &g->call; }
  int get(int slot, size_t bytes, void** out) {
    SKY_TRY(buf_grow(buffer(slot), bytes));
    *out = buffer(slot)->p;
    return SKY_OK;
  }

  HopGeom geom(uint32_t h) const {
    HopGeom hg;
    hg.h = h;
    hg.k = fanout[h + 1];
    hg.fan_h = fanout[h];
    hg.width = width[h];
    hg.off = off[h];
    hg.off_next = off[h + 1];
    hg.loff = loff[h];
    hg.loff_prev = h ? loff[h - 1] : 0;
    hg.lps = lps;
    hg.slen = slen;
    return hg;
  }

  int begin(bool online_, const uint32_t* seeds_, uint32_t N_, const uint32_t* fanout_, uint32_t hops_, uint64_t seed_,
            uint32_t* data_, uint32_t* sl_) {
    hipStream_t st = g->stream;
    online = online_;
    seeds = seeds_;
    N = N_;
    hops = hops_;
    seed = seed_;
    data = data_;
    sample_lengths = sl_;
    distinct = option(g, OPT_SAMPLE_DISTINCT) != 0;
    fanout.assign(fanout_, fanout_ + hops);
    if (distinct) {
      if (hops > 256) return fail(SKY_ERR_LIMIT, "sample: distinct children need at most 256 hops");
      for (uint32_t h = 1; h < hops; ++h)
        if (fanout[h] > DISTINCT_MAX_K) return fail(SKY_ERR_LIMIT, "sample: distinct children need fanouts of at most 64");
    }
    if (g->has_tables) online = false;  // every row is already there: nothing to build on the way
    // Without the option the host reads the size of every frontier and sizes the launches of its build exactly;
    // with it (the default) nothing inside the call waits for the device.
    dev_sized = online && fused_possible(g) && option(g, OPT_ONLINE_DEVICE_SIZED) != 0;
    width.assign(hops, 0);
    off.assign(hops, 0);
    loff.assign(hops, 0);
    made.assign(hops, 0);
    uint64_t wd = 1;
    for (uint32_t h = 0; h < hops; ++h) {
      wd *= fanout[h];
      width[h] = wd;
      off[h] = lps;
      lps += wd;
      if (h + 1 < hops) {
        loff[h] = slen;
        slen += wd;
      }
    }
    if ((uint64_t)N * lps > (1ull << 40)) return fail(SKY_ERR_LIMIT, "sample: output too large");
    const uint32_t bits = frontier_mask(g->V) / 32 + 1;  // words of the bitmap
    uint32_t counters = 0;
    SKY_TRY(call_begin(g, words(), &call));
    if (online) {
      SKY_TRY(ensure_table_storage(g));
      if (dev_sized) {
        SKY_TRY(ensure_plan(g, &call));
        plan = g->plan;
        // room for the largest hop's rows from the start: growing it at a later hop would free and allocate with that
        // hop's predecessor running (first call on a graph, 40,000 seeds: 1.80 -> 1.20 ms)
        uint64_t most = 0;
        for (uint32_t h = 0; h + 1 < hops; ++h) most = std::max(most, (uint64_t)N * width[h]);
        SKY_TRY(frontier_lists(g, *plan, (uint32_t)std::min<uint64_t>(most, g->V), buffer(sky_graph::POOL_SEGMENTS), &front));
      } else {
        SKY_TRY(prepare_build_scratch(g, g->V));
      }
      counters = (hops - 1) * (1 + (dev_sized ? FRONTIER_WORDS : 0u)) + (dev_sized ? plan->n_trows : 0u);
      SKY_TRY(get(sky_graph::POOL_FRONT, (size_t)counters * 4, (void**)&list_counts));
      d_count = list_counts;
      if (dev_sized) {
        front_counts = list_counts + (hops - 1);
        built = front_counts + (hops - 1) * FRONTIER_WORDS;
      }
      SKY_TRY(get(sky_graph::POOL_BITMAP, (size_t)bits * 4, (void**)&bitmap));
      if (want_list || !dev_sized) SKY_TRY(get(sky_graph::POOL_LIST, (size_t)g->V * 4, (void**)&list));
    }
    if (N && one_workgroup()) SKY_TRY(get(sky_graph::POOL_TOTALS, (size_t)N * 4, (void**)&totals));
    const uint64_t lengths = want_list ? (uint64_t)N * slen : 0;  // to be cleared
    const uint64_t items = std::max<uint64_t>(std::max(std::max(N, bits), 1u), lengths);  // an empty graph has counters too
    init = [=] {
      hipLaunchKernelGGL(sample_init_kernel, dim3((uint32_t)std::min<uint64_t>((items + 255) / 256, 2048)), dim3(256), 0, st, seeds,
                         N, lps, data, bitmap, bits, list_counts, counters, lengths ? sample_lengths : nullptr, lengths,
                         want_list ? totals : nullptr, stamped ? nullptr : call);
      stamped = true;
    };
    if (dev_sized && !want_list && !distinct && N) choose_direct();
    if (online && !all_direct()) init();
    return SKY_OK;
  }
  bool is_direct(uint32_t h) const { return !direct.empty() && direct[h]; }
  bool all_direct() const { return !direct.empty() && std::find(direct.begin(), direct.end(), 0) == direct.end(); }

  // All hops in turn.
  int run() {
    if (!online && totals) return draw(0, hops - 1);
    for (uint32_t h = 0; h + 1 < hops; ++h) {
      SKY_TRY(frontier(h));
      SKY_TRY(build(h, nullptr));
      SKY_TRY(draw(h, h + 1));
      if (!is_direct(h) || !budget[h]) continue;
      unsigned long long refused = 0;
      SKY_TRY(call_answered(g, words(), &refused, 1));
      if (!refused) continue;
      if (all_direct()) init();
      direct.clear();  // the hop once more, with tables, and those behind it
      --h;
    }
    return SKY_OK;
  }

  // Online: the distinct parents of hop h whose rows this call has not built yet, into `list`; their number stays in
  // the hop's device word d_count (and is read by the host only when the build needs it there).
  int frontier(uint32_t h) {
    frontier_upper = frontier_count = 0;
    if (!online || !N || is_direct(h)) return SKY_OK;
    hipStream_t st = g->stream;
    const HopGeom hg = geom(h);
    const uint64_t slots = (uint64_t)N * hg.width;
    frontier_upper = (uint32_t)std::min<uint64_t>(slots, g->V);
    d_count = list_counts + h;
    if (dev_sized) SKY_TRY(frontier_lists(g, *plan, frontier_upper, buffer(sky_graph::POOL_SEGMENTS), &front));
    hipLaunchKernelGGL(frontier_collect_kernel, dim3((uint32_t)((slots + COLLECT_T - 1) / COLLECT_T)), dim3(COLLECT_T), 0, st,
                       data, sample_lengths, slots, g->V, hg, bitmap, frontier_mask(g->V), g->xadj, g->valid, front,
                       dev_sized ? front_counts + h * FRONTIER_WORDS : nullptr, list, d_count);
    if (!dev_sized) {
      SKY_HIP(hipMemcpyAsync(&frontier_count, d_count, 4, hipMemcpyDeviceToHost, st));
      SKY_HIP(hipStreamSynchronize(st));
    }
    return SKY_OK;
  }

  // Online: the rows of the last frontier, from `weights` (null: the graph's own).  The length of the list stays
  // on the device where it can: the kernels of the build find it there, and the host goes on to enqueue the hop
  // without waiting (the reference's sampler never leaves the device either, src/online_sample_new.cu:191-270).
  int build(uint32_t h, const float* weights) {
    if (!online || !N || !frontier_upper) return SKY_OK;
    float* const own = g->adjwgt;
    if (weights) g->adjwgt = const_cast<float*>(weights);  // the build only reads it
    const int rc = dev_sized ? build_frontier(g, *plan, front, front_counts + h * FRONTIER_WORDS, made[h], bitmap, built, h)
                             : build_rows(g, list, frontier_count, nullptr);
    made[h] = 1;
    g->adjwgt = own;
    return rc;
  }

  // Passes a wavefront (distinct children: a workgroup of 256) would need for one start vertex at hop h.
  uint64_t passes(uint32_t h) const {
    const uint64_t per_pass = distinct ? (fanout[h + 1] <= 16 ? 16u : fanout[h + 1] <= 32 ? 8u : 4u) : (uint64_t)SAMPLE_T * SAMPLE_U;
    const uint64_t items = distinct ? width[h] : width[h] * fanout[h + 1];
    return (items + per_pass - 1) / per_pass;
  }
  // A workgroup takes its start vertex through every hop when the widest of them keeps it busy for a few passes only, or
  // when there are start vertices enough to fill the GPU anyway (8,192 wavefronts); otherwise several workgroups
  // share a start vertex, hop by hop.
  bool one_workgroup() const { return passes(hops - 2) <= 8 || N >= 8192; }

  int draw(uint32_t h0, uint32_t h1) {
    if (!N) return SKY_OK;
    if (is_direct(h0)) return draw_direct(h0);
    hipStream_t st = g->stream;
    SampleArgs a = {};
    a.xadj = g->xadj;
    a.adjncy = g->adjncy;
    a.table = g->table;
    a.valid = g->valid;
    a.seeds = online ? nullptr : seeds;
    a.call = online ? nullptr : call;
    a.data = data;
    a.sl = sample_lengths;
    a.totals = totals;
    a.V = g->V;
    a.h0 = h0;
    a.h1 = h1;
    a.N = N;
    a.seed = seed;
    for (uint32_t h = h0; h < h1; ++h) a.hop[h] = geom(h);
    const uint64_t parts = totals ? 1 : std::min<uint64_t>(passes(h0), 65536);
    a.parts = (uint32_t)parts;
    a.lanes = 64;
    if (totals && !distinct) {
      const uint64_t draws = width[h1 - 1] * fanout[h1];
      while (a.lanes > 1 && draws <= a.lanes / 2) a.lanes /= 2;
    }
    // Distinct children: lanes for every parent of the widest hop at once, as long as the GPU holds all wavefronts (2,500 seeds,
    // 10 x 10 on the scale-18 graph 46 -> 42 us; 5,000, 25 x 10 on the scale-20 graph 79 -> 78).
    uint32_t T = 64;
    if (distinct && parts > 1) {
      T = 256;
    } else if (distinct) {
      uint64_t lanes = 0;
      for (uint32_t h = h0; h < h1; ++h) lanes = std::max(lanes, width[h] * distinct_lanes(fanout[h + 1]));
      while (T < 1024 && T < lanes && (uint64_t)N * (2 * T / 64) <= 8192) T *= 2;
    }
    const uint32_t per_block = distinct ? 1 : SAMPLE_T / a.lanes;
    const uint64_t most = 0xFFFFFFFFull / T / parts * per_block;  // start vertices of one launch (below 2^32 threads)
    for (a.first = 0; a.first < N; a.first += most) {
      const dim3 grid((uint32_t)((std::min<uint64_t>(most, N - a.first) + per_block - 1) / per_block * parts));
      auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(T), 0, st, a); };
      if (!distinct) go(sample_draw_kernel);
      else if (T == 64) go(sample_distinct_kernel<64>);
      else if (T == 128) go(sample_distinct_kernel<128>);
      else if (T == 256) go(sample_distinct_kernel<256>);
      else if (T == 512) go(sample_distinct_kernel<512>);
      else go(sample_distinct_kernel<1024>);
      a.call = nullptr;
    }
    return SKY_OK;
  }

  // Which hops do without tables, unless their rows turn out to be long (sample_check_kernel).  The six launches that collect, build and
  // draw take 50 us even of a few rows; start vertices are mostly any vertices, whose rows are short, and a draw from the weights of one
  // costs little more than the draw from its table.  Up to DIRECT_SEEDS of them (40,000 x 20 on the scale-16 graph 81 / 79, 60,000 86 / 98);
  // of a call of several hops only up to DIRECT_FEW, and no more than there are vertices: rows built for the first hop are met again at
  // the second.  (Built / direct, us: 10,000 seeds x 20 on the scale-14 graph 66 / 48, 39,000 on the scale-22 graph 125 / 92; 700 x 5 x 3, scale 13,
  // 103 / 91; 3,000 x 5 x 3, scale 16, 134 / 115; 401 x 10 x 10, scale 22, 299 / 249; 15,900 x 5 x 3 on 4,096 vertices 111 / 145, 36,000 x
  // 5 x 3 on the scale-20 graph 402 / 450.)  Later hops lead to long rows, again and again: the call does without tables altogether where they
  // come to few entries and none is very long (70 x 5 x 3, scale 18, 97 / 68; 200 x 25 x 10, scale 15, 106 / 75; 400 x 10 x 10 with 3.4 M
  // entries, scale 14, 107 / 122; 100 x 5 x 3 on the scale-20 graph, whose longest row has 69,000 entries, 107 / 145).
  static constexpr uint32_t DIRECT_SEEDS = 40960, DIRECT_FEW = 8192, DIRECT_ROW = 52000;
  static constexpr double DIRECT_ENTRIES = 2e6, DIRECT_SPARE = 1e6;
  void choose_direct() {
    const long long mode = option(g, OPT_ONLINE_DIRECT);
    if (mode == 0) return;
    budget.assign(hops - 1, 0);
    if (mode > 0) return direct.assign(hops - 1, 1);
    if (N > DIRECT_SEEDS || (hops > 2 && N > std::min(DIRECT_FEW, g->V))) return;
    double mean = 0;  // entries of the row that an edge leads to
    for (int c = CLS_G2; c < CLS_COUNT; ++c)
      if (g->bin_counts[c]) mean += (double)g->bin_edges[c] * g->bin_edges[c] / g->bin_counts[c] / std::max(1u, g->E);
    bool all = g->max_degree <= DIRECT_ROW;
    auto limit = [&](uint32_t h, double entries) {  // rows that are all short and few are not looked at
      const uint64_t most = (uint64_t)(DIRECT_SPARE + entries);
      if (g->max_degree > DIRECT_LONG || (double)N * width[h] * g->max_degree > (double)most) budget[h] = most;
    };
    limit(0, (double)N * g->E / std::max(1u, g->V));
    for (uint32_t h = 1; h + 1 < hops; ++h) {
      const double entries = (double)N * width[h] * std::max(1.0, mean);
      all = all && entries <= DIRECT_ENTRIES;
      limit(h, entries);
    }
    direct.assign(hops - 1, all);
    direct[0] = 1;
  }
  int draw_direct(uint32_t h) {
    SampleArgs a = {};
    a.xadj = g->xadj;
    a.adjncy = g->adjncy;
    a.seeds = h == 0 ? seeds : nullptr;
    a.call = stamped ? nullptr : call;
    a.words = budget[h] ? words()->dev : nullptr;
    stamped = true;
    a.data = data;
    a.sl = sample_lengths;
    a.totals = totals;
    a.V = g->V;
    a.h0 = h;
    a.h1 = h + 1;
    a.seed = seed;
    a.hop[h] = geom(h);
    a.N = N;
    constexpr uint64_t PER = DIRECT_T / 64;
    const uint64_t slots = (uint64_t)N * width[h], most = PER << 22;  // slots of one launch: below 2^32 threads
    if (budget[h]) {  // of few enough slots, by choose_direct, for one launch
      const uint32_t chain = DIRECT_CHAIN + std::min(plan->n_tiles, 65536u);  // a build passes over the plan's tiles, 1.1 ns each too
      hipLaunchKernelGGL(sample_check_kernel, dim3((uint32_t)((slots + CHECK_T * CHECK_U - 1) / (CHECK_T * CHECK_U))), dim3(CHECK_T), 0,
                         g->stream, a, budget[h], chain, words()->host, call_ask(words()));
      a.call = nullptr;
    }
    for (a.first = 0; a.first < slots; a.first += most) {
      const dim3 grid((uint32_t)((std::min<uint64_t>(most, slots - a.first) + PER - 1) / PER));
      hipLaunchKernelGGL(sample_direct_kernel, grid, dim3(DIRECT_T), 0, g->stream, a, g->adjwgt);
      a.call = nullptr;
    }
    return SKY_OK;
  }

  int end(uint64_t* sampled, double* seconds) {
    if (totals) return call_end(g, words(), sampled, seconds, totals, N);
    return call_end(g, words(), sampled, seconds, sample_lengths, (uint64_t)N * slen);
  }
};

int sample_khop(sky_graph* g, bool online, const uint32_t* seeds, uint32_t N, const uint32_t* fanout, uint32_t hops,
                uint64_t seed, uint32_t* data, uint32_t* sample_lengths, uint64_t* sampled, double* seconds) {
  SampleSession s(g);
  SKY_TRY(s.begin(online, seeds, N, fanout, hops, seed, data, sample_lengths));
  SKY_TRY(s.run());
  return s.end(sampled, seconds);
}

// The same steps behind the C interface (sky_sample_session_*).
int sample_session_begin(sky_graph* g, const uint32_t* seeds, uint32_t N, const uint32_t* fanout, uint32_t hops,
                         uint64_t seed, uint32_t* data, uint32_t* sample_lengths, SampleSession** out) {
  SampleSession* s = new SampleSession(g);
  s->want_list = true;
  const int rc = s->begin(true, seeds, N, fanout, hops, seed, data, sample_lengths);
  if (rc != SKY_OK) {
    delete s;
    return rc;
  }
  *out = s;
  return SKY_OK;
}
int sample_session_frontier(SampleSession* s, uint32_t hop, const uint32_t** list, const uint32_t** count,
                            uint32_t* upper) {
  if (hop + 1 >= s->hops) return fail(SKY_ERR_ARG, "sky_sample_session_frontier: no such hop");
  SKY_TRY(s->frontier(hop));
  if (list) *list = s->list;
  if (count) *count = s->d_count;
  if (upper) *upper = s->frontier_upper;
  return SKY_OK;
}
int sample_session_hop(SampleSession* s, uint32_t hop, const float* weights) {
  if (hop + 1 >= s->hops) return fail(SKY_ERR_ARG, "sky_sample_session_hop: no such hop");
  SKY_TRY(s->build(hop, weights));
  return s->draw(hop, hop + 1);
}
int sample_session_end(SampleSession* s, uint64_t* sampled, double* seconds) {
  const int rc = s->end(sampled, seconds);
  delete s;
  return rc;
}
bool sample_session_online(const SampleSession* s) { return s->online; }

}  // namespace sky
