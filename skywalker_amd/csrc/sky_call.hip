// End of a call: results and completion through pinned host words (sky_call.h).
#include <chrono>
#include <cstddef>
#include <mutex>
#include <vector>

#include "sky_graph.h"

namespace sky {

// One workgroup: adds up `counts` if there are any, reports.
__global__ __launch_bounds__(1024) void call_end_kernel(CallDevice* call, CallHost* host, unsigned long long seq,
                                                        const uint32_t* __restrict__ counts, uint32_t n, uint32_t parts) {
  __shared__ unsigned long long s_w[16];
  const unsigned long long start = call->start;  // on its way meanwhile
  unsigned long long t = 0, x = 0;
  if (threadIdx.x < parts) {
    unsigned long long* const part = &call->part[threadIdx.x * CALL_PART_WORDS];
    x = *part;
    if (x) *part = 0;
  }
  if (n) {
    for (uint32_t i = threadIdx.x; i < n; i += 4 * blockDim.x) {
      uint32_t c[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) c[k] = i + k * blockDim.x < n ? counts[i + k * blockDim.x] : 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) t += c[k];
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) t += shfl_xor_u64(t, m);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = t;
    __syncthreads();
    t = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; ++w) t += s_w[w];
  }
  if (threadIdx.x >= 64) return;
  if (parts > 1) x = shfl_u64(group_scan_u64<64>(x), 63);
  // The host may go on before the device words are zero again; who uses them next is a kernel behind this one on the device's null
  // stream, whichever graph it belongs to.
  if (threadIdx.x == 0) {
    call_report(host, seq, start, t + x);
    call->start = 0;
  }
}
static_assert(CALL_PARTS == 64, "by the first wavefront");

// The end of a call over several streams, which samples no edges: the last kernel of each.
struct SideEnd {
  CallDevice* call;
  CallHost* host;
  unsigned long long seq;
  __device__ uint32_t arrive() const { return __hip_atomic_fetch_add(&call->joined, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u; }
  __device__ unsigned long long clear() const {
    const unsigned long long start = __hip_atomic_load(&call->start, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&call->start, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&call->joined, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return start;
  }
  __device__ void report(unsigned long long start) const {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    call_report(host, seq, start, 0);
  }
};
__global__ void call_end_sides_kernel(CallDevice* call, CallHost* host, unsigned long long seq, uint32_t of) { side_arrive(SideEnd{call, host, seq}, of); }

__global__ __launch_bounds__(256) void sum_counts_kernel(const uint32_t* __restrict__ x, uint64_t n, CallDevice* call) {
  __shared__ unsigned long long s_w[4];
  unsigned long long t = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) t += x[i];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) t += shfl_xor_u64(t, m);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) call_sampled(call, blockIdx.x, CALL_PARTS, s_w[0] + s_w[1] + s_w[2] + s_w[3]);
}

// The call words of all graphs and sessions: chunks of 64, per device, handed out one to an owner for its lifetime.  A chunk none of
// whose words is in use goes back to the runtime when another one has free words.
namespace {
constexpr int CHUNK = 64;
struct Chunk {
  int device = 0, used = 0, khz = 0;
  CallDevice* dev = nullptr;
  CallHost* host = nullptr;
  bool taken[CHUNK] = {false};
};
std::mutex g_mutex;
std::vector<Chunk*> g_chunks;

void free_chunk(Chunk* c) {
  if (c->dev) (void)hipFree(c->dev);
  if (c->host) (void)hipHostFree(c->host);
  delete c;
}
int take_words(int device, CallWords* w) {
  std::lock_guard<std::mutex> lock(g_mutex);
  Chunk* use = nullptr;
  for (Chunk* c : g_chunks)
    if (c->device == device && c->used < CHUNK) use = c;
  if (!use) {
    Chunk* c = new Chunk();
    c->device = device;
    auto body = [&]() -> int {
      SKY_HIP(hipDeviceGetAttribute(&c->khz, hipDeviceAttributeWallClockRate, device));
      if (c->khz <= 0) return fail(SKY_ERR_HIP, "the device reports no wall clock rate");
      SKY_HIP(hipMalloc((void**)&c->dev, CHUNK * sizeof(CallDevice)));
      SKY_HIP(hipMemset(c->dev, 0, CHUNK * sizeof(CallDevice)));
      SKY_HIP(hipHostMalloc((void**)&c->host, CHUNK * sizeof(CallHost), hipHostMallocCoherent | hipHostMallocPortable));
      return SKY_OK;
    };
    const int rc = body();
    if (rc != SKY_OK) {
      free_chunk(c);
      return rc;
    }
    for (int k = 0; k < CHUNK; ++k) c->host[k] = CallHost{};
    g_chunks.push_back(c);
    use = c;
  }
  int k = 0;
  while (use->taken[k]) ++k;
  use->taken[k] = true;
  ++use->used;
  w->dev = use->dev + k;
  w->host = use->host + k;
  w->khz = use->khz;
  w->seq = use->host[k].sampled >> CALL_VALUE_BITS;  // not the next call's
  w->asked = use->host[k].answer[0] >> CALL_VALUE_BITS;
  w->forks = use->host[k].begun;
  return SKY_OK;
}
}  // namespace

void call_release(CallWords* w) {
  if (!w->host) return;
  std::lock_guard<std::mutex> lock(g_mutex);
  for (size_t i = 0; i < g_chunks.size(); ++i) {
    Chunk* c = g_chunks[i];
    if (w->host < c->host || w->host >= c->host + CHUNK) continue;
    const size_t k = (size_t)(w->host - c->host);
    if (w->dirty) (void)hipMemset(c->dev + k, 0, sizeof(CallDevice));
    c->taken[k] = false;
    --c->used;
    bool other = false;
    for (Chunk* o : g_chunks) other = other || (o != c && o->device == c->device && o->used < CHUNK);
    if (c->used == 0 && other) {
      g_chunks.erase(g_chunks.begin() + (long)i);
      free_chunk(c);
    }
    break;
  }
  *w = CallWords{};
}

int call_begin(sky_graph* g, CallWords* w, CallDevice** call) {
  if (!w->host) SKY_TRY(take_words(g->device, w));
  if (w->dirty) SKY_HIP(hipMemsetAsync(w->dev, 0, sizeof(CallDevice), g->stream));
  w->dirty = true;  // until it has ended well
  w->parts = 0;
  ++g->calls;
  *call = w->dev;
  return SKY_OK;
}
int call_begin(sky_graph* g, CallDevice** call) { return call_begin(g, &g->call, call); }

void call_cancel(sky_graph* g) { g->call.dirty = false; }

// ---------------------------------------------------------------- beside the graph's stream
namespace {
struct SideRuntime {
  using Stream = hipStream_t;
  int device;
  bool can() const {
    int yes = 0;
    return worked(hipDeviceGetAttribute(&yes, hipDeviceAttributeCanUseStreamWaitValue, device)) && yes;
  }
  bool create(Stream* s) const { return worked(hipStreamCreateWithFlags(s, hipStreamNonBlocking)); }
  void destroy(Stream s) const { (void)hipStreamDestroy(s); }

 private:
  static bool worked(hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();  // not an error of the call, which does without
    return e == hipSuccess;
  }
};
SidePool<SideRuntime> g_side[SIDE_DEVICES];
}  // namespace

// The last kernel of each of the n side streams of a fork.  (A word for each, and a wait for each on the graph's stream: 4.5 us apiece.)
__global__ void beside_done_kernel(CallDevice* dev, CallHost* host, uint32_t n, uint32_t number) {
  if (__hip_atomic_fetch_add(&dev->joined, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u != n) return;
  __hip_atomic_store(&dev->joined, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&host->done, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int beside_begin(sky_graph* g, Beside* b, ForkMark* mark, int streams) {
  *b = Beside{};
  *mark = ForkMark{nullptr, 0};
  int current = -1;
  SKY_HIP(hipGetDevice(&current));
  const SideAsk ask{option(g, OPT_BUILD_STREAMS), g->device, current, g->calls, streams};
  if (!ask.allowed()) return SKY_OK;
  if (!g->call.host) SKY_TRY(take_words(g->device, &g->call));
  std::lock_guard<std::mutex> lock(g_mutex);
  SideRuntime runtime{g->device};
  if (!g_side[g->device].take(runtime, &g->sides, ask)) return SKY_OK;
  for (int k = 0; k < streams; ++k) b->stream[k] = g_side[g->device].stream[k];
  b->main = g->stream;
  b->dev = g->call.dev;
  b->host = g->call.host;
  b->number = ++g->call.forks;
  *mark = ForkMark{&b->host->begun, b->number};
  return SKY_OK;
}
int beside_fork(Beside* b, int k) {
  if (b->used[k]) return SKY_OK;
  SKY_HIP(hipStreamWaitValue32(b->stream[k], &b->host->begun, b->number, hipStreamWaitValueEq, 0xFFFFFFFFu));
  b->used[k] = true;
  return SKY_OK;
}
int beside_join(Beside* b) {
  uint32_t n = 0;
  for (bool u : b->used) n += u;
  if (!n) return SKY_OK;
  for (int k = 0; k < SIDE_STREAMS; ++k)
    if (b->used[k]) {
      if (b->last) hipLaunchKernelGGL(call_end_sides_kernel, dim3(1), dim3(1), 0, b->stream[k], b->dev, b->host, b->last->seq + 1, n + 1);
      else hipLaunchKernelGGL(beside_done_kernel, dim3(1), dim3(1), 0, b->stream[k], b->dev, b->host, n, b->number);
    }
  SKY_HIP(hipGetLastError());
  if (!b->last) SKY_HIP(hipStreamWaitValue32(b->main, &b->host->done, b->number, hipStreamWaitValueEq, 0xFFFFFFFFu));
  for (int k = 0; k < SIDE_STREAMS; ++k)
    if (b->last && b->used[k]) b->last->side[b->last->sides++] = b->stream[k];
  for (bool& u : b->used) u = false;
  return SKY_OK;
}
void beside_drop(Beside* b) {
  bool any = false;
  for (int k = 0; k < SIDE_STREAMS; ++k)
    if (b->used[k]) {
      any = true;
      (void)hipStreamSynchronize(b->stream[k]);
    }
  if (any) (void)hipMemset(&b->dev->joined, 0, sizeof(b->dev->joined));
  for (bool& u : b->used) u = false;
}

void beside_release(sky_graph* g) {
  if (g->device < 0 || g->device >= SIDE_DEVICES) return;
  std::lock_guard<std::mutex> lock(g_mutex);
  SideRuntime runtime{g->device};
  g_side[g->device].give(runtime, &g->sides);
}

// ---------------------------------------------------------------- the end
// Up to this many counts are added up by the end kernel itself; more get a grid of their own.
constexpr uint64_t END_COUNTS = 32768;
// The host polls this long before it hands the wait to the runtime: a call that takes longer does not notice the
// five microseconds, and one whose kernels fault ends with the runtime's error instead of polling for ever.
constexpr auto POLL_FOR = std::chrono::microseconds(3000);

// Waits until n host words from `from` on carry the number `seq`, and takes their values.  They are written from the graph's stream or one of `sides`.
static int take_values(sky_graph* g, const unsigned long long* from, int n, unsigned long long seq, unsigned long long* values, const hipStream_t* sides = nullptr,
                       int n_sides = 0) {
  constexpr unsigned long long VALUE = (1ull << CALL_VALUE_BITS) - 1;
  auto there = [&] {
    unsigned long long other = 0;
    for (int i = 0; i < n; ++i) {
      const unsigned long long x = __atomic_load_n(from + i, __ATOMIC_ACQUIRE);
      other |= (x ^ seq << CALL_VALUE_BITS) & ~VALUE;
      values[i] = x & VALUE;
    }
    return !other;
  };
  bool done = there();
  if (!done) {
    const auto t0 = std::chrono::steady_clock::now();
    do {
      for (int k = 0; k < 64 && !done; ++k) {
        __builtin_ia32_pause();
        done = there();
      }
    } while (!done && std::chrono::steady_clock::now() - t0 < POLL_FOR);
  }
  if (!done) {
    const int waited = side_wait(1 + n_sides, [&](int k) { return (int)hipStreamSynchronize(k ? sides[k - 1] : g->stream); });
    SKY_HIP((hipError_t)waited);
    if (!there()) return fail(SKY_ERR_HIP, "the call's end was not reported");
  }
  return SKY_OK;
}

int call_answered(sky_graph* g, CallWords* w, unsigned long long* values, int n) {
  return take_values(g, w->host->answer, n, w->asked, values);
}

static int end_call(sky_graph* g, CallWords* w, uint64_t* sampled, double* seconds, const uint32_t* counts, uint64_t n) {
  hipStream_t st = g->stream;
  if (w->sides && (n || w->parts)) return fail(SKY_ERR_ARG, "a call that samples edges does not end over side streams");
  if (n > END_COUNTS) {
    hipLaunchKernelGGL(sum_counts_kernel, dim3((uint32_t)std::min<uint64_t>((n + 255) / 256, 1024)), dim3(256), 0, st, counts,
                       n, w->dev);
    n = 0;
    w->parts = CALL_PARTS;
  }
  const unsigned long long seq = ++w->seq;
  if (w->sides) hipLaunchKernelGGL(call_end_sides_kernel, dim3(1), dim3(1), 0, st, w->dev, w->host, seq, (uint32_t)w->sides + 1);
  else
    hipLaunchKernelGGL(call_end_kernel, dim3(1), dim3(n > 64 ? 1024 : 64), 0, st, w->dev, w->host, seq, counts, (uint32_t)n, w->parts);
  w->parts = 0;
  SKY_HIP(hipGetLastError());
  static_assert(offsetof(CallHost, ticks) == offsetof(CallHost, sampled) + 8, "taken together");
  unsigned long long words[2];
  SKY_TRY(take_values(g, &w->host->sampled, 2, seq, words, w->side, w->sides));
  w->dirty = false;
  if (sampled) *sampled = words[0];
  if (seconds) *seconds = (double)words[1] / ((double)w->khz * 1e3);
  return SKY_OK;
}
int call_end(sky_graph* g, CallWords* w, uint64_t* sampled, double* seconds, const uint32_t* counts, uint64_t n) {
  const int rc = end_call(g, w, sampled, seconds, counts, n);
  if (rc != SKY_OK) (void)side_wait(w->sides, [&](int k) { return (int)hipStreamSynchronize(w->side[k]); });  // the next call clears the words that these write
  w->sides = 0;
  return rc;
}
int call_end(sky_graph* g, uint64_t* sampled, double* seconds, const uint32_t* counts, uint64_t n) {
  return call_end(g, &g->call, sampled, seconds, counts, n);
}

}  // namespace sky
