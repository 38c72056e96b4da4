// How a call on a graph ends: one small kernel behind the call's last one writes the call's results (sampled edges,
// duration) and a sequence number into pinned host words, which the host polls.  The usual way -- a counter cleared by
// a memset, two events around the kernels, a stream synchronisation, a copy of the counter to the host -- costs
// 29 microseconds around an empty kernel, this one 9 (MI355X, ROCm 7.2: 11 for launch and stream synchronisation, 4 for the events, 3
// for the memset, 11 for the copy; against 6 for a launch that is polled for, 3 for the second launch).
#pragma once
#include <cstddef>

#include "sky_common.h"
#include "sky_sides.h"

struct sky_graph;

namespace sky {

// Device words of a call.  All zero between calls: the end kernel clears what it has read.
// Edges sampled so far, in parts: a word serves its atomics one after another, 5 to 6 ns each, so that 3,900 wavefronts that add to one, each
// at its end, took 23 us of a walk of 104.  A cache line each, and as many as a wavefront has lanes to add them up, for CALL_MANY wavefronts
// and more; fewer have the first (64 parts cost the end 0.6 us).  (One word / parts, us: 250,007 PPR walkers on the scale-24 graph with the index 104 /
// 81, without 127 / 107, 1 M with 277 / 183, 1 M x 5 273 / 160, 200,000 x 40, scale 20, with the index 146 / 126, 100,000 x 60, scale 18, 126 / 120.)
constexpr uint32_t CALL_PARTS = 64, CALL_PART_WORDS = 16, CALL_MANY = 512;
struct CallDevice {
  unsigned long long start;  // wall clock of the first kernel
  unsigned long long entries, arrived, refused;  // sample_check_kernel; the last is left as it is
  uint32_t joined, pad0;     // side streams of a fork that have nothing left (Beside)
  unsigned long long pad[11];
  unsigned long long part[CALL_PARTS * CALL_PART_WORDS];
};
constexpr int CALL_ANSWERS = 10;
// Pinned host words of a call, written by the end kernel: each carries the number of the call in its upper 16 bits, so that the
// host knows which of them has arrived and neither waits for the other on its way over PCIe (results first, then, released, a
// number of their own: a round trip more, 0.4 to 0.8 us of a call of 15 to 30).
struct CallHost {
  unsigned long long sampled, ticks;
  unsigned long long answer[CALL_ANSWERS];  // in the course of a call, with a number of their own (call_ask)
  uint32_t begun, done;                     // what streams wait for (Beside)
  unsigned long long pad[3];
};
constexpr int CALL_VALUE_BITS = 48;  // 2^48 edges fill the GPU's memory a thousand times over; 2^48 ticks of 10 ns are a month
static_assert(sizeof(CallDevice) % 128 == 0 && offsetof(CallDevice, part) == 128 && sizeof(CallHost) == 128, "cache lines of their own");
// Where a call reports.  A graph has one for the calls that begin and end within one entry point; a call that stays open
// between entry points (a sampling session) has its own, because other calls on the graph begin and end meanwhile.
struct CallWords {
  CallDevice* dev = nullptr;
  CallHost* host = nullptr;
  unsigned long long seq = 0, asked = 0;  // numbers of the last end and of the last question
  uint32_t forks = 0;                     // and of the last fork
  int khz = 0;
  int sides = 0;  // side streams over which the call ends beside the graph's, and these
  hipStream_t side[SIDE_STREAMS] = {nullptr, nullptr, nullptr};
  uint32_t parts = 0;  // words that the call's kernels add sampled edges to: none, one or CALL_PARTS
  bool dirty = false;  // a call has begun and not ended well: its device words may not be zero
};

// The call's first kernel: its first thread notes when it began.
__device__ __forceinline__ void call_stamp(CallDevice* call) {
  if (call && blockIdx.x == 0 && threadIdx.x == 0) call->start = wall_clock64();
}
// Adds to the edges sampled; `who`: the number of the workgroup or wavefront, parts: the call's (CallWords).
__device__ __forceinline__ void call_sampled(CallDevice* call, uint32_t who, uint32_t parts, unsigned long long n) {
  if (n) atomicAdd(&call->part[(who & (parts - 1u)) * CALL_PART_WORDS], n);
}
// By one thread of the call's last kernel, which has seen every other thread's contribution.
__device__ __forceinline__ void call_report(CallHost* host, unsigned long long seq, unsigned long long start, unsigned long long sampled) {
  const unsigned long long ticks = start ? wall_clock64() - start : 0;  // 0: the call had nothing to launch
  constexpr unsigned long long VALUE = (1ull << CALL_VALUE_BITS) - 1;
  __hip_atomic_store(&host->sampled, (sampled & VALUE) | seq << CALL_VALUE_BITS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&host->ticks, (ticks & VALUE) | seq << CALL_VALUE_BITS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// How many words `waves` wavefronts that each add once should have.
inline uint32_t call_parts(uint64_t waves) { return waves >= CALL_MANY ? CALL_PARTS : 1u; }
// The device words of `w` (taken on first use), cleared; a call that ended in an error may have left something in them.
int call_begin(sky_graph* g, CallWords* w, CallDevice** call);
// Enqueues the end kernel behind what the call has put on the graph's stream, waits for it and hands out the results.
// Outputs may be null.  `counts` (n of them, device, may be null) are added to the sampled edges; a call that ends over side streams has none.  After
// an error nothing of the call is left on its side streams.
int call_end(sky_graph* g, CallWords* w, uint64_t* sampled, double* seconds, const uint32_t* counts = nullptr, uint64_t n = 0);
// The host's questions in the course of a call: a kernel answers question number call_ask(w) by call_answer, word by word, and
// call_answered waits for the first n.
inline unsigned long long call_ask(CallWords* w) { return ++w->asked; }
__device__ __forceinline__ void call_answer(CallHost* host, unsigned long long number, int word, unsigned long long value) {
  __hip_atomic_store(&host->answer[word], value | number << CALL_VALUE_BITS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
int call_answered(sky_graph* g, CallWords* w, unsigned long long* values, int n);
// Kernels beside those of the graph's stream, on streams that all graphs of a device share (sky_sides.h).  These and the graph's stream wait for one
// another by words in pinned memory: a kernel on the graph's stream notes that it runs (fork_mark), so that everything in front of it has
// ended, and of small last ones on the others the one that finds all of them there that everything in front of these has.  Who waits, by a stream operation (one
// thread of the runtime's that reads the word until the number is there), is always enqueued behind the kernel that writes.  The runtime
// gives a hardware queue what is enqueued in the order of the calls, so that every wait ends: also where other threads' calls lie
// between, where streams share a hardware queue, and where there is only one.  Who waits for the whole device after a call, which does
// not need it, waits 8 to 10 us longer for every side stream that has had work.  2 us
// each way, where events and stream waits take 9 (two kernels of 40 us side by side 55 us in all, with events 68, one after
// the other 89).
struct Beside {
  hipStream_t main = nullptr;
  hipStream_t stream[SIDE_STREAMS] = {nullptr, nullptr, nullptr};  // null: no fork
  bool used[SIDE_STREAMS] = {false, false, false};
  CallDevice* dev = nullptr;
  CallHost* host = nullptr;
  uint32_t number = 0;
  CallWords* last = nullptr;  // of the call that ends with the join: the graph's stream waits for nothing
};
struct ForkMark {
  uint32_t* word;  // null: none
  uint32_t number;
};
__device__ __forceinline__ void fork_mark(const ForkMark& f) {
  if (f.word && blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(f.word, f.number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// A fork over so many side streams, and the mark for the next kernel on the graph's stream.  b->stream stays null where the knob
// build_streams is 0, in the first call of a graph that asks unless the streams are there, on a device without such waits, where the
// streams cannot be made, and where another device than the graph's is current.
int beside_begin(sky_graph* g, Beside* b, ForkMark* mark, int streams);
// With that kernel on its way: side stream k waits for its mark, if it does not already.
int beside_fork(Beside* b, int k);
// The graph's stream waits for what the side streams of the fork hold.  Where nothing but the call's end follows no stream waits: the last kernels of all
// of them report the call together (side_arrive), while a stream's wait takes 4.5 us and 3 more until the next kernel runs.  (A stream's wait / so, us:
// scale 16 with 16 edges a vertex 47.0 / 45.0, scale 18 with 10 61.0 / 58.1, scale 20 with 6 78.9 / 75.5, with 16 120.6 / 118.5, 3 M entries in rows
// of up to 20,000 57.5 / 55.4, 40 M of up to 300,007 311.7 / 309.3, scale 23 with 8 371.8 / 369.6.  An end kernel that waits for the words
// of the others took 0.5 to 1.5 us less, but wants kernels of two queues to run at once, and to give up where they do not.)
int beside_join(Beside* b);
// Instead of a join, after an error: the host waits for them.
void beside_drop(Beside* b);
// A graph that is about to be freed, with nothing of it on the way, gives back its share of the streams.
void beside_release(sky_graph* g);
// With the graph's own words.
int call_begin(sky_graph* g, CallDevice** call);
int call_end(sky_graph* g, uint64_t* sampled, double* seconds, const uint32_t* counts = nullptr, uint64_t n = 0);
// Instead of call_end, for a call that has launched nothing after all.
void call_cancel(sky_graph* g);
void call_release(CallWords* w);

}  // namespace sky
