// Which graphs have side streams (sky_call.h, Beside), how long these are there, and how a call over several streams ends.  Tests compile it for
// the CPU with a runtime of their own.
#pragma once
#include <cstdint>

namespace sky {

constexpr int SIDE_STREAMS = 3;
constexpr int SIDE_IDLE = 16;

// What a graph has of them.
struct SideHold {
  bool held = false;             // they stay as long as it does
  bool refused = false;          // it asked for some that could not be made
  unsigned long long first = 0;  // its first call that asked for some
};
constexpr int SIDE_DEVICES = 64;
// What a call asks with.
struct SideAsk {
  long long knob;       // build_streams
  int device, current;  // the graph's and the one that is current, whose null stream the graph's kernels go to
  unsigned long long call;  // which of the graph's calls, from 1 on
  int streams = SIDE_STREAMS;
  bool allowed() const { return knob != 0 && device == current && device >= 0 && device < SIDE_DEVICES; }
};

// The side streams of one device, shared by the graphs that have asked for them.
// One to three of them take 0.05 to 0.5 ms to make where the process has had as many before, 3.5 ms each where it has not, and 0.7 to 1.2 ms to
// destroy, most of it in the next allocations and frees; a call gains 5 to 100 us by them (MI355X, ROCm 7.2).  So a graph's first call
// that asks finds those that are there and makes none (a graph that is built once never has that back, one whose rows are built again is built
// many times), and they outlast the graphs that had them until SIDE_IDLE graphs in a row have been freed that did without: a program
// that takes one graph after another makes them once.  (The first build of a graph of 17 M entries with its lists and the tables' allocation, no
// other graph there, us: in order 400, on streams that are there 380, on streams of its own 600, of which a process's first 12,000; the
// graph after one that has taken its streams with it also 0.5 ms later to upload.)
// Calls are the caller's to serialise.  Runtime: can(), whether the device has what they wait with; create(Stream*); destroy(Stream).
template <class Runtime>
struct SidePool {
  using Stream = typename Runtime::Stream;
  Stream stream[SIDE_STREAMS] = {};
  int holders = 0, without = 0;  // graphs freed since the last holder

  // Whether the graph has them for the present call; without, its kernels go out in order, after some that could not be made for good.
  bool take(Runtime& rt, SideHold* h, const SideAsk& ask) {
    if (!ask.allowed() || h->refused) return false;
    if (!h->first) h->first = ask.call;
    for (int k = 0; k < ask.streams; ++k) {
      Stream& s = stream[k];
      if (s) continue;
      if (h->first == ask.call) return false;
      if (rt.can() && rt.create(&s)) continue;
      s = Stream{};
      h->refused = true;  // those made before it are for graphs that need fewer
      return false;
    }
    if (!h->held) ++holders;
    h->held = true;
    return true;
  }
  // The graph is about to be freed.
  void give(Runtime& rt, SideHold* h) {
    if (h->held) {
      --holders;
      without = 0;
    } else if (holders == 0 && ++without >= SIDE_IDLE) {
      clear(rt);
    }
    *h = SideHold{};
  }

 private:
  void clear(Runtime& rt) {
    for (Stream& s : stream) {
      if (s) rt.destroy(s);
      s = Stream{};
    }
  }
};

// The last kernels of the streams of a call that ends over `of` of them, one each.  The one that finds all the others there reports, whatever the order
// they run in: none waits for another, so that they may also run one at a time.  What the next call uses is cleared before the report, behind which
// its kernels may follow on any of the streams.
template <class Words>
constexpr bool side_arrive(Words words, uint32_t of) {
  if (words.arrive() != of) return false;
  words.report(words.clear());
  return true;
}
// The host's wait for n streams: for all of them, also after an error.  The first error, or 0.
template <class Wait>
int side_wait(int n, Wait wait) {
  int first = 0;
  for (int k = 0; k < n; ++k) {
    const int rc = wait(k);
    if (!first) first = rc;
  }
  return first;
}

}  // namespace sky
