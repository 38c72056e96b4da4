// Which graphs have side streams (sky_call.h, Beside), and how long these are there.  Host code without a kernel: tests compile it for the CPU
// with a runtime of their own.
#pragma once
#include <cstdint>

namespace sky {

constexpr int SIDE_STREAMS = 3;

// What a graph has of them.
struct SideHold {
  bool held = false;     // they stay as long as it does
  bool refused = false;  // it asked for some that could not be made
};
constexpr int SIDE_DEVICES = 64;
// What a call asks with.
struct SideAsk {
  long long knob;       // build_streams
  int device, current;  // the graph's and the one that is current, whose null stream the graph's kernels go to
  bool allowed() const { return knob != 0 && device == current && device >= 0 && device < SIDE_DEVICES; }
};

// The side streams of one device: shared by the graphs that have asked for them, and destroyed when the last of these is freed.  Calls
// are the caller's to serialise.  Runtime: can(), whether the device has what they wait with; create(Stream*); destroy(Stream).
template <class Runtime>
struct SidePool {
  using Stream = typename Runtime::Stream;
  Stream stream[SIDE_STREAMS] = {};
  int holders = 0;

  // Whether the graph has them for the present call; without, its kernels go out in order, after some that could not be made for good.
  bool take(Runtime& rt, SideHold* h, const SideAsk& ask) {
    if (!ask.allowed() || h->refused) return false;
    for (Stream& s : stream) {
      if (s || (rt.can() && rt.create(&s))) continue;
      s = Stream{};
      h->refused = true;
      if (!holders) clear(rt);
      return false;
    }
    if (!h->held) ++holders;
    h->held = true;
    return true;
  }
  // The graph is about to be freed.
  void give(Runtime& rt, SideHold* h) {
    if (h->held && --holders == 0) clear(rt);
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

}  // namespace sky
