// Which graphs have side streams (sky_call.h, Beside), and how long these are there.  Host code without a kernel: tests compile it for the CPU
// with a runtime of their own.
#pragma once
#include <cstdint>

namespace sky {

constexpr int SIDE_STREAMS = 3;

// What a graph has of them.
struct SideHold {
  bool held = false;  // they stay as long as it does
};

// The side streams of one device: shared by the graphs that have asked for them, and destroyed when the last of these is freed.  Calls
// are the caller's to serialise.  Runtime: int create(Stream*), 0 or an error, and destroy(Stream).
template <class Runtime>
struct SidePool {
  using Stream = typename Runtime::Stream;
  Stream stream[SIDE_STREAMS] = {};
  int holders = 0;

  int take(Runtime& rt, SideHold* h) {
    for (Stream& s : stream) {
      const int rc = s ? 0 : rt.create(&s);
      if (rc == 0) continue;
      s = Stream{};
      if (!holders) clear(rt);
      return rc;
    }
    if (!h->held) ++holders;
    h->held = true;
    return 0;
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
