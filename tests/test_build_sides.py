"""Which graphs have side streams for their builds and how long these are there, compiled for the host with a runtime that counts (CPU only)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skywalker_amd", "csrc")
MAIN = """
#undef NDEBUG
#include <cassert>
#include <set>
#include "sky_sides.h"
using namespace sky;
struct Runtime {
  using Stream = int*;
  std::set<int*> live;
  int made = 0, fail_from = 1000;  // streams made so far; number of the first that cannot be made
  bool able = true;
  bool can() const { return able; }
  bool create(Stream* s) {
    if (made >= fail_from) {
      *s = (int*)8;  // whatever a failing call leaves behind
      return false;
    }
    ++made;
    live.insert(*s = new int);
    return true;
  }
  void destroy(Stream s) {
    assert(live.erase(s) == 1);
    delete s;
  }
};
int main() {
  Runtime rt;
  SidePool<Runtime> pool;
  const SideAsk yes{1, 0, 0};
  %s
}
"""


@pytest.fixture()
def run(tmp_path):
    def go(body):
        (tmp_path / "sides.cpp").write_text(MAIN % body)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "sides.cpp"), "-o", str(tmp_path / "sides")], check=True)
        subprocess.run([str(tmp_path / "sides")], check=True)
    return go


def test_streams_are_shared_and_go_with_the_last_graph_that_has_them(run):
    run("""
  for (int round = 0; round < 3; ++round) {
    SideHold a, b, never;
    assert(pool.take(rt, &a, yes) && pool.take(rt, &a, yes) && pool.take(rt, &b, yes));
    assert(rt.live.size() == SIDE_STREAMS && rt.made == SIDE_STREAMS * (round + 1));
    pool.give(rt, &never);
    pool.give(rt, &a);
    pool.give(rt, &a);
    assert(rt.live.size() == SIDE_STREAMS && !a.held && b.held);
    pool.give(rt, &b);
    assert(rt.live.empty() && pool.holders == 0);
  }
""")


@pytest.mark.parametrize("able,fail_from", [(0, 1000), (1, 0), (1, 1), (1, 2)])
def test_a_graph_does_without_streams_that_cannot_be_made(run, able, fail_from):
    # those that were made before the one that failed go back; the graph does not ask again, others do
    run("""
  SideHold a, b;
  rt.able = %d, rt.fail_from = %d;
  assert(!pool.take(rt, &a, yes) && !a.held && rt.live.empty() && pool.holders == 0);
  rt.able = true, rt.fail_from = 1000;
  const int made = rt.made;
  assert(!pool.take(rt, &a, yes) && rt.made == made);
  assert(pool.take(rt, &b, yes) && rt.live.size() == SIDE_STREAMS);
  pool.give(rt, &a);
  assert(rt.live.size() == SIDE_STREAMS && pool.take(rt, &a, yes));
  pool.give(rt, &b);
  pool.give(rt, &a);
  assert(rt.live.empty());
""" % (able, fail_from))


@pytest.mark.parametrize("ask", ["0, 0, 0", "1, 0, 1", "1, 1, 0", "1, 0, -1", "1, -1, -1", "1, 64, 64"])
def test_no_fork_with_the_knob_off_or_another_device_current(run, ask):
    # nor where the streams are there, for this graph too; nothing is made, nothing held
    run("""
  const SideAsk no{%s};
  SideHold a, b;
  assert(!pool.take(rt, &a, no) && rt.made == 0 && !a.held);
  assert(pool.take(rt, &a, yes) && !pool.take(rt, &a, no) && a.held);
  assert(!pool.take(rt, &b, no) && !b.held && pool.holders == 1);
  assert(pool.take(rt, &b, yes) && pool.holders == 2);
  pool.give(rt, &a);
  pool.give(rt, &b);
  assert(rt.live.empty());
""" % ask)
