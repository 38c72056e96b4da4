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
  int create(Stream* s) {
    if (made >= fail_from) return 7;
    ++made;
    live.insert(*s = new int);
    return 0;
  }
  void destroy(Stream s) {
    assert(live.erase(s) == 1);
    delete s;
  }
};
int main() {
  Runtime rt;
  SidePool<Runtime> pool;
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
    assert(pool.take(rt, &a) == 0 && pool.take(rt, &a) == 0 && pool.take(rt, &b) == 0);
    assert(rt.live.size() == SIDE_STREAMS && rt.made == SIDE_STREAMS * (round + 1));
    pool.give(rt, &never);
    pool.give(rt, &a);
    pool.give(rt, &a);
    assert(rt.live.size() == SIDE_STREAMS && !a.held && b.held);
    pool.give(rt, &b);
    assert(rt.live.empty() && pool.holders == 0);
  }
""")


def test_streams_made_before_one_that_fails_go_back_unless_another_graph_has_them(run):
    run("""
  SideHold a, b;
  rt.fail_from = 2;
  assert(pool.take(rt, &a) == 7 && !a.held && rt.live.empty());
  rt.fail_from = 1000;
  assert(pool.take(rt, &a) == 0 && pool.take(rt, &b) == 0);
  pool.give(rt, &b);
  pool.give(rt, &a);
  assert(rt.live.empty());
""")
