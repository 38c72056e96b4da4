"""Which graphs have side streams for their builds, how long these are there and how a call over several streams ends, compiled for the host with a runtime that counts (CPU only)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skywalker_amd", "csrc")
MAIN = """
#undef NDEBUG
#include <algorithm>
#include <cassert>
#include <set>
#include <vector>
#include "sky_sides.h"
using namespace sky;
struct Asked : SideHold {
  Asked() { first = 1; }  // a graph that asked in its first call
};
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
  const SideAsk yes{1, 0, 0, 2}, first{1, 0, 0, 1};
  (void)yes, (void)first;
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


def test_streams_are_shared_and_go_when_graphs_do_without(run):
    # graph after graph, one at a time or several, on the streams of the first; after SIDE_IDLE freed in a row without, they are made again
    run("""
  for (int round = 1; round <= 3; ++round) {
    for (int k = 0; k < 40; ++k) {
      Asked a, b;
      SideHold never;
      assert(pool.take(rt, &a, yes) && pool.take(rt, &a, yes) && pool.take(rt, &b, yes) && pool.holders == 2);
      pool.give(rt, &a);
      pool.give(rt, &b);
      assert(!a.held && !a.first && pool.holders == 0 && rt.made == SIDE_STREAMS * round);
      pool.give(rt, &never);
    }
    Asked c;
    assert(pool.take(rt, &c, yes));
    SideHold never;
    for (int k = 0; k < 2 * SIDE_IDLE; ++k) pool.give(rt, &never);
    assert(rt.live.size() == SIDE_STREAMS);  // whatever others do, not while a graph has them
    pool.give(rt, &c);
    for (int k = 0; k < SIDE_IDLE; ++k) {
      assert(rt.live.size() == SIDE_STREAMS);
      pool.give(rt, &never);
    }
    assert(rt.live.empty() && rt.made == SIDE_STREAMS * round);
  }
""")


@pytest.mark.parametrize("able,fail_from", [(0, 1000), (1, 0), (1, 1), (1, 2)])
def test_a_graph_does_without_streams_that_cannot_be_made(run, able, fail_from):
    # the graph does not ask again, others do
    run("""
  Asked a, b;
  rt.able = %d, rt.fail_from = %d;
  assert(!pool.take(rt, &a, yes) && !a.held && pool.holders == 0);
  rt.able = true, rt.fail_from = 1000;
  const int made = rt.made;
  assert(!pool.take(rt, &a, yes) && rt.made == made);
  assert(pool.take(rt, &b, yes) && rt.live.size() == SIDE_STREAMS);
  pool.give(rt, &a);
  a.first = 1;
  assert(rt.live.size() == SIDE_STREAMS && pool.take(rt, &a, yes));
  pool.give(rt, &b);
  pool.give(rt, &a);
  for (int k = 0; k < SIDE_IDLE; ++k) pool.give(rt, &b);
  assert(rt.live.empty());
""" % (able, fail_from))


@pytest.mark.parametrize("ask", ["0, 0, 0", "1, 0, 1", "1, 1, 0", "1, 0, -1", "1, -1, -1", "1, 64, 64"])
def test_no_fork_with_the_knob_off_or_another_device_current(run, ask):
    # nor where the streams are there, for this graph too; nothing is made, nothing held
    run("""
  const SideAsk no{%s, 2};
  Asked a, b;
  assert(!pool.take(rt, &a, no) && rt.made == 0 && !a.held);
  assert(pool.take(rt, &a, yes) && !pool.take(rt, &a, no) && a.held);
  assert(!pool.take(rt, &b, no) && !b.held && pool.holders == 1);
  assert(pool.take(rt, &b, yes) && pool.holders == 2 && rt.made == SIDE_STREAMS);
""" % ask)


def test_a_graphs_first_call_makes_no_streams(run):
    # however often it asks; it takes those that another graph has, as many as there are
    run("""
  SideHold a, b, c, d;
  SideAsk one = yes, later{1, 0, 0, 7};
  one.streams = 1;
  for (int k = 0; k < 3; ++k) assert(!pool.take(rt, &a, first) && !a.held && !a.refused);
  assert(rt.made == 0 && pool.take(rt, &a, one) && rt.made == 1 && pool.take(rt, &a, one) && rt.made == 1);
  SideAsk b1 = first;
  b1.streams = 1;
  assert(pool.take(rt, &b, b1) && b.held && rt.made == 1 && !pool.take(rt, &b, first) && rt.made == 1);
  assert(pool.take(rt, &b, yes) && rt.made == SIDE_STREAMS && pool.holders == 2);
  assert(pool.take(rt, &c, later) && rt.made == SIDE_STREAMS);
  pool.give(rt, &a), pool.give(rt, &b), pool.give(rt, &c);
  for (int k = 0; k < SIDE_IDLE; ++k) pool.give(rt, &d);
  assert(rt.live.empty() && !pool.take(rt, &d, later) && rt.live.empty());
""")


def test_a_graph_that_holds_one_stream_keeps_it_where_another_cannot_be_made(run):
    run("""
  Asked a, b;
  SideAsk one = yes;
  one.streams = 1;
  rt.fail_from = 2;
  assert(pool.take(rt, &a, one) && !pool.take(rt, &a, yes) && a.held && a.refused && !pool.take(rt, &a, one));
  assert(pool.take(rt, &b, one) && rt.live.size() == 2 && pool.holders == 2);
""")


@pytest.mark.parametrize("sides", [1, 2, 3])
def test_a_call_over_several_streams_ends_with_whichever_kernel_is_last(run, sides):
    # the last kernels of the streams one at a time, in every order: each runs to its end, the last of them reports, once, with the words cleared
    # before it does; call after call
    run("""
  static uint32_t joined, reports;
  static unsigned long long start;
  struct Words {
    uint32_t arrive() { return ++joined; }
    unsigned long long clear() {
      const unsigned long long s = start;
      joined = 0, start = 0;
      return s;
    }
    void report(unsigned long long s) {
      assert(s == 77 && joined == 0 && start == 0);
      ++reports;
    }
  };
  const uint32_t of = %d + 1;
  std::vector<int> order(of);
  for (uint32_t k = 0; k < of; ++k) order[k] = k;  // 0: the graph's stream
  uint32_t calls = 0;
  do {
    start = 77;
    for (uint32_t k = 0; k < of; ++k) {
      assert(reports == calls);
      assert(side_arrive(Words{}, of) == (k + 1 == of));
    }
    assert(reports == ++calls && joined == 0);
  } while (std::next_permutation(order.begin(), order.end()));
""" % sides)


@pytest.mark.parametrize("failing", [-1, 0, 1, 2])
def test_every_stream_of_a_call_is_waited_for_also_after_an_error(run, failing):
    run("""
  const int failing = %d;
  std::vector<int> waited;
  const int rc = side_wait(4, [&](int k) {
    waited.push_back(k);
    return k == failing ? 700 : k == 3 && failing >= 0 ? 701 : 0;
  });
  assert(rc == (failing >= 0 ? 700 : 0) && waited == (std::vector<int>{0, 1, 2, 3}));
  assert(side_wait(0, [&](int) { return 1; }) == 0);
""" % failing)
