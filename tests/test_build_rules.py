"""Rules by which builds choose their kernels, compiled for the host (CPU only)."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skywalker_amd", "csrc")
DEFAULT = 4000000  # of stream_min_edges
STREAMED, SOME, TILED = range(3)


@pytest.fixture(scope="module")
def narrow_rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rule.cpp").write_text("""
#include <cstdio>
#include "sky_build_rules.h"
int main() {
  long long limit;
  unsigned long long last, stream, wide;
  unsigned longest;
  while (std::scanf("%lld %llu %llu %llu %u", &limit, &last, &stream, &wide, &longest) == 5)
    std::printf("%d\\n", (int)sky::narrow_rows(limit, last, stream, wide, longest));
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "rule.cpp"), "-o", str(d / "rule")], check=True)

    def rule(cases):
        r = subprocess.run([str(d / "rule")], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True, check=True)
        return np.array(r.stdout.split(), int)
    return rule


def test_limit_of_the_streamed_rows(narrow_rows):
    # 0 streams every row of 8,190 to 65,533 entries; a value that the rows do not pass makes all of them tile by tile, if it is not the
    # default, whatever else the build holds; above the limit a build streams them, or the shorter ones, or none by what it would take
    rng = np.random.default_rng(1)
    cases = []
    for _ in range(20000):
        last, stream, wide = (int(10 ** rng.uniform(4, 8.5)) * (rng.random() < 0.8) for _ in range(3))
        longest = int(rng.integers(24577, 3000000)) if stream else int(rng.integers(8190, 24577)) if last else 8000
        limit = [0, DEFAULT, int(10 ** rng.uniform(4, 9)), 1 << 30, last + stream, max(0, last + stream - 1)][rng.integers(0, 6)]
        cases.append((limit, last, stream, wide, longest))
    got = narrow_rows(cases)
    limit, last, stream, wide, longest = (np.array(x) for x in zip(*cases))
    below = last + stream <= limit
    assert (got[limit == 0] == STREAMED).all()
    assert (got[below & (limit > 0) & (limit != DEFAULT)] == TILED).all()
    assert not (got[below & (limit > 0)] == STREAMED).any()
    some = got == SOME
    assert some[below & (limit == DEFAULT)].any() and some[~below].any() and (last[some] > 0).all() and (stream[some] > 0).all()
    for kind in (STREAMED, SOME, TILED):
        assert (got[~below & (limit > 0)] == kind).any()


@pytest.mark.parametrize("limit,last,stream,wide,longest,want", [
    (DEFAULT, 3000000, 600000, 9000000, 30000, SOME),      # 250 rows of 12,000, 20 of 30,000, 1,500 of 6,000
    (1 << 30, 3000000, 600000, 9000000, 30000, TILED),
    (0, 3000000, 600000, 9000000, 30000, STREAMED),
    (DEFAULT, 0, 4500000, 0, 45000, TILED),                # 100 rows of 45,000: 116 us, 142 streamed
    (DEFAULT, 0, 4500000, 2400000, 30000, STREAMED),       # 150 rows of 30,000, 400 of 6,000: 115 us, 135 by tiles
    (DEFAULT, 9000000, 0, 0, 9000, STREAMED),
])
def test_narrow_rows_of_some_builds(narrow_rows, limit, last, stream, wide, longest, want):
    assert narrow_rows([(limit, last, stream, wide, longest)])[0] == want


def test_units_behind_others_go_once_to_a_workgroup_each(tmp_path):
    # every unit from n on to exactly one workgroup, which has it after its own of the n in front and strides on by the grid; the first of
    # them to the workgroup whose turn it is
    (tmp_path / "behind.cpp").write_text("""
#include <cstdio>
#include "sky_build_rules.h"
int main() {
  for (unsigned grid : {1u, 2u, 3u, 7u, 64u, 512u, 2048u, 5120u})
    for (unsigned n : {0u, 1u, 2u, grid - 1u, grid, grid + 1, 3 * grid - 1, 3 * grid, 3 * grid + 5, 4194304u})
      for (unsigned block = 0; block < grid; ++block) {
        const unsigned u = sky::first_behind(n, block, grid);
        if (u < n || u >= n + grid || u % grid != block) return std::printf("%u %u %u: %u\\n", n, block, grid, u), 1;
      }
}
""")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(tmp_path / "behind.cpp"), "-o", str(tmp_path / "behind")], check=True)
    subprocess.run([str(tmp_path / "behind")], check=True)
