// How a build in few launches makes its rows of 8190..65533 entries, and who has which of a launch's units; plain C++, without the device.
#pragma once
#include <algorithm>
#include <cstdint>

namespace sky {

constexpr long long STREAM_MIN_EDGES = 4000000;  // default of the option stream_min_edges

enum class NarrowRows { STREAMED, TO_24576_STREAMED, TILED };

// Rows of 8190..65533 entries are streamed, one workgroup each, by builds that hold enough of them to fill the GPU that way (more than
// `limit` entries, and always if that is 0), and made tile by tile by the others; where the longest of them would outlast everything else
// either all of them or those of more than 24,576 entries are made tile by tile whatever they hold together.  At the default limit,
// which is where the two take about as long, builds below it stream those of up to 24,576 as well if that takes less.
// A workgroup takes 2.4 ns an entry for such a row, and the launch lasts at least as long as the longest of them.
// The launch of the rows of 2558..65533 entries as a whole takes 6 ps an entry, the tile passes 13 ps (one
// MI355X; this tells the faster way for 13 of 13 graphs of 4 to 117 M entries: 40 M entries in rows of 1..300,000
// 409 -> 367 us by tiles, R-MAT scale 22 edge factor 28 754 us streamed, 888 by tiles).  Rows of up to 24,576 streamed and the longer ones
// by tiles: an online walk of 10,000 x 8 on the scale-22 graph with 16 edges a vertex 222 -> 197 us, a build with 10 272 -> 264, below the
// limit one of 250 rows of 12,000, 20 of 30,000 and 1,500 of 6,000 169 -> 156.
// last, stream: entries in rows of 8190..24576 and of 24577..65533; wide: in those of 2558..8189.
inline NarrowRows narrow_rows(long long limit, uint64_t last, uint64_t stream, uint64_t wide, uint32_t max_degree) {
  constexpr uint32_t HELD = 8189, LAST = 24576, STREAM = 65533;
  const uint64_t narrow = last + stream;
  if (limit == 0) return NarrowRows::STREAMED;
  auto us = [&](uint64_t streamed, uint32_t longest) {
    return std::max(std::min(max_degree, longest) * 2.4e-3, (double)(wide + streamed) * 6e-6) + (double)(narrow - streamed) * 13e-6;
  };
  const double none_us = us(0, HELD), last_us = us(last, LAST), all_us = us(narrow, stream ? STREAM : LAST);
  const bool below = (long long)narrow <= limit;
  const bool some = last > 0 && stream > 0 && last_us < none_us && (!below || limit == STREAM_MIN_EDGES);
  if (!below && all_us <= (some ? last_us : none_us)) return NarrowRows::STREAMED;
  return some ? NarrowRows::TO_24576_STREAMED : NarrowRows::TILED;
}

// The first unit from n on for workgroup `block` of `grid`, which of the n in front has units block, block + grid, ...: what follows few
// goes to workgroups without (476 seeds 5 x 3 on the scale-22 graph with 5 edges a vertex 88 us where the first ones have both, 75 so).
// A division of 32-bit numbers takes a wavefront a good part of a microsecond, launches of short rows as long as a tenth of their work:
// none where nothing is in front.
constexpr uint32_t first_behind(uint32_t n, uint32_t block, uint32_t grid) {
  if (n == 0) return block;
  const uint32_t at = block + grid - n % grid;
  return n + (at < grid ? at : at - grid);
}

}  // namespace sky
