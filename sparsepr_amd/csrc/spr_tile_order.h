// Order in which a call's 256-row attention tiles go to the workgroups of attn_pipe_kernel.
//
// Workgroup b runs on XCD b % 8 and the workgroups start in order, so the order decides which
// tiles share an L2 and which run last.  The heads come in decreasing work and each head's tiles in
// decreasing key count (the plan's orders).
//   - First a run of the longest tiles of every head that would start in the last eight rounds over
//     the chip, then everything else: a tile that starts late has to be short.  A prompt's query
//     tile keeps every key and walks 1 / density times the chunks of its neighbours: 8 heads of
//     35,400 tokens with 512 of a prompt 1.80 ms head by head, 1.27 so.  The first part reads many
//     heads' keys at once, so it is kept short: with a sixteenth of every head's tiles in it 24
//     heads of 118,800 tokens take 1.5 % longer.
//   - Within each of the two the heads follow one another and a head's tiles go to the XCDs in
//     turn, `run` at a time: the XCDs end together whatever the heads' number and densities, all
//     read the same head's keys (61 MB at 118,800 tokens, which the 256 MB last-level cache holds;
//     eight heads it does not), and the tiles of a q-cluster mostly share an L2.  Against whole
//     heads dealt to XCDs: 5 heads of 35,400 tokens 0.94 -> 0.78 ms, 8 heads whose densities differ
//     by up to 4 2.06 -> 1.31, 24 heads of 119,056 45.3 -> 42.9, 8, 16 or 24 heads alike in
//     density 0 to 4 % slower.
//   - Runs of 8, in heads of less than 128 tiles of 4: a longer run costs a short call up to 5 %
//     where its last round is uneven, a shorter one the 24 x 118,800 layer 0.5 to 1.5 %.  Heads of
//     less than 32 tiles take runs of 2 (256 heads of 1,024 tokens 122 us against 136).
//   - A head's share of either part is an odd number of runs, so its longest tiles fall to
//     another XCD than those of the head before it.
#pragma once

#include <algorithm>
#include <cstdint>

namespace spr {

struct TileOrder {
  int32_t run;              // consecutive tiles of a head on one XCD
  int32_t heads, whole;     // the call's heads; the first `whole` have all their tiles in the second part
  int32_t lead, rest, all;  // tiles of a head in the first part (a run), the second, in all: whole runs
  int32_t lead_groups;      // workgroups of the first part (a whole number of turns over the XCDs)
  int64_t groups;           // of both

  // tiles_of_rows = ceil(rows / 256), max_tiles the most tiles a head can have
  __host__ static TileOrder make(int64_t tiles_of_rows, int64_t max_tiles, int64_t heads) {
    constexpr int64_t CUS = 256, LATE_ROUNDS = 8;
    TileOrder o{};
    o.run = tiles_of_rows >= 128 ? 8 : tiles_of_rows >= 32 ? 4 : 2;
    auto part = [&](int64_t tiles) { return (((tiles + o.run - 1) / o.run) | 1) * o.run; };
    auto groups = [&](int64_t tiles) { return (tiles + 8 * o.run - 1) / (8 * o.run) * (8 * o.run); };
    const int64_t late = std::min(heads, LATE_ROUNDS * CUS / std::max<int64_t>(tiles_of_rows, 1) + 1);
    const int64_t lead = o.run;
    const int64_t rest = max_tiles > lead ? part(max_tiles - lead) : 0;
    const int64_t all = part(max_tiles);
    o.heads = static_cast<int32_t>(heads);
    o.whole = static_cast<int32_t>(heads - late);
    o.lead = static_cast<int32_t>(lead);
    o.rest = static_cast<int32_t>(rest);
    o.all = static_cast<int32_t>(all);
    o.lead_groups = static_cast<int32_t>(groups(lead * late));
    o.groups = groups(lead * late) + groups(all * o.whole + rest * late);
    return o;
  }

  // The head and tile of workgroup b; a head at or past the call's heads is none.
  __host__ __device__ void at(uint32_t b, int64_t& head, int32_t& tile) const {
    const bool first = b < static_cast<uint32_t>(lead_groups);
    const uint32_t w = first ? b : b - lead_groups, r = run;
    uint32_t pos = (w / (8 * r) * 8 + w % 8) * r + w / 8 % r;  // [turn][XCD][in the run]
    const bool late = first || pos >= static_cast<uint32_t>(whole) * all;
    if (!first && late) pos -= static_cast<uint32_t>(whole) * all;
    const uint32_t per = first ? lead : late ? rest : all;
    if (per == 0) {  // padding behind heads that the first part held whole
      head = heads;
      tile = 0;
      return;
    }
    const uint32_t h = pos / per;
    head = h + (late ? whole : 0);
    tile = static_cast<int32_t>(pos - h * per + (late && !first ? lead : 0));
  }
};

}  // namespace spr
