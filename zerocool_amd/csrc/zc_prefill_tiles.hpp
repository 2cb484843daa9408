// How a prefill batch's sorted rows are cut into tiles, and what the host knows of their number before the routing is there.  Plain C++: the
// kernels, the launches and a host test share it.
#pragma once
#include <cstdint>

namespace zc {

constexpr uint32_t kTileRows = 32, kTileRowsMax = 48;
// tiles of an expert's `count` rows: whole ones of 32; what is left joins the last of them when that gives at most 48 rows, else it is a tile of its own
constexpr int32_t prefill_tiles_of(int32_t count) {
    const int32_t whole = count / int32_t(kTileRows), left = count % int32_t(kTileRows);
    return count == 0 ? 0 : (whole == 0 ? 1 : whole + (left > int32_t(kTileRowsMax - kTileRows) ? 1 : 0));
}
// The most tiles that n rows of so many experts can be: one more than its whole 32s for every expert that has rows at all.  An upper bound: a
// batch whose tokens agree on their experts has fewer.
constexpr uint32_t prefill_max_tiles(uint64_t n, uint32_t experts) { return uint32_t(n / kTileRows + (n < experts ? n : experts)); }
// Blocks of 128 weight rows that a workgroup of the down product of rows of 512 takes in turn: four, or so many fewer that there are two workgroups
// a compute unit by that bound.  (While every expert counted in it, used or not, a token's ten experts of 512 had 40 workgroups of 2048 weight rows,
// where a workgroup a block is 160.  The line is by count: batches of fewer than twelve tokens, the only ones it moves there, have not been timed on its two sides.)
constexpr uint32_t prefill_short_share(uint32_t tiles, uint32_t blocks) {
    uint32_t share = 4;
    while (share > 1 && uint64_t(tiles) * ((blocks + share - 1) / share) < 512) share /= 2;
    return share;
}

}  // namespace zc
