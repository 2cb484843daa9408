// Host-only harness over the tile counts of a prefill batch (zerocool_amd/csrc/zc_prefill_tiles.hpp), meant to be built with
// -fsanitize=address,undefined (make asan): no split of a batch's rows over its experts gives more tiles than the host makes room and workgroups for, and
// that many can be, but for what the bound cannot know; the down product's workgroups fill the chip where the batch's tiles allow it.
#include "../../zerocool_amd/csrc/zc_prefill_tiles.hpp"
#include <algorithm>
#include <cstdio>
#include <vector>

static int checks = 0, failures = 0;
#define CHECK(cond) do { ++checks; if (!(cond)) { ++failures; std::printf("  FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond); } } while (0)

int main() {
    for (int32_t count = 0; count <= 10000; ++count) {   // every row is in one tile, none has more than 48
        const int32_t tiles = zc::prefill_tiles_of(count), last = count - (tiles - 1) * 32;
        if (count == 0) CHECK(tiles == 0);
        else CHECK(tiles >= 1 && last >= 1 && last <= 48);
        if (count) CHECK(tiles <= (count + 31) / 32);    // (the shared expert's room)
    }
    constexpr int kRows = 600, kExperts = 24;
    std::vector<int> most(kRows + 1, -1);                // the most tiles that r rows of exactly so many experts can be
    most[0] = 0;
    for (int experts = 1; experts <= kExperts; ++experts) {
        std::vector<int> next(kRows + 1, -1);
        for (int r = 0; r <= kRows; ++r)
            for (int mine = 0; mine <= r; ++mine) next[r] = std::max(next[r], most[r - mine] + zc::prefill_tiles_of(mine));
        most = next;
        for (int r = 0; r <= kRows; ++r) {
            CHECK(most[r] <= int(zc::prefill_max_tiles(r, experts)));
            if (r <= experts) CHECK(most[r] == int(zc::prefill_max_tiles(r, experts)));
        }
    }
    CHECK(zc::prefill_max_tiles(1ull << 31, 1024) == (1u << 26) + 1024);
    for (uint32_t tiles = 8; tiles <= 1024; tiles += 8)
        for (uint32_t blocks = 1; blocks <= 32; ++blocks) {
            const uint32_t share = zc::prefill_short_share(tiles, blocks);
            auto workgroups = [&](uint32_t s) { return tiles * ((blocks + s - 1) / s); };
            CHECK(share == 1 || share == 2 || share == 4);
            if (share > 1) CHECK(workgroups(share) >= 512);
            if (share < 4) CHECK(workgroups(2 * share) < 512);
        }
    // 512 experts, top 10, 2048 weight rows: up to five tokens have a workgroup for every block, twelve and more four blocks a workgroup
    auto share_of = [](uint32_t tokens) { return zc::prefill_short_share((zc::prefill_max_tiles(10ull * tokens, 512) + 7) / 8 * 8, 16); };
    CHECK(share_of(1) == 1 && share_of(5) == 1 && share_of(6) == 2 && share_of(11) == 2 && share_of(12) == 4 && share_of(2048) == 4);
    std::printf("%d checks, %d failures\n", checks, failures);
    return failures ? 1 : 0;
}
