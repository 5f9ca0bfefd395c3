// Host-side enumeration of the narrow-tile launches: every workgroup's item lies inside the launch, and every (tile, K stage) is
// taken exactly once. Built and run by tests/test_mid_plan.py; exits non-zero with a message on the first violation.
#include <cstdio>
#include <vector>

#include "gemm_mid.h"

using namespace qmm;

static int check(int tiles_m, int tiles_n, int stages, int want_parts, int groups) {
    // as mid_choose cuts K
    const int share = int(cdiv(cdiv(stages, want_parts), groups)) * groups, parts = int(cdiv(stages, share));
    MidPlan plan{};
    plan.tiles_m = tiles_m;
    plan.tiles_n = tiles_n;
    plan.stages = stages;
    plan.parts = parts;
    plan.share = share;
    plan.tiles_m_magic = mid_magic(tiles_m);
    plan.parts_magic = mid_magic(parts);
    const long long items = 1LL * tiles_m * tiles_n * parts, grid = 8 * cdiv(items, 8);
    std::vector<int> seen(size_t(tiles_m) * tiles_n * stages, 0);
    long long taken = 0;
    for (long long b = 0; b < grid; ++b) {
        MidItem it;
        if (!mid_item(plan, int(b), &it)) continue;
        ++taken;
        if (it.tile_m < 0 || it.tile_m >= tiles_m || it.tile_n < 0 || it.tile_n >= tiles_n || it.tile != it.tile_n * tiles_m + it.tile_m || it.part < 0 ||
            it.part >= parts || it.s_begin < 0 || it.s_begin >= it.s_end || it.s_end > stages)
            return std::printf("%d x %d tiles, %d stages in %d: workgroup %lld has tile (%d, %d) part %d stages %d .. %d\n", tiles_m, tiles_n, stages, parts, b,
                               it.tile_m, it.tile_n, it.part, it.s_begin, it.s_end), 1;
        for (int s = it.s_begin; s < it.s_end; ++s) ++seen[size_t(it.tile) * stages + s];
    }
    if (taken != items) return std::printf("%d x %d tiles: %lld of %lld items\n", tiles_m, tiles_n, taken, items), 1;
    for (size_t i = 0; i < seen.size(); ++i)
        if (seen[i] != 1) return std::printf("%d x %d tiles, %d stages in %d: unit %zu taken %d times\n", tiles_m, tiles_n, stages, parts, i, seen[i]), 1;
    return 0;
}

int main() {
    for (int d = 1; d < 3000; d += d < 40 ? 1 : 37)
        for (long long n : {0LL, 1LL, 2LL, 7LL, 63LL, 64LL, 65LL, 4095LL, 1000003LL, (1LL << 28) - 1, 1LL << 30})
            for (long long e = -1; e <= 1; ++e) {
                const long long v = n / d * d + e;
                if (v >= 0 && mid_div(int(v), d, mid_magic(d)) != int(v) / d) return std::printf("%lld / %d\n", v, d), 1;
            }
    long long count = 0;
    for (int tiles_m : {1, 2, 3, 4, 7, 16, 32})
        for (int tiles_n : {1, 2, 7, 8, 12, 32, 43, 86, 301})
            for (int stages : {1, 2, 3, 8, 17, 32, 128, 344})
                for (int parts = 1; parts <= 8; ++parts)
                    for (int groups : {2, 4, 8}) {
                        if (check(tiles_m, tiles_n, stages, parts, groups)) return 1;
                        ++count;
                    }
    std::printf("ok: %lld launches\n", count);
    return 0;
}
