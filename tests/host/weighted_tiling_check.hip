// Host-side enumeration of launches laid out by for_each_gemm_tiling: every tile of the output must be computed exactly once
// whatever the regions and the panel width, its K ranges in slots of their own. And the plans of the FP8 tiles: what they promise fits the
// workspace, and a deep matrix is cut into K ranges where make_gemm_tiling's layout allows it, within one and a half times the rounds of as many ranges as that allows. Built and run by
// tests/test_weighted_tiling.py.
#include <cstdio>
#include <vector>

#include "gemm_fp8_plan.h"

using namespace qmm;

static int check(const GemmTiling &t, int concurrent, const GemmTail &tail) {
    const int tiles_m = t.tiles_m, tiles_n = t.tiles_n;
    int busiest = 0;
    for (int x = 0; x < 8; ++x) busiest = std::max(busiest, gemm_region_tiles(t, x));
    if (t.xm * t.xn != 8 || t.panel < 1 || t.region_tiles < busiest)
        return std::printf("%dx%d: %d x %d regions, panel %d, %d tiles of %d\n", tiles_m, tiles_n, t.xm, t.xn, t.panel, busiest, t.region_tiles), 1;
    std::vector<int> seen(size_t(tiles_m) * tiles_n * 4, 0), slot_owner(size_t(8) * std::max(1, tail.max_tiles), -1);
    for (long long b = 0, grid = gemm_grid_with_tail(t, concurrent, tail); b < grid; ++b) {
        GemmWorkItem it;
        if (!gemm_work_item_of_block(int(b), tiles_m, tiles_n, t.xm, t.xn, concurrent, tail.parts, tail.max_tiles, &it, t.panel)) continue;
        const int tile = it.tile_m * tiles_n + it.tile_n;
        if (it.tile_m < 0 || it.tile_m >= tiles_m || it.tile_n < 0 || it.tile_n >= tiles_n || it.parts != tail.parts || seen[size_t(tile) * 4 + it.part]++)
            return std::printf("%dx%d panel %d: block %lld -> (%d, %d) part %d of %d\n", tiles_m, tiles_n, t.panel, b, it.tile_m, it.tile_n, it.part, it.parts), 1;
        if (it.parts > 1) {
            if (it.slot < 0 || it.slot >= int(slot_owner.size()) || (slot_owner[it.slot] >= 0 && slot_owner[it.slot] != tile))
                return std::printf("%dx%d panel %d: slot %d of block %lld\n", tiles_m, tiles_n, t.panel, it.slot, b), 1;
            slot_owner[it.slot] = tile;
        }
    }
    for (int tile = 0; tile < tiles_m * tiles_n; ++tile)
        for (int p = 0; p < tail.parts; ++p)
            if (seen[size_t(tile) * 4 + p] != 1) return std::printf("%dx%d panel %d: tile %d part %d missing\n", tiles_m, tiles_n, t.panel, tile, p), 1;
    return 0;
}

// Rounds of whole tiles on the busiest XCD.
static double rounds(const GemmTiling &t, int parts) {
    return double(cdiv(int64_t(t.region_tiles) * parts, kConcurrent8)) / parts;
}

static int check_plan(int64_t m, int64_t n, int64_t k, bool scaled, const Workspace &ws) {
    const Fp8Plan plan = make_fp8_plan(m, n, k, scaled, ws);
    const GemmTail most = fp8_most_ranges(plan.tiling, k, ws);
    if (plan.tail.parts < 1 || plan.tail.parts > most.parts || plan.tail.max_tiles != most.max_tiles || !(plan.us > 0.0) ||
        (plan.tail.parts > 1 && int64_t(8) * plan.tail.max_tiles * plan.tail.parts * kM8 * kN8 * 4 > ws.scratch_bytes))
        return std::printf("%lld x %lld x %lld: %d ranges of %d\n", (long long)m, (long long)k, (long long)n, plan.tail.parts, most.parts), 1;
    if (check(plan.tiling, kConcurrent8, plan.tail)) return 1;
    if (k < 7168) return 0;
    const GemmTiling square = make_gemm_tiling(int(cdiv(m, kM8)), int(cdiv(n, kN8)), kConcurrent8);
    const GemmTail ranges = fp8_most_ranges(square, k, ws);
    if (plan.tail.parts < std::min(2, ranges.parts) || rounds(plan.tiling, plan.tail.parts) > 1.5 * rounds(square, ranges.parts))
        return std::printf("%lld x %lld x %lld: %d regions by %d of %d tiles in %d ranges, make_gemm_tiling's of %d in %d\n", (long long)m, (long long)k, (long long)n,
                           plan.tiling.xm, plan.tiling.xn, plan.tiling.region_tiles, plan.tail.parts, square.region_tiles, ranges.parts), 1;
    return 0;
}

int main() {
    const int weights[][2] = {{256, 128}, {1, 1}, {512, 64}, {64, 512}};
    long long n = 0;
    int wrong = 0;
    for (const auto &w : weights)
        for (int concurrent : {32, 64})
            for (int tm = 1; tm <= 70; tm += (tm < 20 ? 1 : 7))
                for (int tn = 1; tn <= 130; tn += (tn < 50 ? 1 : 9))
                    for_each_gemm_tiling(tm, tn, concurrent, w[0], w[1], [&](const GemmTiling &t, int64_t) {
                        ++n;
                        wrong += check(t, concurrent, make_gemm_tail(t, concurrent, 32, 4));
                    });
    if (wrong) return 1;
    char *const somewhere = reinterpret_cast<char *>(4096);
    for (bool scaled : {false, true})
        for (int64_t k : {128, 1024, 2048, 3072, 7168})
            for (int tm = 1; tm <= 64; tm += (tm < 20 ? 1 : 7))
                for (int tn = 1; tn <= 64; tn += (tn < 25 ? 1 : 5))
                    for (int64_t scratch : {int64_t(0), int64_t(20) << 20, int64_t(256) << 20}) {
                        Workspace ws{};
                        if (scratch > 0) ws.scratch = somewhere, ws.scratch_bytes = scratch;
                        ++n;
                        if (check_plan(int64_t(tm) * kM8 - (tm * 37 + tn * 11) % kM8, int64_t(tn) * kN8, k, scaled, ws)) return 1;
                    }
    std::printf("ok %lld launches\n", n);
    return 0;
}
