// Host-side enumeration of launches laid out by make_gemm_tiling_weighted: every tile of the output must be computed exactly once
// whatever the panel width, its K ranges in slots of their own. Built and run by tests/test_weighted_tiling.py.
#include <cstdio>
#include <vector>

#include "gemm_tiling.h"

using namespace qmm;

static int check(int tiles_m, int tiles_n, int concurrent, int row_bytes, int col_bytes) {
    const GemmTiling t = make_gemm_tiling_weighted(tiles_m, tiles_n, concurrent, row_bytes, col_bytes);
    int busiest = 0;
    for (int x = 0; x < 8; ++x) busiest = std::max(busiest, gemm_region_tiles(t, x));
    if (t.xm * t.xn != 8 || t.panel < 1 || t.region_tiles < busiest)
        return std::printf("%dx%d: %d x %d regions, panel %d, %d tiles of %d\n", tiles_m, tiles_n, t.xm, t.xn, t.panel, busiest, t.region_tiles), 1;
    const GemmTail tail = make_gemm_tail(t, concurrent, 32, 4);
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

int main() {
    const int weights[][2] = {{256, 128}, {1, 1}, {512, 64}, {64, 512}};
    long long n = 0;
    for (const auto &w : weights)
        for (int concurrent : {32, 64})
            for (int tm = 1; tm <= 70; tm += (tm < 20 ? 1 : 7))
                for (int tn = 1; tn <= 130; tn += (tn < 50 ? 1 : 9), ++n)
                    if (check(tm, tn, concurrent, w[0], w[1])) return 1;
    std::printf("ok %lld launches\n", n);
    return 0;
}
