// Launch plans of the 256 x 128 FP8 tiles (gemm_fp8_scaled.hip).
#pragma once
#include "gemm_tiling.h"

namespace qmm {

constexpr int kM8 = 256, kN8 = 128;  // workgroup tile
constexpr int kConcurrent8 = 32;     // workgroups of an XCD at a time

struct Fp8Plan {
    GemmTiling tiling;
    GemmTail tail;
    double us;  // beside what every launch costs
};

// K ranges that a tile may be cut into at most: tiles that do not fill a round of one workgroup per CU are computed in up to 4 ranges of at
// least 4 k blocks, and only with a workspace that holds the partial tiles (8 XCDs x their tail tiles x parts) in its scratch part.
inline GemmTail fp8_most_ranges(const GemmTiling &tiling, int64_t k, const Workspace &ws) {
    GemmTail tail = make_gemm_tail(tiling, kConcurrent8, kConcurrent8, 4);
    static_assert(tail_counters_fit(kConcurrent8), "one counter per tile that is cut");
    if (ws.scratch == nullptr) tail.parts = 1;
    while (tail.parts > 1 &&
           (k / 128 < 4 * tail.parts || ws.scratch_bytes < int64_t(8) * tail.max_tiles * tail.parts * kM8 * kN8 * 4))
        --tail.parts;
    return tail;
}

// Microseconds of the busiest XCD: the k blocks of its rounds, the longer the more workgroups run together, or the bytes its L2 pulls in where those
// take longer, and the partial tiles of K ranges, out and back in. Fitted to every layout and number of ranges of 28 grids of 5 x 4 to 32 x 4
// tiles, K = 1024 to 7168, so that the plan of the least estimate is the fastest one (0.2 % behind it on average, 2 % at most). Whole rounds alone tell neither
// what K ranges give (10 x 12 tiles, K = 7168, with block scales: regions of 15 tiles in two ranges 41 us, of 18 in one 51) nor what they cost (K = 1024:
// 20.4 and 14.8), and bytes alone leave XCDs without work (13 x 16 tiles, K = 7168: regions of 32 tiles, 24 on some, 59 us, of 26 on each 55).
struct Fp8PlanTime {
    double us, pulled;  // the estimate; what the pulling takes by itself
};
inline Fp8PlanTime fp8_plan_us(const GemmTiling &tiling, int64_t bytes, int parts, int64_t m, int64_t k, bool scaled) {
    struct Cost {
        double least, block, per_tile, pull, exchange, per_part, per_part_tile;
    };
    const Cost c = scaled ? Cost{0.784, 0.649, 0.0062, 0.84e6, 1.0, 1.38, 0.026} : Cost{0.583, 0.279, 0.0121, 1.2e6, 0.84, 1.13, 0.0254};
    const double blocks = double(k) / 128.0;
    const int rounds = int(cdiv(tiling.region_tiles, kConcurrent8)), together = std::min(kConcurrent8, tiling.region_tiles * parts);
    // What the busiest XCD exchanges, times eight: where a part-filled last tile row falls to some XCDs, the others exchange whole tiles only (366 x
    // 7552 x 3328 on one grid row of regions 25.3 us, on two 28.6).
    const double region_rows = double(cdiv(tiling.tiles_m, tiling.xm)) * kM8, exchanged = double(tiling.tiles_m) * tiling.tiles_n * std::min(1.0, double(m) / region_rows);
    const double busy = rounds * blocks * std::max(c.least, c.block + c.per_tile * together) / parts, pulled = double(bytes) * 128.0 * blocks / c.pull;
    return {std::max(busy, pulled) + (parts > 1 ? c.exchange + (c.per_part + c.per_part_tile * exchanged) * parts : 0.0), pulled};
}

// The regions, panels and K ranges of the smallest estimated time, a share of the pulling added to each: of plans that take about the same the one
// that leaves more of the memory system to others.
inline Fp8Plan make_fp8_plan(int64_t m, int64_t n, int64_t k, bool scaled, const Workspace &ws) {
    Fp8Plan best{};
    double least = -1.0;
    for_each_gemm_tiling(int(cdiv(m, kM8)), int(cdiv(n, kN8)), kConcurrent8, kM8, kN8, [&](const GemmTiling &tiling, int64_t bytes) {
        GemmTail tail = fp8_most_ranges(tiling, k, ws);
        for (int parts = tail.parts; parts >= 1; --parts) {
            const Fp8PlanTime t = fp8_plan_us(tiling, bytes, parts, m, k, scaled);
            const double cost = t.us + 0.3 * t.pulled;
            if (least >= 0.0 && cost >= least) continue;
            least = cost;
            tail.parts = parts;
            best = Fp8Plan{tiling, tail, t.us};
        }
    });
    return best;
}

}  // namespace qmm
