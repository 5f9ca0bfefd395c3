// W4A16 on small weights: c[m, n] = sum_k a[m, k] * q[k, n] * scales[k / group, n] (+ bias[n]), packed int4 codes (two columns to a byte, row-major), a workgroup per 16 RB rows and
// 16 CB columns (CB = 2 or 4) for all of K, without an exchange between workgroups: as skinny_w8a16_small.hip, which says what bounds it and why.
//
// Codes are widened exactly (bfloat16: q / 16 of a nibble by v_cvt_off_f32_i4, float16: 1032 + q less 1032); the products of 32 G rows of a group (G = 2 or 4, groups of a multiple of 64
// or 128) are summed from zero and added times the group's scale in float32. bfloat16, groups of 128, us, before -> here, weights from the last-level cache: 1 x 1024 x 512 6.3 -> 3.6, 4 x
// 1536 x 2048 7.6 -> 4.5, 16 x 1024 x 4096 7.2 -> 3.9, 16 x 2048 x 6144 8.7 -> 6.4, 64 x 1536 x 4096 8.6 -> 5.9, 128 x 512 x 512 6.3 -> 3.4.
#include "common.h"
#include "skinny_w4a16_small.h"
#include "w4_traits.h"

#include <cmath>

namespace qmm {
namespace {

constexpr int64_t kSmallMostRows = 512, kSmallMostK = 4096, kSmallMostBytes = 6300000, kFewRowsMostK = 2944;  // (kFewRows...: up to 16 rows)
// Rounds of one workgroup per CU, beyond which the estimate is up to 40 % too low. us, strips -> the other kernels, from the cache and from memory: 504 x 1024 x 7040 28.9 and 31.7 -> 22.0 and
// 23.9, 150 x 1024 x 11008 18.7 and 21.3 -> 16.9 and 18.7, 330 x 1024 x 7040 21.8 and 23.6 -> 21.4 and 22.7; but 260 x 1024 x 8192 18.9 and 21.8 -> 20.5 and 21.9.
constexpr double kSmallMostRounds = 2.0;
constexpr int kWideSteps = 16;  // 128-deep steps of K from which on workgroups have sixteen waves
template <int WAVES, int RB, int CB>
constexpr int small_lds_bytes() {
    const int stage = WAVES * RB * 16 * 17 * 16, sums = WAVES * RB * CB * 16 * 17 * 4;
    return stage > sums ? stage : sums;
}

template <int DT, int G, int WAVES, int RB, int CB>
__global__ __launch_bounds__(64 * WAVES) void skinny_w4a16_small_kernel(const char *a, const char *w, int lda, int m, int n, int k, int tiles_m, int tiles_n, uint32_t group_magic,
                                                                              const uint16_t *scales, const uint16_t *__restrict__ bias, uint16_t *__restrict__ c) {
    using T = W4Traits<DT>;
    constexpr int kTile = RB * 16 * 17;  // a wave's activations of a step, 16-byte pieces: rows of 256 + 16 bytes
    extern __shared__ uint4v_t memory[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = lane >> 4, ls = lane & 15;
    // (a run of the column tiles per XCD, the row tiles of a column tile next to each other)
    const int xcd = int(blockIdx.x & 7), local = int(blockIdx.x >> 3), tile_n = tiles_n * xcd / 8 + local / tiles_m;
    if (tile_n >= tiles_n * (xcd + 1) / 8) return;
    const int m0 = local % tiles_m * (16 * RB), n0 = tile_n * (16 * CB);
    const int steps = k >> 7;
    const int steps_per_wave = (steps + WAVES - 1) / WAVES;
    const int s_begin = wave * steps_per_wave, s_end = min(steps, s_begin + steps_per_wave);
    const int rows = min(m - m0, 16 * RB), col = min(n0 + CB * ls, n - CB);

    float4_t acc[RB][CB];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int t = 0; t < CB; ++t) acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w), 0, k * (n >> 1), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(a) + int64_t(m0) * lda * 2, 0, ((rows - 1) * lda + k) * 2, 0x00020000);
    const int w_off = 8 * kg * (n >> 1) + (col >> 1);
    int a_off[4 * RB];  // 4 rows each
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) a_off[i] = (min(4 * i + kg, rows - 1) * lda + 8 * ls) * 2;
    uint4v_t *const tile = memory + wave * kTile;
    for (int st = s_begin; st < s_end; ++st) {
        uint32_t raw[4][8];
        uint4v_t x[4 * RB];
        uint32_t factor[4 / G][CB / 2];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int row = (st * 128 + 32 * s + j) * (n >> 1);
                raw[s][j] = CB == 4 ? uint32_t(__builtin_amdgcn_raw_buffer_load_b16(rsrc_w, w_off, row, 0)) : uint32_t(__builtin_amdgcn_raw_buffer_load_b8(rsrc_w, w_off, row, 0));
            }
#pragma unroll
        for (int f = 0; f < 4 / G; ++f) {  // the group of the 32 G rows: their number over the group's
            const uint32_t block = uint32_t(st * (4 / G) + f), group = group_magic == 0 ? block : uint32_t((uint64_t(block) * group_magic) >> 32);
            __builtin_memcpy(factor[f], scales + int64_t(group) * n + col, CB * 2);
        }
#pragma unroll
        for (int i = 0; i < 4 * RB; ++i) x[i] = __builtin_bit_cast(uint4v_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, a_off[i], st * 256, 0));
        __builtin_amdgcn_sched_barrier(0);  // all of the step's loads are under way
#pragma unroll
        for (int i = 0; i < 4 * RB; ++i) tile[(4 * i + kg) * 17 + ls] = x[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int f = 0; f < 4 / G; ++f) {
            uint32_t q[G][CB][4];
#pragma unroll
            for (int s = 0; s < G; ++s)
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t lo = raw[f * G + s][2 * p], hi = raw[f * G + s][2 * p + 1];
                    if constexpr (DT == HIDET_QMM_BF16) {
                        // (upper halves and bytes are operand selections of the conversion)
                        const uint32_t u = __builtin_amdgcn_perm(hi, lo, CB == 4 ? 0x05040100u : 0x0c040c00u);
                        uint32_t v = u >> 4;
                        asm("" : "+v"(v));
#pragma unroll
                        for (int t = 0; t < CB; ++t) {
                            typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
                            const uint32_t from = (t & 1 ? v : u) >> (8 * (t >> 1));
                            const bf16x2_t pair = {static_cast<__bf16>(__builtin_amdgcn_cvt_off_f32_i4(int(from))), static_cast<__bf16>(__builtin_amdgcn_cvt_off_f32_i4(int(from >> 16)))};
                            q[s][t][p] = __builtin_bit_cast(uint32_t, pair);
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < CB / 2; ++e) {
                            const uint32_t u = __builtin_amdgcn_perm(hi, lo, 0x0c040c00u + uint32_t(e) * 0x00010001u);
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const half2_t v = __builtin_bit_cast(half2_t, ((u >> (4 * h)) & 0x000F000Fu) ^ T::kMagic) - half2_t{_Float16(T::kBias), _Float16(T::kBias)};
                                q[s][2 * e + h][p] = __builtin_bit_cast(uint32_t, v);
                            }
                        }
                    }
                }
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                uint4 xa[G];
#pragma unroll
                for (int s = 0; s < G; ++s) xa[s] = __builtin_bit_cast(uint4, tile[(16 * r + ls) * 17 + 4 * (f * G + s) + kg]);
#pragma unroll
                for (int t = 0; t < CB; ++t) {
                    float4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < G; ++s) part = T::mfma(xa[s], uint4{q[s][t][0], q[s][t][1], q[s][t][2], q[s][t][3]}, part);
                    const float by = T::to_f32(uint16_t(factor[f][t >> 1] >> (16 * (t & 1)))) * (DT == HIDET_QMM_BF16 ? 16.0f : 1.0f);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[r][t][e] = __builtin_fmaf(part[e], by, acc[r][t][e]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the sums take the place of the activations
    float *red = reinterpret_cast<float *>(memory);  // [wave][RB][CB][16][17]
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int t = 0; t < CB; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[(((wave * RB + r) * CB + t) * 16 + 4 * kg + v) * 17 + ls] = acc[r][t][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (RB * CB * 256 + 64 * WAVES - 1) / (64 * WAVES); ++i) {
        const int at = i * 64 * WAVES + tid, in_row = at % (16 * CB), row = at / (16 * CB), ns = in_row / CB, t = in_row % CB, out = n0 + in_row;
        if (row < rows && out < n) {
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < WAVES; ++p) v += red[(((p * RB + (row >> 4)) * CB + t) * 16 + (row & 15)) * 17 + ns];
            const float add = bias != nullptr ? T::to_f32(bias[out]) : -0.0f;
            c[int64_t(m0 + row) * n + out] = DT == HIDET_QMM_BF16 ? biased_bf16_bits(v, add) : __builtin_bit_cast(uint16_t, scaled_biased_f16(v, 1.0f, add));
        }
    }
}

}  // namespace

bool skinny_w4a16_small_supported(const void *a, const void *scales, int64_t n, int64_t k, int64_t lda, int group) {
    constexpr int64_t kMost = (int64_t(1) << 31) - (1 << 20);
    return k > 0 && k % 128 == 0 && group > 0 && group % 64 == 0 && n % 8 == 0 && lda % 2 == 0 && aligned(a, 4) && aligned(scales, 4) && (k + 128) * n / 2 < kMost && lda * 128 + k * 2 < kMost;
}

// Row blocks and columns per lane of the smallest estimated time: a fit (13 %) to 2132 launches on 478 shapes of 1 to 256 rows, K of 256 to 2048 and N of 256 to 6144, in the mean of
// weights from memory and from the last-level cache. Where it is ahead of the other kernels' estimates by 5 % those calls take 37 % less time in the mean (34 on weights
// from memory) and none takes 3 % more. Beyond, 180 shapes of K 2176 to 4096, weights from the cache (from memory): 17 rows and more 15 to 25 % less time to K = 3328 (10 to 20), 5
// to 9 to 4096 (4 to 6), none 3 % more; up to 16 rows 26 to 38 % less to 2944 (18 to 37), but at 3072 x 2048 and 4096 x 2872 20 % more from memory, hence not there; K = 6144 11 % more (29).
// (796 x 1024 x 3776, outside the fit, 23 us and 29 here: no more than 512 rows.)
// The smallest strips (one row block, two columns per lane) of at most one workgroup per CU take sixteen waves where each then has a step: 3 to 7 % off at K = 2048 and 2 to 7 at 3072
// (weights from memory: 2), but 1 % more at 1536, 5 at 1024, 16 to 26 where a CU gets two workgroups (of eight waves it holds them at once) and 2 to 5 on larger strips.
SkinnyW4SmallPlan skinny_w4a16_small_plan(const void *a, const void *scales, int64_t m, int64_t n, int64_t k, int64_t lda, int group) {
    SkinnyW4SmallPlan best;
    if (m > kSmallMostRows || k > (m <= 16 ? kFewRowsMostK : kSmallMostK) || k * n / 2 > kSmallMostBytes || !skinny_w4a16_small_supported(a, scales, n, k, lda, group)) return best;
    const double cus = std::max(1, device_cus()), steps = double(cdiv(k / 128, 8));  // steps of a wave, of eight
    for (int most = 1; most <= 4; ++most) {
        const int64_t tiles_m = cdiv(m, 16 * most);
        const int rb = int(cdiv(cdiv(m, tiles_m), 16));
        for (int cb = 2; cb <= 4; cb += 2) {
            // (of the XCD with the most column tiles, times eight)
            const double groups = double(tiles_m) * double(8 * cdiv(cdiv(n, 16 * cb), 8)), share = std::max(1.0, groups / cus), rounds = std::ceil(share);
            if (rounds > kSmallMostRounds) continue;
            const int waves = rb == 1 && cb == 2 && groups <= cus && k >= 128 * kWideSteps ? 16 : 8;
            const double us = (waves == 16 ? 0.95 : 1.0) * (1.915 + 0.0134 * share * rb * cb + rounds * steps * (0.545 + 0.342 * rb + 0.154 * cb + 0.114 * rb * cb));
            if (us < best.us) best = SkinnyW4SmallPlan{us, rb, cb, waves};
        }
    }
    return best;
}

void skinny_w4a16_small_launch(const SkinnyW4SmallPlan &plan, const void *a, const void *w, const void *scales, const void *bias, void *c, int64_t m, int64_t k, int64_t n, int64_t lda,
                               int group, int dtype, hipStream_t stream) {
    using std::integral_constant;
    const int64_t tiles_m = cdiv(m, 16 * plan.rb), tiles_n = cdiv(n, 16 * plan.cb), grid = tiles_m * cdiv(tiles_n, 8) * 8;
    QMM_CHECK(grid < (int64_t(1) << 31), "problem too large for one launch");
    const int fold = group % 128 == 0 ? 4 : 2;
    const uint32_t magic = uint32_t(((uint64_t(1) << 32) + uint32_t(group / (32 * fold)) - 1) / uint32_t(group / (32 * fold)));  // (0 for a divisor of 1)
    auto go = [&](auto kern, int lds) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
        launch(kern, dim3(uint32_t(grid)), dim3(uint32_t(64 * plan.waves)), size_t(lds), stream, static_cast<const char *>(a), static_cast<const char *>(w), int(lda), int(m), int(n), int(k),
               int(tiles_m), int(tiles_n), magic, static_cast<const uint16_t *>(scales), static_cast<const uint16_t *>(bias), static_cast<uint16_t *>(c));
    };
    auto of = [&](auto rb, auto cb) {
        constexpr int RB = decltype(rb)::value, CB = decltype(cb)::value;
        auto by = [&](auto waves) {
            constexpr int W = decltype(waves)::value, kLds = small_lds_bytes<W, RB, CB>();
            if (dtype == HIDET_QMM_BF16) fold == 4 ? go(skinny_w4a16_small_kernel<HIDET_QMM_BF16, 4, W, RB, CB>, kLds) : go(skinny_w4a16_small_kernel<HIDET_QMM_BF16, 2, W, RB, CB>, kLds);
            else fold == 4 ? go(skinny_w4a16_small_kernel<HIDET_QMM_F16, 4, W, RB, CB>, kLds) : go(skinny_w4a16_small_kernel<HIDET_QMM_F16, 2, W, RB, CB>, kLds);
        };
        if constexpr (RB == 1 && CB == 2) {
            if (plan.waves == 16) return by(integral_constant<int, 16>());
        }
        by(integral_constant<int, 8>());
    };
    auto rows = [&](auto cb) {
        if (plan.rb == 1) of(integral_constant<int, 1>(), cb);
        else if (plan.rb == 2) of(integral_constant<int, 2>(), cb);
        else if (plan.rb == 3) of(integral_constant<int, 3>(), cb);
        else of(integral_constant<int, 4>(), cb);
    };
    if (plan.cb == 2) rows(integral_constant<int, 2>());
    else rows(integral_constant<int, 4>());
}

}  // namespace qmm
