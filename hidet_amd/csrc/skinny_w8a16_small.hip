// W8A16 on small row-major weights: c[m, n] = (sum_k a[m, k] * w[k, n]) * scale[n] (+ bias[n]), a workgroup per 16 RB rows and 16 CB columns (CB = 2 or 4) for all of K.
//
// The bandwidth-bound kernel and the narrow tiles (gemm_mid.h) read rows of 256 and 128 columns and therefore cut K between workgroups, whose exchange and rings take 5 us of
// the 7 that a weight of 2 MB does. Here eight independent waves cut K and meet once, in LDS. What bounds it is what a CU gets from the L2, about 60 KB per us: few
// workgroups, each with its strip of the weight and all of its rows' activations.
//
// Per step of 128 k a lane (kg, ls) reads CB bytes of rows 32 s + 8 kg + j (s = 0 .. 3, j = 0 .. 7) at columns CB ls and on, whatever their alignment: 16 lanes
// read 64 or 32 bytes of a row. Byte permutations make the operands of v_mfma_f32_16x16x32_f16 of them, column ls of fragment t being column CB ls + t; codes are
// widened exactly, to q / 512 (a byte q ^ 0x80 as a subnormal number, times 2^15 less 0.25). Activations go through an LDS tile of the wave's own; one wave's LDS operations
// execute in order. us, before -> here, weights from the last-level cache: 1 x 1024 x 4096 6.9 -> 3.9, 8 x 1024 x 3072 6.8 -> 4.0, 16 x 256 x 4096 5.6 -> 3.0, 32 x 1024 x 3072 7.0 ->
// 4.2, 64 x 1536 x 1024 7.2 -> 4.3, 128 x 512 x 512 5.5 -> 3.2. The last columns of a row that is no multiple of CB are moved back into it: two lanes then store the same results.
#include "common.h"
#include "skinny_w8a16_small.h"

#include <cmath>

namespace qmm {
namespace {

constexpr int kSmallWaves = 8;
constexpr int64_t kSmallMostRows = 512, kSmallLeastK = 32, kSmallMostK = 2560, kSmallMostBytes = 8500000;
template <int RB, int CB>
constexpr int small_lds_bytes() {
    const int stage = kSmallWaves * RB * 16 * 17 * 16, sums = kSmallWaves * RB * CB * 16 * 17 * 4;
    return stage > sums ? stage : sums;
}

// TAIL: K is no multiple of 128 (but even).
template <bool TAIL, int RB, int CB>
__global__ __launch_bounds__(64 * kSmallWaves) void skinny_w8a16_small_kernel(const _Float16 *a, const char *w, int lda, int m, int n, int k, int tiles_m, int tiles_n,
                                                                              const _Float16 *__restrict__ scale, const _Float16 *__restrict__ bias, _Float16 *__restrict__ c) {
    constexpr int kTile = RB * 16 * 17;  // a wave's activations of a step, 16-byte pieces: rows of 256 + 16 bytes
    constexpr uint32_t kOutside = 0x7FFFFFF0u;
    extern __shared__ uint4v_t memory[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = lane >> 4, ls = lane & 15;
    // An XCD has a run of the column tiles: several of them share a cache line of the weight (dealt out one by one, every XCD pulls in twice or four times its
    // share: 16 x 3072 x 2048 9.4 us), and the row tiles of a column tile, next to each other, read the same weights.
    const int xcd = int(blockIdx.x & 7), local = int(blockIdx.x >> 3), tile_n = tiles_n * xcd / 8 + local / tiles_m;
    if (tile_n >= tiles_n * (xcd + 1) / 8) return;
    const int m0 = local % tiles_m * (16 * RB), n0 = tile_n * (16 * CB);
    const int steps = (k + 127) >> 7;
    const int steps_per_wave = (steps + kSmallWaves - 1) / kSmallWaves;
    const int s_begin = wave * steps_per_wave, s_end = min(steps, s_begin + steps_per_wave);
    const int rows = min(m - m0, 16 * RB), col = min(n0 + CB * ls, n - CB);

    float4_t acc[RB][CB];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int t = 0; t < CB; ++t) acc[r][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w), 0, k * n, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(a) + int64_t(m0) * lda, 0, ((rows - 1) * lda + k) * 2, 0x00020000);
    const int w_off = 8 * kg * n + col;
    int a_off[4 * RB];  // 4 rows each
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) a_off[i] = (min(4 * i + kg, rows - 1) * lda + 8 * ls) * 2;
    auto load_codes = [&](int voff, int soff) -> uint32_t {
        if constexpr (CB == 4) return __builtin_amdgcn_raw_buffer_load_b32(rsrc_w, voff, soff, 0);
        else return __builtin_amdgcn_raw_buffer_load_b16(rsrc_w, voff, soff, 0);
    };
    uint4v_t *const tile = memory + wave * kTile;
    for (int st = s_begin; st < s_end; ++st) {
        uint32_t raw[4][8];
        uint4v_t x[4 * RB];
        const int left = k - st * 128;
        if (!TAIL || left >= 128) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < 8; ++j) raw[s][j] = load_codes(w_off, (st * 128 + 32 * s + j) * n);
#pragma unroll
            for (int i = 0; i < 4 * RB; ++i) x[i] = __builtin_bit_cast(uint4v_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, a_off[i], st * 256, 0));
        } else {  // the step that K ends in (the whole offset in the register that is range-checked)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < 8; ++j) raw[s][j] = load_codes(32 * s + 8 * kg + j < left ? w_off + (st * 128 + 32 * s + j) * n : int(kOutside), 0);
#pragma unroll
            for (int i = 0; i < 4 * RB; ++i) {
                x[i] = __builtin_bit_cast(uint4v_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, a_off[i] + st * 256, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][e] = 8 * ls + 2 * e < left ? x[i][e] : 0u;  // (the next row's values; K is even)
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // all of the step's loads are under way
#pragma unroll
        for (int i = 0; i < 4 * RB; ++i) tile[(4 * i + kg) * 17 + ls] = x[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            half8_t q[CB];
#pragma unroll
            for (int j = 0; j < 8; ++j) raw[s][j] ^= 0x80808080u;
#pragma unroll
            for (int t = 0; t < CB; ++t)
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t u = __builtin_amdgcn_perm(raw[s][2 * p + 1], raw[s][2 * p], 0x0c000c00u | uint32_t((4 + t) << 16 | t));
                    const half2_t v = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, u), half2_t{_Float16(32768.0f), _Float16(32768.0f)}, half2_t{_Float16(-0.25f), _Float16(-0.25f)});
                    q[t][2 * p] = v[0];
                    q[t][2 * p + 1] = v[1];
                }
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const half8_t xa = __builtin_bit_cast(half8_t, tile[(16 * r + ls) * 17 + 4 * s + kg]);
#pragma unroll
                for (int t = 0; t < CB; ++t) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa, q[t], acc[r][t], 0, 0, 0);
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
    for (int i = 0; i < (RB * CB + 1) / 2; ++i) {
        const int at = i * 512 + tid, in_row = at % (16 * CB), row = at / (16 * CB), ns = in_row / CB, t = in_row % CB;
        if (row < rows && n0 + CB * ns < n) {
            const int out = min(n0 + CB * ns, n - CB) + t;
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < kSmallWaves; ++p) v += red[(((p * RB + (row >> 4)) * CB + t) * 16 + (row & 15)) * 17 + ns];
            c[int64_t(m0 + row) * n + out] = scaled_biased_f16(v * 512.0f, float(scale[out]), bias != nullptr ? float(bias[out]) : -0.0f);
        }
    }
}

}  // namespace

bool skinny_w8a16_small_supported(const void *a, int64_t n, int64_t k, int64_t lda) {
    constexpr int64_t kMost = (int64_t(1) << 31) - (1 << 20);
    return k > 0 && k % 2 == 0 && n >= 4 && lda % 2 == 0 && aligned(a, 4) && (k + 128) * n < kMost && lda * 128 + k * 2 < kMost;
}

// Row blocks and columns per lane of the smallest estimated time: a fit (14 %) to 2040 launches on 456 shapes of 1 to 256 rows, K of 256 to 2048 and N of 256 to 6144, in the mean of
// weights from memory and from the last-level cache. Weights of more than 8.5 MB or 2560 rows stay with the others: there the strips of rows that a workgroup reads of a weight
// in memory cost more than the exchange that they save (1 x 2048 x 6144 8.2 us and 11.2 here, 16 x 3072 x 1024 7.1 and 8.5, 16 x 3072 x 3072 9.0 and 13.3; 64 x 3072 x 2260 27 % more, 16 x 2772
// x 2572 18; K of 2601 to 2944 4 to 12 % less time from the cache and the same from memory). K of 1900 to 2600, 64 shapes: 14 to 27 % less time, 7 to 17 % from memory, there six of 64 more than 3 %
// slower (4 to 7 %; of 500 other shapes 71 x 2496 x 2048 9.5 us and 11.6 here, from the cache 9.0 and 6.4).
// Within K = 2048, where this is ahead of the other kernels' estimates by 8 %, those 456 calls take 36 % less time in the mean (30 on weights from memory), and one of them in the former case and two in the latter take 3 to 4 % more.
SkinnySmallPlan skinny_w8a16_small_plan(const void *a, int64_t m, int64_t n, int64_t k, int64_t lda) {
    SkinnySmallPlan best;
    if (m > kSmallMostRows || k < kSmallLeastK || k > kSmallMostK || k * n > kSmallMostBytes || !skinny_w8a16_small_supported(a, n, k, lda)) return best;
    const double cus = std::max(1, device_cus()), steps = double(cdiv(cdiv(k, 128), kSmallWaves));  // steps of a wave
    for (int most = 1; most <= 4; ++most) {
        const int64_t tiles_m = cdiv(m, 16 * most);
        const int rb = int(cdiv(cdiv(m, tiles_m), 16));
        for (int cb = 2; cb <= 4; cb += 2) {
            // (of the XCD with the most column tiles, times eight)
            const double groups = double(tiles_m) * double(8 * cdiv(cdiv(n, 16 * cb), 8)), share = std::max(1.0, groups / cus), rounds = std::ceil(share);
            const double us = 1.755 + 0.0585 * share * rb * cb + rounds * steps * (0.814 + 0.306 * rb + 0.0755 * cb + 0.082 * rb * cb);
            if (us < best.us) best = SkinnySmallPlan{us, rb, cb};
        }
    }
    return best;
}

void skinny_w8a16_small_launch(const SkinnySmallPlan &plan, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                               int64_t lda, hipStream_t stream) {
    const int64_t tiles_m = cdiv(m, 16 * plan.rb), tiles_n = cdiv(n, 16 * plan.cb), grid = tiles_m * cdiv(tiles_n, 8) * 8;
    QMM_CHECK(grid < (int64_t(1) << 31), "problem too large for one launch");
    auto go = [&](auto kern, int lds) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
        launch(kern, dim3(uint32_t(grid)), dim3(64 * kSmallWaves), size_t(lds), stream, static_cast<const _Float16 *>(a), static_cast<const char *>(w), int(lda), int(m), int(n), int(k),
               int(tiles_m), int(tiles_n), static_cast<const _Float16 *>(scale), static_cast<const _Float16 *>(bias), static_cast<_Float16 *>(c));
    };
    auto of = [&](auto rb, auto cb) {
        constexpr int RB = decltype(rb)::value, CB = decltype(cb)::value;
        if (k % 128 == 0) go(skinny_w8a16_small_kernel<false, RB, CB>, small_lds_bytes<RB, CB>());
        else go(skinny_w8a16_small_kernel<true, RB, CB>, small_lds_bytes<RB, CB>());
    };
    auto rows = [&](auto cb) {
        using std::integral_constant;
        if (plan.rb == 1) of(integral_constant<int, 1>(), cb);
        else if (plan.rb == 2) of(integral_constant<int, 2>(), cb);
        else if (plan.rb == 3) of(integral_constant<int, 3>(), cb);
        else of(integral_constant<int, 4>(), cb);
    };
    if (plan.cb == 2) rows(std::integral_constant<int, 2>());
    else rows(std::integral_constant<int, 4>());
}

}  // namespace qmm
