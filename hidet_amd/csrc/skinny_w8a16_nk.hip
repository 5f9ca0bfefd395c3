// W8A16 decode GEMV / skinny GEMM for weights stored K-contiguous: w is the [K, N] operand of the operator held as
// [N, K] in memory (row n = the K codes of output column n, stride ldw) - the layout of torch's nn.Linear weight, or
// of a [K, N] tensor with strides (1, ldw).  c[m, n] = (sum_k a[m, k] * w[n, k]) * scale[n], fp32 accumulation, M <= 16
// rows per pass.
//
// The reduction runs along the contiguous axis, so nothing has to be exchanged between workgroups: a workgroup owns 16
// output columns, its 4 or 8 waves split K and meet in LDS, N / 16 workgroups stream the weights exactly once.  Lane
// (kg, ls) of a wave reads 32 consecutive bytes of row n0 + ls at k = kbase + 32 kg per 128-deep step (the 16 lanes x 4
// k-groups of a step cover 16 rows x 128 contiguous bytes).  Bytes 8j .. 8j+7 of those 32 are, for j = 0 .. 3, the B
// operand of one v_mfma_f32_16x16x32_f16: the k positions an MFMA sums over may be any 32 as long as both operands
// agree, so MFMA j takes k = kbase + 32 kg + 8 j + (0 .. 7) from lane group kg, and the activation fragment is loaded
// from exactly those positions.  Two bytes become two float16 values with v_perm_b32 (spread) and v_xor_b32 (0x6400 |
// (q ^ 0x80) == 1152 + q): one VALU op per weight; the constant is removed at the end with 1152 * sum_k a[m, k], which
// one more MFMA per fragment (against ones) accumulates on the otherwise idle matrix pipe - exact in fp32 for the
// few thousand terms of a wave's K range.  With K a multiple of 128 (FULL) the loop has no conditions at all: lanes
// of rows >= M and columns >= N read a clamped row and their results are dropped at the end.  Each step of that loop
// sits behind a wave-uniform break, and the compiler moves the step's loads down into its block: a wave has one step in
// flight at a time and the 8 to 11 waves per CU hide the latency (the FP8 kernel of the same shape was measured a third
// slower with all of a trip's loads really issued up front).
#include "common.h"
#include "skinny_w8a16_nk_tall.h"

#include <cmath>

namespace qmm {
namespace {

template <bool ALIGNED_A, bool FULL, int WAVES, bool STAGE = false>
__global__ __launch_bounds__(64 * WAVES) void skinny_w8a16_nk_kernel(const _Float16 *__restrict__ a, int64_t lda,
                                                              const int8_t *__restrict__ w, int64_t ldw,
                                                              const _Float16 *__restrict__ scale, const _Float16 *__restrict__ bias,
                                                              _Float16 *__restrict__ c, int m, int k, int n) {
    __shared__ float red[WAVES][16][17];
    constexpr int kNkDepth = FULL ? 8 : 4;  // 128-deep steps per trip of the outer loop
    static_assert(FULL || !ALIGNED_A, "aligned activations with a K off the steps go to the tall kernel");
    // STAGE (FULL with aligned activations, more than two rows): a wave fetches its 16 x 128 activation block of a step
    // with four fully coalesced loads (4 rows x 256 bytes each) and turns it into MFMA fragments through a private LDS
    // tile of 16 rows x (256 + 16) bytes, two slots.  Fetching the fragments straight from memory touches every cache
    // line of the block four times, and made 16 rows cost 8 us more than one; with one or two rows the direct fetch
    // is a broadcast and a little faster.  No barrier: the LDS operations of one wave execute in order.
    static_assert(!STAGE || (FULL && ALIGNED_A), "staging needs the condition-free loop and 16-byte loads");
    constexpr bool kStage = STAGE;
    __shared__ uint4 stage[kStage ? WAVES : 1][2][16 * 17];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int kg = lane >> 4, ls = lane & 15;
    const int n0 = blockIdx.x * 16;
    const bool n_ok = n0 + ls < n;
    const bool m_ok = ls < m;

    // K is cut into 128-deep steps dealt to the waves in contiguous runs
    const int steps = (k + 127) >> 7;
    const int steps_per_wave = (steps + WAVES - 1) / WAVES;
    const int s_begin = wave * steps_per_wave, s_end = min(steps, s_begin + steps_per_wave);

    float4_t acc = {0.f, 0.f, 0.f, 0.f}, xsum = {0.f, 0.f, 0.f, 0.f};
    half8_t ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = _Float16(1.0f);
    // FULL: rows past the end are clamped to the last one instead of being masked in the loop
    const int8_t *wp = w + int64_t(FULL ? min(n0 + ls, n - 1) : n0 + ls) * ldw + 32 * kg;
    const _Float16 *ap = a + int64_t(FULL ? min(ls, m - 1) : ls) * lda + 32 * kg;

    for (int s0 = s_begin; s0 < s_end; s0 += kNkDepth) {
        uint4 wv[kNkDepth][2];
        half8_t xa[kNkDepth][4];
        uint4 ax[kStage ? kNkDepth : 1][4];
#pragma unroll
        for (int d = 0; d < kNkDepth; ++d) {
            if (FULL) {
                const int st = min(s0 + d, s_end - 1);  // a step past the wave's range re-reads its last one; not used
                wv[d][0] = *reinterpret_cast<const uint4 *>(wp + int64_t(st) * 128);
                wv[d][1] = *reinterpret_cast<const uint4 *>(wp + int64_t(st) * 128 + 16);
            } else {
                const int kb = (s0 + d) * 128 + 32 * kg;
                wv[d][0] = wv[d][1] = uint4{0u, 0u, 0u, 0u};
                if (n_ok && s0 + d < s_end) {  // K % 16 == 0: a 16-byte piece is inside K or outside as a whole
                    if (kb < k) wv[d][0] = *reinterpret_cast<const uint4 *>(wp + int64_t(s0 + d) * 128);
                    if (kb + 16 < k) wv[d][1] = *reinterpret_cast<const uint4 *>(wp + int64_t(s0 + d) * 128 + 16);
                }
            }
        }
#pragma unroll
        for (int d = 0; d < kNkDepth; ++d) {
            const int kb = (s0 + d) * 128 + 32 * kg;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (FULL) {
                    const int st = min(s0 + d, s_end - 1);
                    if (kStage) {  // load j: rows 4j .. 4j+3, 16 lanes x 16 bytes per row
                        const int r = min(4 * j + kg, m - 1);
                        ax[d][j] = *reinterpret_cast<const uint4 *>(a + int64_t(r) * lda + int64_t(st) * 128 + 8 * ls);
                    } else if (ALIGNED_A) {
                        xa[d][j] = *reinterpret_cast<const half8_t *>(ap + int64_t(st) * 128 + 8 * j);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e) xa[d][j][e] = ap[int64_t(st) * 128 + 8 * j + e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) xa[d][j][e] = _Float16(0.0f);
                    if (m_ok && s0 + d < s_end && kb + 8 * j < k) {  // K % 8 == 0 on this path
#pragma unroll
                        for (int e = 0; e < 8; ++e) xa[d][j][e] = ap[int64_t(s0 + d) * 128 + 8 * j + e];
                    }
                }
            }
        }
#pragma unroll
        for (int d = 0; d < kNkDepth; ++d) {
            if (FULL && s0 + d >= s_end) break;  // wave-uniform
            if (kStage) {
                uint4 *tile = stage[wave][d & 1];
#pragma unroll
                for (int j = 0; j < 4; ++j) tile[(4 * j + kg) * 17 + ls] = ax[d][j];
#pragma unroll
                for (int j = 0; j < 4; ++j) xa[d][j] = __builtin_bit_cast(half8_t, tile[ls * 17 + 4 * kg + j]);
            }
            const uint32_t raw[8] = {wv[d][0].x, wv[d][0].y, wv[d][0].z, wv[d][0].w, wv[d][1].x, wv[d][1].y, wv[d][1].z, wv[d][1].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // bytes 8j .. 8j+7 = dwords 2j, 2j+1; selectors spread bytes (0, 1) and (2, 3) of a dword into two halves
                constexpr uint32_t kLo = 0x0c010c00u, kHi = 0x0c030c02u;
                union {
                    uint32_t u[4];
                    half8_t h8;
                } b;
                b.u[0] = __builtin_amdgcn_perm(raw[2 * j], raw[2 * j], kLo) ^ 0x64806480u;
                b.u[1] = __builtin_amdgcn_perm(raw[2 * j], raw[2 * j], kHi) ^ 0x64806480u;
                b.u[2] = __builtin_amdgcn_perm(raw[2 * j + 1], raw[2 * j + 1], kLo) ^ 0x64806480u;
                b.u[3] = __builtin_amdgcn_perm(raw[2 * j + 1], raw[2 * j + 1], kHi) ^ 0x64806480u;
                // rows = activation rows, columns = weight rows (output columns); the weights carry + 1152 each
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[d][j], b.h8, acc, 0, 0, 0);
                xsum = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[d][j], ones, xsum, 0, 0, 0);
            }
        }
    }
    // acc[v] = partial c[4 kg + v][n0 + ls]; zero weights of masked lanes also carried + 1152, which xsum removes as well
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][4 * kg + v][ls] = acc[v] - 1152.0f * xsum[v];
    __syncthreads();
    const int row = tid >> 4, cn = tid & 15;
    if (row < m && n0 + cn < n) {  // row < 16 <= the first four waves
        float v = 0.f;
#pragma unroll
        for (int p = 0; p < WAVES; ++p) v += red[p][row][cn];
        c[int64_t(row) * n + n0 + cn] = scaled_biased_f16(v, float(scale[n0 + cn]), bias != nullptr ? float(bias[n0 + cn]) : -0.0f);
    }
}

// More than a few activation rows: the kernel above re-reads the activation rows once per 16 output columns, which at 16
// rows is twice the weight bytes.  Here a wave keeps one activation fragment for CG column groups (16 CG columns per
// workgroup), so that traffic drops by CG; the workgroup's waves split K as before.  K a multiple of 128, aligned
// activations; the loop has no conditions (clamped rows, see above).
template <int CG, int WAVES, int DEPTH>
__global__ __launch_bounds__(64 * WAVES) void skinny_w8a16_nk_wide_kernel(const _Float16 *__restrict__ a, int64_t lda,
                                                                          const int8_t *__restrict__ w, int64_t ldw,
                                                                          const _Float16 *__restrict__ scale,
                                                                          const _Float16 *__restrict__ bias,
                                                                          _Float16 *__restrict__ c, int m, int k, int n) {
    __shared__ float red[WAVES][CG][16][17];
    __shared__ uint4 stage[WAVES][2][16 * 17];  // per wave: activation block of a step, see the kernel above
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int kg = lane >> 4, ls = lane & 15;
    const int n0 = blockIdx.x * (16 * CG);

    const int steps = k >> 7;
    const int steps_per_wave = (steps + WAVES - 1) / WAVES;
    const int s_begin = wave * steps_per_wave, s_end = min(steps, s_begin + steps_per_wave);

    float4_t acc[CG], xsum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < CG; ++g) acc[g] = float4_t{0.f, 0.f, 0.f, 0.f};
    half8_t ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = _Float16(1.0f);
    const int8_t *wp[CG];
#pragma unroll
    for (int g = 0; g < CG; ++g) wp[g] = w + int64_t(min(n0 + 16 * g + ls, n - 1)) * ldw + 32 * kg;

    for (int s0 = s_begin; s0 < s_end; s0 += DEPTH) {
        uint4 wv[DEPTH][CG][2];
        half8_t xa[DEPTH][4];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int st = min(s0 + d, s_end - 1);  // a step past the wave's range re-reads its last one; not used
#pragma unroll
            for (int g = 0; g < CG; ++g) {
                wv[d][g][0] = *reinterpret_cast<const uint4 *>(wp[g] + int64_t(st) * 128);
                wv[d][g][1] = *reinterpret_cast<const uint4 *>(wp[g] + int64_t(st) * 128 + 16);
            }
        }
        uint4 ax[DEPTH][4];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int st = min(s0 + d, s_end - 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = min(4 * j + kg, m - 1);
                ax[d][j] = *reinterpret_cast<const uint4 *>(a + int64_t(r) * lda + int64_t(st) * 128 + 8 * ls);
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            if (s0 + d >= s_end) break;  // wave-uniform
            uint4 *tile = stage[wave][d & 1];
#pragma unroll
            for (int j = 0; j < 4; ++j) tile[(4 * j + kg) * 17 + ls] = ax[d][j];
#pragma unroll
            for (int j = 0; j < 4; ++j) xa[d][j] = __builtin_bit_cast(half8_t, tile[ls * 17 + 4 * kg + j]);
#pragma unroll
            for (int g = 0; g < CG; ++g) {
                const uint32_t raw[8] = {wv[d][g][0].x, wv[d][g][0].y, wv[d][g][0].z, wv[d][g][0].w,
                                         wv[d][g][1].x, wv[d][g][1].y, wv[d][g][1].z, wv[d][g][1].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    constexpr uint32_t kLo = 0x0c010c00u, kHi = 0x0c030c02u;
                    union {
                        uint32_t u[4];
                        half8_t h8;
                    } b;
                    b.u[0] = __builtin_amdgcn_perm(raw[2 * j], raw[2 * j], kLo) ^ 0x64806480u;
                    b.u[1] = __builtin_amdgcn_perm(raw[2 * j], raw[2 * j], kHi) ^ 0x64806480u;
                    b.u[2] = __builtin_amdgcn_perm(raw[2 * j + 1], raw[2 * j + 1], kLo) ^ 0x64806480u;
                    b.u[3] = __builtin_amdgcn_perm(raw[2 * j + 1], raw[2 * j + 1], kHi) ^ 0x64806480u;
                    acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[d][j], b.h8, acc[g], 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) xsum = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[d][j], ones, xsum, 0, 0, 0);
        }
    }
#pragma unroll
    for (int g = 0; g < CG; ++g)
#pragma unroll
        for (int v = 0; v < 4; ++v) red[wave][g][4 * kg + v][ls] = acc[g][v] - 1152.0f * xsum[v];
    __syncthreads();
    for (int o = tid; o < CG * 256; o += 64 * WAVES) {
        const int g = o >> 8, row = (o >> 4) & 15, cn = o & 15;
        const int col = n0 + 16 * g + cn;
        if (row < m && col < n) {
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < WAVES; ++p) v += red[p][g][row][cn];
            c[int64_t(row) * n + col] = scaled_biased_f16(v, float(scale[col]), bias != nullptr ? float(bias[col]) : -0.0f);
        }
    }
}

// 17 rows and more of small weights, or any number where K is no multiple of 128, aligned activations: 16 RB rows x 16 CG columns per workgroup, eight waves that split K and meet once, in LDS. The narrow tiles (gemm_mid.h)
// take 7 us for what this reads in 1 to 2: no ring, no barrier before the end, no exchange. What bounds it is what a CU gets from the L2 (every workgroup reads its rows' activations
// for 16 or 32 columns only), so wide and deep matrices stay with the narrow tiles. A wave has one step in flight, its activations turned into fragments through
// an LDS tile of its own as above; codes are widened exactly, to q / 512 (a byte q ^ 0x80 as a subnormal number, times 2^15 less 0.25), once for all rows.
// us, narrow tiles -> here, weights from the last-level cache: 17 x 1024 x 1024 6.9 -> 3.0, 32 x 2048 x 1024 7.7 -> 3.6, 32 x 4096 x 4096 10.2 -> 7.5, 48 x 1536 x 3072 8.3 -> 4.8, 64 x
// 2048 x 2048 8.0 -> 4.5, 64 x 3072 x 4096 11.3 -> 8.0. TAIL: K is no multiple of 128 (but of 16).
constexpr int kTallWaves = 8;
template <int RB, int CG>
constexpr int tall_lds_bytes() {
    const int stage = kTallWaves * RB * 16 * 17 * 16, sums = kTallWaves * RB * CG * 16 * 17 * 4;
    return stage > sums ? stage : sums;
}
template <bool TAIL, int RB, int CG>
__global__ __launch_bounds__(64 * kTallWaves) void skinny_w8a16_nk_tall_kernel(const _Float16 *a, const int8_t *w, int64_t lda, int64_t ldw, int m, int n, int k, int tiles_m,
                                                                               int tiles_n, const _Float16 *__restrict__ scale, const _Float16 *__restrict__ bias,
                                                                               _Float16 *__restrict__ c) {
    constexpr int kTile = RB * 16 * 17;  // a wave's activations of a step, 16-byte pieces: rows of 256 + 16 bytes
    extern __shared__ uint4v_t memory[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = lane >> 4, ls = lane & 15;
    // the row tiles of a column tile are neighbours on one XCD: they read the same weights
    const int local = int(blockIdx.x >> 3), tile_n = local / tiles_m * 8 + int(blockIdx.x & 7), m0 = local % tiles_m * (16 * RB), n0 = tile_n * (16 * CG);
    if (tile_n >= tiles_n) return;
    const int steps = (k + 127) >> 7;
    const int steps_per_wave = (steps + kTallWaves - 1) / kTallWaves;
    const int s_begin = wave * steps_per_wave, s_end = min(steps, s_begin + steps_per_wave);

    float4_t acc[RB][CG];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < CG; ++g) acc[r][g] = float4_t{0.f, 0.f, 0.f, 0.f};
    const int8_t *wp[CG];
    const _Float16 *ap[4 * RB];
#pragma unroll
    for (int g = 0; g < CG; ++g) wp[g] = w + int64_t(min(n0 + 16 * g + ls, n - 1)) * ldw + 32 * kg;
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) ap[i] = a + int64_t(min(m0 + 4 * i + kg, m - 1)) * lda + 8 * ls;  // 4 rows each
    uint4v_t *const tile = memory + wave * kTile;
    for (int st = s_begin; st < s_end; ++st) {
        uint4v_t raw[CG][2], x[4 * RB];
        const int left = k - st * 128;
        if (!TAIL || left >= 128) {
#pragma unroll
            for (int g = 0; g < CG; ++g) {
                raw[g][0] = *reinterpret_cast<const uint4v_t *>(wp[g] + int64_t(st) * 128);
                raw[g][1] = *reinterpret_cast<const uint4v_t *>(wp[g] + int64_t(st) * 128 + 16);
            }
#pragma unroll
            for (int i = 0; i < 4 * RB; ++i) x[i] = *reinterpret_cast<const uint4v_t *>(ap[i] + int64_t(st) * 128);
        } else {  // the step that K ends in: activations past it are zeros, whatever the codes
#pragma unroll
            for (int g = 0; g < CG; ++g)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    raw[g][h] = uint4v_t{0, 0, 0, 0};
                    if (32 * kg + 16 * h < left) raw[g][h] = *reinterpret_cast<const uint4v_t *>(wp[g] + int64_t(st) * 128 + 16 * h);
                }
#pragma unroll
            for (int i = 0; i < 4 * RB; ++i) {
                x[i] = uint4v_t{0, 0, 0, 0};
                if (8 * ls < left) x[i] = *reinterpret_cast<const uint4v_t *>(ap[i] + int64_t(st) * 128);
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // all of the step's loads are under way
#pragma unroll
        for (int i = 0; i < 4 * RB; ++i) tile[(4 * i + kg) * 17 + ls] = x[i];
        __builtin_amdgcn_wave_barrier();
        half8_t q[CG][4];
#pragma unroll
        for (int g = 0; g < CG; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t u[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t src = raw[g][j >> 1][2 * (j & 1) + (p >> 1)] ^ 0x80808080u;
                    u[p] = __builtin_amdgcn_perm(src, src, (p & 1) ? 0x0c030c02u : 0x0c010c00u);
                    const half2_t v = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, u[p]), half2_t{_Float16(32768.0f), _Float16(32768.0f)}, half2_t{_Float16(-0.25f), _Float16(-0.25f)});
                    q[g][j][2 * p] = v[0];
                    q[g][j][2 * p + 1] = v[1];
                }
            }
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const half8_t xa = __builtin_bit_cast(half8_t, tile[(16 * r + ls) * 17 + 4 * kg + j]);
#pragma unroll
                for (int g = 0; g < CG; ++g) acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa, q[g][j], acc[r][g], 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // the sums take the place of the activations
    float *red = reinterpret_cast<float *>(memory);  // [wave][RB][CG][16][17]
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < CG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[(((wave * RB + r) * CG + g) * 16 + 4 * kg + v) * 17 + ls] = acc[r][g][v];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (RB * CG + 1) / 2; ++i) {
        const int at = i * 512 + tid, cn = at & 15, row = (at >> 4) % (16 * RB), g = at / (256 * RB);
        const int col = n0 + 16 * g + cn;
        if (g < CG && m0 + row < m && col < n) {
            float v = 0.f;
#pragma unroll
            for (int p = 0; p < kTallWaves; ++p) v += red[(((p * RB + (row >> 4)) * CG + g) * 16 + (row & 15)) * 17 + cn];
            c[int64_t(m0 + row) * n + col] = scaled_biased_f16(v * 512.0f, float(scale[col]), bias != nullptr ? float(bias[col]) : -0.0f);
        }
    }
}

}  // namespace

// Row blocks and column groups per workgroup of the smallest estimated time: a fit (9 %) to 2224 launches on 390 shapes of 17 to 64 rows, K and N of 1024 to 11008, in the mean of
// weights from memory and from the last-level cache. The caller takes this kernel where it is ahead of the narrow tiles' estimate, which is about 17 % too high, by 20 %: of those
// shapes 1 to 2 % over the faster kernel in the mean, and none more than 3 % slower than on the tiles alone at 25 %, eight of 780 at 15.
SkinnyNkTallPlan skinny_w8a16_nk_tall_plan(const void *a, int64_t m, int64_t n, int64_t k, int64_t lda) {
    SkinnyNkTallPlan best;
    if (lda % 8 != 0 || !aligned(a, 16)) return best;
    const double cus = std::max(1, device_cus()), steps = double(cdiv(cdiv(k, 128), kTallWaves));  // steps of a wave
    for (int most = 1; most <= 4; ++most) {
        const int64_t tiles_m = cdiv(m, 16 * most);
        const int rb = int(cdiv(cdiv(m, tiles_m), 16));
        for (int cg = 1; cg <= 2; ++cg) {
            // (of the XCD with the most column tiles, times eight)
            const double groups = double(tiles_m) * double(8 * cdiv(cdiv(n, 16 * cg), 8)), share = std::max(1.0, groups / cus), rounds = std::ceil(share);
            const double us = 2.07 + 0.122 * share * rb * cg + rounds * steps * (0.319 * rb + 0.343 * cg + 0.086 * rb * cg);
            if (us < best.us) best = SkinnyNkTallPlan{us, rb, cg};
        }
    }
    return best;
}

void skinny_w8a16_nk_tall_launch(const SkinnyNkTallPlan &plan, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                                 int64_t lda, int64_t ldw, hipStream_t stream) {
    const int64_t tiles_m = cdiv(m, 16 * plan.rb), tiles_n = cdiv(n, 16 * plan.cg), grid = tiles_m * cdiv(tiles_n, 8) * 8;
    QMM_CHECK(grid < (int64_t(1) << 31), "problem too large for one launch");
    auto go = [&](auto kern, int lds) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
        launch(kern, dim3(uint32_t(grid)), dim3(64 * kTallWaves), size_t(lds), stream, static_cast<const _Float16 *>(a), static_cast<const int8_t *>(w), lda, ldw, int(m), int(n), int(k),
               int(tiles_m), int(tiles_n), static_cast<const _Float16 *>(scale), static_cast<const _Float16 *>(bias), static_cast<_Float16 *>(c));
    };
    auto of = [&](auto rb, auto cg) {
        constexpr int RB = decltype(rb)::value, CG = decltype(cg)::value;
        if (k % 128 == 0) go(skinny_w8a16_nk_tall_kernel<false, RB, CG>, tall_lds_bytes<RB, CG>());
        else go(skinny_w8a16_nk_tall_kernel<true, RB, CG>, tall_lds_bytes<RB, CG>());
    };
    auto rows = [&](auto cg) {
        using std::integral_constant;
        if (plan.rb == 1) of(integral_constant<int, 1>(), cg);
        else if (plan.rb == 2) of(integral_constant<int, 2>(), cg);
        else if (plan.rb == 3) of(integral_constant<int, 3>(), cg);
        else of(integral_constant<int, 4>(), cg);
    };
    if (plan.cg == 1) rows(std::integral_constant<int, 1>());
    else rows(std::integral_constant<int, 2>());
}

bool skinny_w8a16_nk_supported(const void *w, int64_t k, int64_t ldw) {
    return (ldw % 16 == 0) && (k % 16 == 0) && aligned(w, 16) && k > 0;
}

// Any M: 16 rows per pass, every pass streams the weights again (beyond a few passes the [K, N] layout and its MFMA
// GEMM are the better choice).
void skinny_w8a16_nk_launch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                            int64_t n, int64_t lda, int64_t ldw, hipStream_t stream) {
    const bool aligned_a = (lda % 8 == 0) && aligned(a, 16);
    // K off the steps: the kernel below, with conditions in all of its loop, only where the activations are not aligned. us, that one and the tall one: 1 x 4032 x 4096 6.8 and
    // 6.3, 16 x 4032 x 4096 9.4 and 6.3, 16 x 2112 x 11008 12.5 and 8.2, 16 x 9024 x 4096 17.7 and 10.0; large weights from the cache and from memory, 1 x 5776 x 9792 15.8 and 19.3, 14.7 and
    // 18.2, 1 x 10320 x 5376 18.1 and 22.1, 14.3 and 19.7, 8 x 10464 x 10240 40.0 and 41.5, 34.2 and 35.7; of 50 shapes of 1 to 16 rows, 1 to 107 MB, none is slower.
    if (k % 128 != 0 && aligned_a) {
        // (as many rows at a time as a launch has threads for, whatever the plan: 32-column tiles of 64 rows need the fewest, 16-column tiles of 16 rows eight times as many)
        const int64_t most = (int64_t(1) << 32) / (64 * kTallWaves) - 1, rows = std::max<int64_t>(1, most / (cdiv(cdiv(n, 16), 8) * 8)) * 16;
        for (int64_t m0 = 0; m0 < m; m0 += rows) {
            const int64_t mt = std::min(rows, m - m0);
            const _Float16 *am = static_cast<const _Float16 *>(a) + m0 * lda;
            skinny_w8a16_nk_tall_launch(skinny_w8a16_nk_tall_plan(am, mt, n, k, lda), am, w, scale, bias, static_cast<_Float16 *>(c) + m0 * n, mt, k, n, lda, ldw, stream);
        }
        return;
    }
    const dim3 grid(uint32_t(cdiv(n, 16)));
    for (int64_t m0 = 0; m0 < m; m0 += 16) {
        const int mt = int(std::min<int64_t>(16, m - m0));
        const _Float16 *ap = static_cast<const _Float16 *>(a) + m0 * lda;
        _Float16 *cp = static_cast<_Float16 *>(c) + m0 * n;
        auto go = [&](auto kern, int waves) {
            launch(kern, grid, dim3(64 * waves), 0, stream, ap, lda, static_cast<const int8_t *>(w), ldw, static_cast<const _Float16 *>(scale),
                   static_cast<const _Float16 *>(bias), cp, mt, int(k), int(n));
        };
        const bool full = k % 128 == 0;
        // more than 8 rows, a wide matrix and a long K: 32 columns per workgroup, the activation rows are read half as often
        if (full && aligned_a && mt > 8 && cdiv(n, 32) >= 256 && k >= 8192) {
            launch(skinny_w8a16_nk_wide_kernel<2, 8, 4>, dim3(uint32_t(cdiv(n, 32))), dim3(512), 0, stream, ap, lda,
                   static_cast<const int8_t *>(w), ldw, static_cast<const _Float16 *>(scale), static_cast<const _Float16 *>(bias), cp,
                   mt, int(k), int(n));
            continue;
        }
        // few column tiles: eight waves per workgroup keep enough loads in flight on each compute unit
        const bool eight = full && cdiv(n, 16) < 512 && k >= 8 * 128;
        const bool stage = full && aligned_a && mt > 2;
        if (eight && stage) go(skinny_w8a16_nk_kernel<true, true, 8, true>, 8);
        else if (eight) aligned_a ? go(skinny_w8a16_nk_kernel<true, true, 8>, 8) : go(skinny_w8a16_nk_kernel<false, true, 8>, 8);
        else if (stage) go(skinny_w8a16_nk_kernel<true, true, 4, true>, 4);
        else if (aligned_a) go(skinny_w8a16_nk_kernel<true, true, 4>, 4);  // (full)
        else full ? go(skinny_w8a16_nk_kernel<false, true, 4>, 4) : go(skinny_w8a16_nk_kernel<false, false, 4>, 4);
    }
}

}  // namespace qmm
