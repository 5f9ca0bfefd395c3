// FP8 e4m3 GEMMs of a few dozen to a few hundred rows on gemm_mid.h: c[m, n] = sum_k a[m, k] b[n, k], with optional per-tensor
// scales or with the block scales of matmul_f8_scaled (float32, scale_a [K/128, M], scale_b [N/128, K/128]), on the block-scaled
// MFMA with unit scales (16 x 16 x 128).
//
// A stage is 128 bytes of K of 128 columns, and goes through LDS to the four waves of a group (32 columns each): fetched in
// whole 128-byte rows it costs a CU's load path a quarter of what the operand's own pattern does, 16 bytes of 16 columns per
// instruction (512 x 7168 x 4096 with block scales: 34 against 49 us). Against the 256 x 128 tiles, block scales, K = 7168,
// N = 1536: 17 / 64 / 128 / 256 / 512 rows 19.0 / 19.7 / 22.4 / 26.8 / 27.7 -> 8.7 / 10.0 / 10.8 / 14.8 / 20.3 us. Block scales: a stage's products start from zero and are
// added times scale_a * scale_b; the row factors come with the stage's operands.
#include "gemm_mid.h"
#include "numeric.h"

namespace qmm {
namespace {

struct MidF8Args {
    void *c;
    const float *scale_a, *scale_b;
    int out_dtype, k_blocks;
};

template <bool SCALED, int RB>
struct MidF8 {
    using Args = MidF8Args;
    static constexpr int kElementBytes = 1;
    static constexpr int kStageK = 128;
    static constexpr bool kKeep = false;
    static constexpr int kGroupWaves = 4;
    static constexpr int kFrags = 2;
    static constexpr int kSpare = 0;
    static constexpr int kFactorBytes = SCALED ? 256 * ((RB + 3) / 4) : 0;  // of a wave: the stage's factors of its rows
    static constexpr int kWLdsBytes = 128 * 128 + kGroupWaves * kFactorBytes;
    static constexpr int kRowBytes = 128;
    static constexpr int kAChunks = 2;
    static constexpr int kMfmas = 2;       // per row block
    static constexpr int kWidenOps = SCALED ? 8 : 1;
    static constexpr int kWLoads = 4 + kFactorBytes / 256;
    struct Weights {
        int4v_t half[2][2];                // column ns * 2 + t: bytes 32 kg .. 32 kg + 31 of the stage
        int4v_t row_scale[SCALED ? RB : 1];  // rows 16 rb + 4 kg ..
        float col_scale;
    };
    using Fragments = Weights;
    __amdgpu_buffer_rsrc_t rsrc, rsrc_sa;
    const float *col_scales;
    int w_stage, side;
    int w_off[4];
    uint32_t w_read[2], sa_read;
    int sa_off, sa_stage;
    const MidF8Args &args;
    int k, n, kg;
    float alpha;

    __device__ __forceinline__ MidF8(const MidF8Args &x, const char *w, int ldb, int depth, int m, int cols, int m0, int n0, int side_, int lane)
        : side(side_), args(x), k(depth), n(cols), kg(lane >> 4) {
        const int ns = lane & 15, last = cols - 1 - n0;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w) + int64_t(n0) * ldb, 0, (last < 127 ? last : 127) * ldb + k, 0x00020000);
        w_stage = 128;
        // LDS row r of the 128 holds the column that fragment t = r / 16 % 2 has at slot r % 16, its chunks swizzled as the
        // activations' are; columns past the last read as zeros
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = (side * 4 + j) * 8 + (lane >> 3);
            const int col = (r & ~31) + (r & 15) * 2 + ((r >> 4) & 1);
            w_off[j] = col * ldb + ((lane & 7) ^ mid_key<128>(r)) * 16;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) w_read[q] = uint32_t((side * 32 + ns) * 128 + ((kg * 2 + q) ^ mid_key<128>(ns)) * 16);
        if constexpr (SCALED) {
            rsrc_sa = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x.scale_a), 0, x.k_blocks * m * 4, 0x00020000);
            col_scales = x.scale_b + int64_t(n0 >> 7) * x.k_blocks;
            sa_off = (m0 + lane) * 4;
            sa_stage = m * 4;
            sa_read = uint32_t(128 * 128 + side * kFactorBytes + kg * 16);
        }
    }
    __device__ __forceinline__ void load(uint4 *lds, uint32_t slot, uint32_t at, int) const {
#pragma unroll
        for (int j = 0; j < 4; ++j) buffer_load_to_lds_b128(rsrc, lds + (slot + (side * 4 + j) * 1024) / 16, int(uint32_t(w_off[j]) + at), 0);
        if constexpr (SCALED) {
            const uint32_t row = at >= kMidOutside ? kMidOutside : (at >> 7) * uint32_t(sa_stage);
#pragma unroll
            for (int j = 0; j < kFactorBytes / 256; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_sa, (__attribute__((address_space(3))) void *)(lds + (slot + 128 * 128 + side * kFactorBytes + j * 256) / 16), 4,
                                                         int(uint32_t(sa_off + j * 256) + row), 0, 0, 0);
        }
    }
    __device__ __forceinline__ void read(Weights &dst, uint32_t at) const {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            dst.half[0][q] = lds_read_b128_early<0>(w_read[q] + at);
            dst.half[1][q] = lds_read_b128_early<16 * 128>(w_read[q] + at);
        }
        if constexpr (SCALED)
            mid_for<0, RB>([&](auto r) { dst.row_scale[decltype(r)::value] = lds_read_b128_early<decltype(r)::value * 64>(sa_read + at); });
    }
    template <int NEWER>
    static __device__ __forceinline__ void settle(Weights &raw) {
        constexpr int kNewer = NEWER < 15 ? NEWER : 15;
        lds_wait_keep_newer<kNewer>(raw.half[0][0], raw.half[0][1]);
        lds_wait_keep_newer<kNewer>(raw.half[1][0], raw.half[1][1]);
        if constexpr (SCALED) mid_for<0, RB>([&](auto r) { lds_wait_keep_newer<kNewer>(raw.row_scale[decltype(r)::value]); });
    }
    __device__ __forceinline__ void factors(int) {
        alpha = 1.0f;
        if constexpr (!SCALED) {
            if (args.scale_a != nullptr) alpha *= *args.scale_a;
            if (args.scale_b != nullptr) alpha *= *args.scale_b;
        }
    }
    // K is a multiple of 16: a fragment's 16-byte chunks lie before its end or behind it
    __device__ __forceinline__ void widen(const Weights &raw, Fragments &b, int st) const {
        b = raw;
        if constexpr (SCALED) {
            // a stage past the end adds nothing, whatever the scales are: its products and row factors are zeros, so is this
            const float f = col_scales[st < args.k_blocks ? st : 0];
            b.col_scale = st < args.k_blocks ? f : 0.0f;
        } else if (st * 128 + 128 > k) {
            mask(b.half[0], st, kg);
            mask(b.half[1], st, kg);
        }
    }
    __device__ __forceinline__ void mask(int4v_t (&half)[2], int st, int group) const {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int keep = st * 128 + group * 32 + h * 16 < k ? -1 : 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) half[h][e] &= keep;
        }
    }
    template <typename R>
    static __device__ __forceinline__ void multiply(const int4v_t (&af)[2], const Fragments &b, float4_t (&acc)[2], R) {
        const int8v_t av = {af[0][0], af[0][1], af[0][2], af[0][3], af[1][0], af[1][1], af[1][2], af[1][3]};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int4v_t &lo = b.half[t][0], &hi = b.half[t][1];
            const int8v_t bv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if constexpr (SCALED) {
                const float4_t part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, float4_t{0.f, 0.f, 0.f, 0.f}, kFmtE4M3, kFmtE4M3, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[t][e] = __builtin_fmaf(part[e], __int_as_float(b.row_scale[R::value][e]) * b.col_scale, acc[t][e]);
            } else {
                acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, acc[t], kFmtE4M3, kFmtE4M3, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
            }
        }
    }
    __device__ __forceinline__ void store(int row, int col, const float (&v)[2]) const {
        if (col >= n) return;  // N is a multiple of 4
        const int64_t at = int64_t(row) * n + col;
        const float x = v[0] * alpha, y = v[1] * alpha;
        switch (args.out_dtype) {
            case HIDET_QMM_F32: *reinterpret_cast<float2 *>(static_cast<float *>(args.c) + at) = float2{x, y}; break;
            case HIDET_QMM_F16: *reinterpret_cast<half2_t *>(static_cast<uint16_t *>(args.c) + at) = half2_t{_Float16(x), _Float16(y)}; break;
            case HIDET_QMM_BF16:
                *reinterpret_cast<uint32_t *>(static_cast<uint16_t *>(args.c) + at) = f32_to_bf16_bits(x) | uint32_t(f32_to_bf16_bits(y)) << 16;
                break;
            default: *reinterpret_cast<uint16_t *>(static_cast<uint8_t *>(args.c) + at) = uint16_t(f32_to_e4m3(x) | uint32_t(f32_to_e4m3(y)) << 8);
        }
    }
};

template <bool SCALED>
bool launch_f8(const void *a, const void *b, const MidF8Args &args, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
               double limit_us, const Workspace &ws, hipStream_t stream) {
    // Fits (7 to 8 %) to the mean of a split's time on weights from memory and from the last-level cache, 427 shapes (block-scaled 424) of 17 to 1100 rows. A workgroup that walks all of K
    // for 32 rows is the fastest from the cache and 10 to 30 % behind two or three pieces from memory, where each round waits for it: us, cache and memory, in one
    // piece -> now: 337 x 5760 x 1824 14.2 and 19.0 -> 15.5 and 16.8, block-scaled 146 x 3584 x 3456 13.4 and 17.9 -> 12.8 and 14.1. Rows of the weight that do not begin on a cache line:
    // a round's 128 bytes of each lie on two (308 x 3024 x 1856 12.4 and 16.3 -> 12.5 and 13.4, 277 x 3680 x 1856 13.7 and 18.5 -> 12.8 and 13.9).
    const double apart = ldb % 128 != 0 ? 0.266 : 0.0;
    const MidCost low = SCALED ? MidCost{3.55, 0.845, 1.67, 0.108, 0.0, 0.004} : MidCost{3.84, 0.576 + apart, 1.72, 0.095, 0.0, 0.0031};
    const MidCost high = SCALED ? MidCost{4.55, 1.071, 1.19, 0.304, 0.0, 0.0092} : MidCost{5.24, 0.699 + apart, 1.01, 0.221, 0.0, 0.0085};
    const MidChoice c2 = mid_choose<MidF8<SCALED, 2>, 2, 3>(low, ws, m, n, k), c4 = mid_choose<MidF8<SCALED, 4>, 4, 3>(high, ws, m, n, k);
    if (std::min(c2.us, c4.us) > limit_us) return false;
    if (c2.us < c4.us) mid_launch<MidF8<SCALED, 2>, 2, 3>(c2, a, b, lda, ldb, args, m, n, k, ws, stream);
    else mid_launch<MidF8<SCALED, 4>, 4, 3>(c4, a, b, lda, ldb, args, m, n, k, ws, stream);
    return true;
}

}  // namespace

// Operands with 16-byte aligned rows, K a multiple of 16, N of 4, an output type of float32, float16, bfloat16 or e4m3. False: the
// estimate exceeds `limit_us`, or what a tile reads does not lie within 2 GiB.
bool mid_fp8_launch(const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int out_dtype,
                    const void *scale_a, const void *scale_b, bool block_scaled, double limit_us, void *workspace, int64_t workspace_bytes,
                    hipStream_t stream) {
    constexpr int64_t kMost = (int64_t(1) << 31) - (1 << 20);
    if (lda * 64 + k >= kMost || ldb * 128 + k >= kMost || cdiv(k, 128) * m * 4 >= kMost || n / 128 * cdiv(k, 128) >= kMost) return false;
    const MidF8Args args{c, static_cast<const float *>(scale_a), static_cast<const float *>(scale_b), out_dtype, int(cdiv(k, 128))};
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    return block_scaled ? launch_f8<true>(a, b, args, m, n, k, lda, ldb, limit_us, ws, stream)
                        : launch_f8<false>(a, b, args, m, n, k, lda, ldb, limit_us, ws, stream);
}

}  // namespace qmm
