// W4A16 GEMMs of a few dozen to a few hundred rows on gemm_mid.h: c[m, n] = sum_k a[m, k] * q[k, n] * scales[k / group, n], bfloat16 or
// float16 activations, packed int4 codes (two columns to a byte).
//
// A stage's codes are widened exactly (bfloat16: v_cvt_off_f32_i4 gives q / 16 of a nibble, float16: 1032 + q by one bit operation
// and one packed subtract) and its sums are added times the group's scale in float32, so the weights are not rounded to 16
// bits as the prefill kernels do. (The bandwidth-bound kernel's form, biased codes and the bias taken off the sums, needs
// fewer vector instructions but turns an infinite activation, or one within a factor of 136 of the largest, into NaN.) bfloat16, groups
// of 128: 4096 x 4096, 49 / 128 / 256 / 512 rows 12.5 / 16.4 / 21.9 / 29.4 us; 11008 x 4096, 17 / 64 / 256 rows 15.6 / 20.8 / 43.8 us.
//
// What bounds it is the vector ALU, widening and scaling: 112 instructions for 64 k of a wave's 64 columns and 64 more per stage to scale 64 rows,
// beside 32 MFMAs of four times the length of an instruction. So a stage is as deep as groups of 64 and 128 and the registers allow: 64 k, scaled once, with
// half the barriers (32 before: 4096 x 4096, 128 / 256 / 512 rows 18.6 / 27.4 / 35.6 us; 11008 x 4096, 64 / 256 rows 23.9 / 48.9, 128 rows on the tall
// tiles 38.7 -> 27.2), and the codes of two rows are gathered in one byte permutation. Groups of an odd number of 32 keep stages of 32, and so do small launches (launch_w4).
#include "gemm_mid.h"
#include "w4_traits.h"

namespace qmm {
namespace {

struct MidW4Args {
    const uint16_t *scales, *bias;
    uint16_t *c;
    int group_stages;  // stages in a group
    uint32_t group_magic;
    int scale_bytes;
    int vector_out;
};

// STEPS: MFMA steps of 32 k in a stage. Two where the groups are whole 64-deep stages.
template <int DT, int RB, int STEPS>
struct MidW4 {
    using Args = MidW4Args;
    using T = W4Traits<DT>;
    static constexpr int kElementBytes = 2;
    static constexpr int kStageK = 32 * STEPS;
    static constexpr bool kKeep = true;
    static constexpr int kGroupWaves = 2;
    static constexpr int kFrags = 4;
    static constexpr int kSpare = 0;
    static constexpr int kCodeBytes = kStageK * 64;                // rows of 128 columns
    static constexpr int kWLdsBytes = kCodeBytes + kGroupWaves * 256;  // and the scales of each wave's 64 columns
    static constexpr int kRowBytes = kStageK * 2;
    static constexpr int kAChunks = STEPS;
    static constexpr int kMfmas = 4 * STEPS;                       // per row block
    static constexpr int kWidenOps = 64 * STEPS + 16 * RB;
    static constexpr int kWLoads = STEPS + 1;
    struct Weights {
        uint64_t pair[STEPS][4];
        uint64_t scale4;
    };
    struct Fragments {
        uint4 b[STEPS][4];
        float scale[4];
    };
    __amdgpu_buffer_rsrc_t rsrc, rsrc_s;
    int w_stage, side;
    int w_off[STEPS], s_off, n2;
    uint32_t w_read[STEPS], s_read;
    uint32_t pick;  // byte gather of the lane's two bytes, of four columns, from the dwords of two rows (float16: of the first, each below a zero byte)
    const MidW4Args &args;
    int n;
    float bias4[4];

    __device__ __forceinline__ MidW4(const MidW4Args &x, const char *w, int row_bytes, int depth, int, int cols, int, int n0, int side_, int lane)
        : side(side_), args(x), n(cols) {
        const int kg = lane >> 4, ns = lane & 15;
        w_stage = kStageK * row_bytes;
        n2 = cols * 2;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w), 0, depth * row_bytes, 0x00020000);
        rsrc_s = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x.scales), 0, x.scale_bytes, 0x00020000);
        // Instruction i brings rows 16 i .. 16 i + 15: its LDS position p (16 bytes each) holds chunk y % 4 of row 8 (y / 4 % 2) + y / 8, y = p
        // with the upper bit of the chunk flipped in the second instruction (one step; lanes of kg read instruction kg / 2, half kg % 2) or with
        // twice i flipped (two steps; instruction kg, half step). A read of one row per lane group (32 bytes each) then
        // touches every bank once.
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const int b = side * STEPS + i, y = lane ^ (b << 1);
            w_off[i] = (16 * b + ((y >> 2) & 1) * 8 + (y >> 3)) * row_bytes + (n0 >> 1) + (y & 3) * 16;
            const int from = STEPS == 1 ? kg >> 1 : kg, half = STEPS == 1 ? kg & 1 : i;
            w_read[i] = uint32_t(from * 1024 + ((half * 4 + side * 2 + (ns >> 3)) ^ (from << 1)) * 16 + ((ns & 7) >> 1) * 4);
        }
        pick = (DT == HIDET_QMM_BF16 ? 0x05040100u : 0x0c040c00u) + (ns & 1) * (DT == HIDET_QMM_BF16 ? 0x02020202u : 0x00020002u);
        s_off = (n0 + side * 64) * 2 + (lane & 31) * 4;
        s_read = uint32_t(kCodeBytes + side * 256 + ns * 8);
    }
    __device__ __forceinline__ void load(uint4 *lds, uint32_t slot, uint32_t at, int st) const {
#pragma unroll
        for (int i = 0; i < STEPS; ++i) buffer_load_to_lds_b128(rsrc, lds + (slot + (side * STEPS + i) * 1024) / 16, int(uint32_t(w_off[i]) + at), 0);
        const uint32_t row = at >= kMidOutside ? kMidOutside : uint32_t(mid_div(st, args.group_stages, args.group_magic)) * uint32_t(n2);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s, (__attribute__((address_space(3))) void *)(lds + (slot + kCodeBytes + side * 256) / 16), 4, int(uint32_t(s_off) + row), 0, 0, 0);
    }
    __device__ __forceinline__ void read(Weights &dst, uint32_t at) const {
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            uint64_t v[4];
            asm volatile("ds_read2_b32 %0, %1 offset0:0 offset1:32" : "=v"(v[0]) : "v"(w_read[i] + at));
            asm volatile("ds_read2_b32 %0, %1 offset0:64 offset1:96" : "=v"(v[1]) : "v"(w_read[i] + at));
            asm volatile("ds_read2_b32 %0, %1 offset0:128 offset1:160" : "=v"(v[2]) : "v"(w_read[i] + at));
            asm volatile("ds_read2_b32 %0, %1 offset0:192 offset1:224" : "=v"(v[3]) : "v"(w_read[i] + at));
#pragma unroll
            for (int p = 0; p < 4; ++p) dst.pair[i][p] = v[p];
        }
        asm volatile("ds_read_b64 %0, %1" : "=v"(dst.scale4) : "v"(s_read + at));
    }
    template <int NEWER>
    static __device__ __forceinline__ void settle(Weights &raw) {
#pragma unroll
        for (int i = 0; i < STEPS; ++i)
            asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(raw.pair[i][0]), "+v"(raw.pair[i][1]), "+v"(raw.pair[i][2]), "+v"(raw.pair[i][3]), "+v"(raw.scale4) : "n"(NEWER));
    }
    __device__ __forceinline__ void widen(const Weights &raw, Fragments &f, int) const {
#pragma unroll
        for (int i = 0; i < STEPS; ++i)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t lo = uint32_t(raw.pair[i][p]), hi = uint32_t(raw.pair[i][p] >> 32);  // rows 2 p and 2 p + 1
                if constexpr (DT == HIDET_QMM_BF16) {
                    // (upper halves and bytes are operand selections of the conversion, unlike second ones: three shifts, five if left to the compiler)
                    const uint32_t u = __builtin_amdgcn_perm(hi, lo, pick);
                    uint32_t v = u >> 4;
                    asm("" : "+v"(v));
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
                        const uint32_t from = (t & 1 ? v : u) >> (8 * (t >> 1));
                        const bf16x2_t pair = {static_cast<__bf16>(__builtin_amdgcn_cvt_off_f32_i4(int(from))), static_cast<__bf16>(__builtin_amdgcn_cvt_off_f32_i4(int(from >> 16)))};
                        reinterpret_cast<uint32_t *>(&f.b[i][t])[p] = __builtin_bit_cast(uint32_t, pair);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const uint32_t u = __builtin_amdgcn_perm(hi, lo, pick + uint32_t(e) * 0x00010001u);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const half2_t v = __builtin_bit_cast(half2_t, ((u >> (4 * h)) & 0x000F000Fu) ^ T::kMagic) - half2_t{_Float16(T::kBias), _Float16(T::kBias)};
                            reinterpret_cast<uint32_t *>(&f.b[i][2 * e + h])[p] = __builtin_bit_cast(uint32_t, v);
                        }
                    }
                }
            }
#pragma unroll
        for (int t = 0; t < 4; ++t) f.scale[t] = T::to_f32(uint16_t(raw.scale4 >> (16 * t))) * (DT == HIDET_QMM_BF16 ? 16.0f : 1.0f);
    }
    static __device__ __forceinline__ void mask(int4v_t (&)[STEPS], int, int) {}  // K is a multiple of the stages
    template <typename R>
    static __device__ __forceinline__ void multiply(const int4v_t (&af)[STEPS], const Fragments &f, float4_t (&acc)[4], R) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < STEPS; ++i) part = T::mfma(__builtin_bit_cast(uint4, af[i]), f.b[i][t], part);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t][e] = __builtin_fmaf(part[e], f.scale[t], acc[t][e]);
        }
    }
    __device__ __forceinline__ void factors(int col) {
#pragma unroll
        for (int t = 0; t < 4; ++t) bias4[t] = args.bias != nullptr && col < n ? T::to_f32(args.bias[col + t]) : -0.0f;
    }
    __device__ __forceinline__ void store(int row, int col, const float (&v)[4]) const {
        if (col >= n) return;  // N is a multiple of 8
        uint16_t o[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            o[t] = DT == HIDET_QMM_BF16 ? biased_bf16_bits(v[t], bias4[t]) : __builtin_bit_cast(uint16_t, scaled_biased_f16(v[t], 1.0f, bias4[t]));
        uint16_t *dst = args.c + int64_t(row) * n + col;
        if (args.vector_out) {
            *reinterpret_cast<uint2 *>(dst) = uint2{o[0] | uint32_t(o[1]) << 16, o[2] | uint32_t(o[3]) << 16};
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) dst[t] = o[t];
        }
    }
};

// `args_of`: the arguments for stages of so many MFMA steps. Tiles of 32 rows have stages of 32 k also where groups allow 64, if a workgroup has few rounds:
// more pieces of K divide the rest better and each costs less. us, stages of 32 and 64 k: 26 rows, 1408 x 2240 8.1 and 8.5, 1920 x 1096 7.8 and
// 8.2, 6528 x 1448 12.0 and 12.2, 128 rows, 1920 x 1096 9.0 and 9.3; 2560 x 4096 13.4 and 12.9, 3072 x 2048 11.3 and 11.1.
template <int DT, int STEPS, typename ArgsOf>
bool launch_w4(const void *a, const void *w, ArgsOf args_of, int64_t m, int64_t n, int64_t k, int64_t lda, double limit_us, const Workspace &ws,
               hipStream_t stream) {
    using Low = MidW4<DT, 2, STEPS>;
    using High = MidW4<DT, 4, STEPS>;
    constexpr int kLow = STEPS == 1 ? 6 : 4, kHigh = STEPS == 1 ? 5 : 3;  // stages in the ring
    const MidCost low = STEPS == 1 ? MidCost{5.5, 0.5, 1.4, 0.4} : MidCost{4.21, 1.019, 1.75, 0.086, 0.0, 0.0058};
    const MidCost high = STEPS == 1 ? MidCost{6.0, 0.9, 1.5, 0.5} : MidCost{5.1, 1.38, 1.51, 0.241, 0.0, 0.009};
    const MidChoice c2 = mid_choose<Low, 2, kLow>(low, ws, m, n, k), c4 = mid_choose<High, 4, kHigh>(high, ws, m, n, k);
    MidChoice shallow;
    if constexpr (STEPS == 2) shallow = mid_choose<MidW4<DT, 2, 1>, 2, 6>({3.91, 0.602, 1.71, 0.0625, 0.0, 0.0049}, ws, m, n, k);
    const double us = std::min({c2.us, c4.us, shallow.us});
    if (us > limit_us) return false;
    if (us == c4.us) {
        mid_launch<High, 4, kHigh>(c4, a, w, lda * 2, n / 2, args_of(STEPS), m, n, k, ws, stream);
        return true;
    }
    if constexpr (STEPS == 2) {
        if (us == shallow.us) {
            mid_launch<MidW4<DT, 2, 1>, 2, 6>(shallow, a, w, lda * 2, n / 2, args_of(1), m, n, k, ws, stream);
            return true;
        }
    }
    mid_launch<Low, 2, kLow>(c2, a, w, lda * 2, n / 2, args_of(STEPS), m, n, k, ws, stream);
    return true;
}

}  // namespace

// Groups of a multiple of 32. False: the estimate exceeds `limit_us`, or the operands have a form this kernel does not take.
bool mid_w4a16_launch(const void *a, const void *w, const void *scales, const void *bias, void *c, int64_t m, int64_t k, int64_t n, int64_t lda,
                      int group, int dtype, double limit_us, void *workspace, int64_t workspace_bytes, hipStream_t stream) {
    constexpr int64_t kMost = (int64_t(1) << 31) - (1 << 20);
    if (k == 0 || group % 32 != 0 || n % 8 != 0 || lda % 2 != 0 || !aligned(a, 4) || !aligned(w, 4) || !aligned(scales, 4) || !aligned(c, 2) || !aligned(bias, 2) ||
        lda * 256 + k * 2 >= kMost || (k + 64) * (n / 2) >= kMost || (k / group) * n * 2 >= kMost)
        return false;
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    auto args_of = [&](int steps) {
        const int group_stages = group / (32 * steps);
        return MidW4Args{static_cast<const uint16_t *>(scales), static_cast<const uint16_t *>(bias), static_cast<uint16_t *>(c), group_stages, mid_magic(group_stages),
                         int((k / group) * n * 2), aligned(c, 8)};
    };
    auto run = [&](auto steps) {
        constexpr int STEPS = decltype(steps)::value;
        return dtype == HIDET_QMM_F16 ? launch_w4<HIDET_QMM_F16, STEPS>(a, w, args_of, m, n, k, lda, limit_us, ws, stream)
                                      : launch_w4<HIDET_QMM_BF16, STEPS>(a, w, args_of, m, n, k, lda, limit_us, ws, stream);
    };
    return group % 64 == 0 ? run(std::integral_constant<int, 2>()) : run(std::integral_constant<int, 1>());
}

}  // namespace qmm
