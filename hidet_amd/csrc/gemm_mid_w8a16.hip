// W8A16 on gemm_mid.h: c[m, n] = (sum_k a[m, k] * w[k, n]) * scale[n] (+ bias[n]), int8 weights widened exactly to float16
// (a byte q ^ 0x80 as a subnormal number, times 2^15 less 0.25, is q / 512), float16 MFMA, fp32 sums; the results are multiplied by 512. Powers of
// two throughout: no bit differs from sums of q. The loop waits for its vector instructions as much as for its MFMAs, and this takes 40 for 32 codes
// of four columns where 1152 + q (0x6400 | (q ^ 0x80)) less 1152 takes 48: 96 x 4096 x 4096 13.2 -> 12.9 us, 128 x 2048 x 6144 10.7 -> 10.3, 64 x 1024 x
// 8192 7.3 -> 7.1. Tiles of 128 rows have MFMAs enough to hide either and keep 1152 + q (160 / 256 x 4096 x 11008 31.7 / 32.2 us with that, 32.0 / 32.5
// with q / 512; 384 x 4096 x 4096 20.8 and 21.5, 852 x 3648 x 3024 31.95 and 32.3).
#include "gemm_mid.h"

namespace qmm {
namespace {

struct MidW8Args {
    const _Float16 *scale, *bias;
    _Float16 *c;
    int ldc, n_out;
    int vector_out;    // rows of c start at multiples of 8 bytes and end with a lane's four columns
};

// SHIFTED: row-major weights of N = 4 i + 2. Their odd rows start between two dwords, which direct-to-LDS loads cannot; they are loaded
// from two bytes in front, so that in LDS a lane's four columns of an odd row lie across two dwords. The second of them is one more read, and the
// last lane's is missing: a tile has 124 columns. (A copy of the weight with rows of whole dwords, for the plain form: 4100 x 4098 11 us.)
// OFFSET: codes widened as 1152 + q less 1152 (row-major, rows of whole dwords).
template <bool NK, bool SHIFTED = false, bool OFFSET = false>
struct MidW8 {
    using Args = MidW8Args;
    // Row-major: a stage is 32 rows of 128 columns, so that memory is read in whole 128-byte lines (64-byte pieces reached
    // half the rate: 3 TB/s), and goes through LDS to the two waves of a group. K-contiguous: 64 k, 16 bytes of each of a
    // lane's 4 columns, straight into its registers.
    static constexpr int kElementBytes = 2;
    static constexpr int kStageK = NK ? 64 : 32;
    static constexpr bool kKeep = false;
    static constexpr int kGroupWaves = NK ? 1 : 2;
    static constexpr int kFrags = 4;
    static constexpr int kSpare = SHIFTED ? 4 : 0;
    static constexpr int kWLdsBytes = NK ? 0 : 32 * 128;
    static constexpr int kRowBytes = kStageK * 2;
    static constexpr int kAChunks = NK ? 2 : 1;
    static constexpr int kWLoads = NK ? 4 : 2;
    struct Weights {
        uint32_t u[NK ? 16 : 1];
        uint64_t pair[SHIFTED ? 6 : 4];
    };
    struct Fragments {
        half8_t h[kAChunks][4];
    };
    static constexpr int kMfmas = 4;      // per row block
    static constexpr int kWidenOps = OFFSET ? 48 : SHIFTED ? 44 : 40;  // VALU instructions of widen()
    int side_;
    __amdgpu_buffer_rsrc_t rsrc;
    int w_stage;       // bytes from one stage to the next
    int w_off[NK ? 4 : 2];
    uint32_t w_read;   // LDS address of this lane's first dword in a slot's weights (row-major)
    uint32_t sel[4];   // byte gathers of the columns
    uint32_t w_odd, w_next;  // SHIFTED: addresses of the lane's dword in the first odd row and of the one behind it
    int last_out;      // SHIFTED: columns from here on are not this tile's
    const MidW8Args &args;
    int k;
    half4_t scale4, bias4;

    __device__ __forceinline__ MidW8(const MidW8Args &x, const char *w, int ldw, int depth, int, int n, int, int n0, int side, int lane) : side_(side), args(x), k(depth) {
        const int kg = lane >> 4, ns = lane & 15;
        if constexpr (NK) {
            const int base = n0 < n - 4 ? n0 : n - 4, col = n0 + ns * 4 < n - 4 ? n0 + ns * 4 : n - 4;
            rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w) + int64_t(base) * ldw, 0, (n - 1 - base < 63 ? n - 1 - base : 63) * ldw + k, 0x00020000);
            w_stage = 64;
#pragma unroll
            for (int t = 0; t < 4; ++t) w_off[t] = (col + t - base) * ldw + kg * 16;
        } else {
            // Instruction b = 2 side + i brings rows 8 b .. 8 b + 7, the rows of the lanes with kg = b: its LDS position p (16
            // bytes each) holds chunk x % 8 of row x / 8, x = p ^ 4 b. A read of one row per kg, 64 bytes each, then
            // touches every bank once; kg 2 and 3 find the rows of a pair the other way round, which the gather undoes.
            rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w), 0, k * n, 0x00020000);  // rows past K read as code 0
            w_stage = 32 * n;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int blk = 2 * side + i, at = lane ^ (4 * blk);
                w_off[i] = (8 * blk + (at >> 3)) * n + n0 + (at & 7) * 16 - (SHIFTED ? 2 * ((at >> 3) & 1) : 0);
            }
            if constexpr (SHIFTED) {
                last_out = x.n_out > n0 + 124 ? n0 + 124 : x.n_out;
                auto position = [&](int row, int dword) { return uint32_t(kg * 1024 + row * 128 + ((dword >> 2) ^ ((kg & 1) * 4)) * 16 + (dword & 3) * 4); };
                const int dword = side * 16 + ns, swapped = kg >> 1;
                w_read = position(swapped, dword);
                w_odd = position(swapped ^ 1, dword);
                w_next = position(swapped ^ 1, dword < 31 ? dword + 1 : dword);
#pragma unroll
                for (int t = 0; t < 4; ++t) sel[t] = 0x0c000c00u | (uint32_t(4 + t) << 16) | uint32_t(t);
                return;
            }
            w_read = uint32_t(kg * 1024 + ((side * 4 + (ns >> 2)) ^ ((kg & 1) * 4)) * 16 + (ns & 3) * 4);
#pragma unroll
            for (int t = 0; t < 4; ++t) sel[t] = 0x0c000c00u | (kg >= 2 ? (uint32_t(t) << 16) | uint32_t(4 + t) : (uint32_t(4 + t) << 16) | uint32_t(t));
        }
    }
    __device__ __forceinline__ int limit() const { return SHIFTED ? last_out : args.n_out; }
    __device__ __forceinline__ void load(Weights &dst, uint32_t at) const {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint4v_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, int(uint32_t(w_off[t]) + at), 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) dst.u[4 * t + e] = v[e];
        }
    }
    __device__ __forceinline__ void load(uint4 *lds, uint32_t slot, uint32_t at, int) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) buffer_load_to_lds_b128(rsrc, lds + (slot + (2 * side_ + i) * 1024) / 16, int(uint32_t(w_off[i]) + at), 0);
    }
    __device__ __forceinline__ void factors(int col) {
        bias4 = half4_t{_Float16(-0.0f), _Float16(-0.0f), _Float16(-0.0f), _Float16(-0.0f)};
        scale4 = bias4;
        if (col >= limit()) return;
        if (SHIFTED) {
#pragma unroll
            for (int t = 0; t < 4; t += 2)
                if (col + t < limit()) {  // (N is even)
                    __builtin_memcpy(reinterpret_cast<_Float16 *>(&scale4) + t, args.scale + col + t, 4);
                    if (args.bias != nullptr) __builtin_memcpy(reinterpret_cast<_Float16 *>(&bias4) + t, args.bias + col + t, 4);
                }
        } else if (args.vector_out) {
            __builtin_memcpy(&scale4, args.scale + col, 8);
            if (args.bias != nullptr) __builtin_memcpy(&bias4, args.bias + col, 8);
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (col + t < args.n_out) {
                    scale4[t] = args.scale[col + t];
                    if (args.bias != nullptr) bias4[t] = args.bias[col + t];
                }
        }
    }
    // rows j and j + 1 of the lane's eight, 128 bytes apart; SHIFTED: rows 0, 2 and 4, 6, then 1, 3 and 5, 7 and the dwords behind those
    __device__ __forceinline__ void read(Weights &dst, uint32_t at) const {
        if constexpr (SHIFTED) {
            const uint32_t from[3] = {w_read + at, w_odd + at, w_next + at};
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                uint64_t lo, hi;
                asm volatile("ds_read2_b32 %0, %1 offset0:0 offset1:64" : "=v"(lo) : "v"(from[i]));
                asm volatile("ds_read2_b32 %0, %1 offset0:128 offset1:192" : "=v"(hi) : "v"(from[i]));
                dst.pair[2 * i] = lo;
                dst.pair[2 * i + 1] = hi;
            }
            return;
        }
        uint64_t v[4];
        asm volatile("ds_read2_b32 %0, %1 offset0:0 offset1:32" : "=v"(v[0]) : "v"(w_read + at));
        asm volatile("ds_read2_b32 %0, %1 offset0:64 offset1:96" : "=v"(v[1]) : "v"(w_read + at));
        asm volatile("ds_read2_b32 %0, %1 offset0:128 offset1:160" : "=v"(v[2]) : "v"(w_read + at));
        asm volatile("ds_read2_b32 %0, %1 offset0:192 offset1:224" : "=v"(v[3]) : "v"(w_read + at));
#pragma unroll
        for (int p = 0; p < 4; ++p) dst.pair[p] = v[p];
    }
    // u: two bytes q ^ 0x80 below zero bytes (the xor is done four codes at a time, where 0x6480 in front of a subtraction takes one for two)
    static __device__ __forceinline__ half8_t over_512(const uint32_t (&u)[4]) {
        half8_t out;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const half2_t v = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, u[p]), half2_t{_Float16(32768.0f), _Float16(32768.0f)}, half2_t{_Float16(-0.25f), _Float16(-0.25f)});
            out[2 * p] = v[0];
            out[2 * p + 1] = v[1];
        }
        return out;
    }
    // u: two bytes q below zero bytes
    static __device__ __forceinline__ half8_t minus_1152(const uint32_t (&u)[4]) {
        half8_t out;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const half2_t v = __builtin_bit_cast(half2_t, u[p] ^ 0x64806480u) - half2_t{_Float16(1152.0f), _Float16(1152.0f)};
            out[2 * p] = v[0];
            out[2 * p + 1] = v[1];
        }
        return out;
    }
    template <int NEWER>
    static __device__ __forceinline__ void settle(Weights &raw) {
        if constexpr (SHIFTED)
            asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(raw.pair[0]), "+v"(raw.pair[1]), "+v"(raw.pair[2]), "+v"(raw.pair[3]), "+v"(raw.pair[4]), "+v"(raw.pair[5]) : "n"(NEWER));
        else
            asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(raw.pair[0]), "+v"(raw.pair[1]), "+v"(raw.pair[2]), "+v"(raw.pair[3]) : "n"(NEWER));
    }
    __device__ __forceinline__ void widen(const Weights &raw, Fragments &b, int) const {
        if constexpr (OFFSET) {
            static_assert(!NK && !SHIFTED, "dwords of four columns");
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                uint32_t u[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) u[p] = __builtin_amdgcn_perm(uint32_t(raw.pair[p] >> 32), uint32_t(raw.pair[p]), sel[t]);
                b.h[0][t] = minus_1152(u);
            }
            return;
        }
        constexpr uint32_t kFlip = 0x80808080u;
        auto dword = [&](int i, int p) { return uint32_t(p & 1 ? raw.pair[i + p / 2] >> 32 : raw.pair[i + p / 2]); };
        uint32_t lo[4], hi[4];  // rows 2 p and 2 p + 1
        if constexpr (!NK) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                lo[p] = (SHIFTED ? dword(0, p) : uint32_t(raw.pair[p])) ^ kFlip;
                hi[p] = (SHIFTED ? __builtin_amdgcn_alignbyte(dword(4, p), dword(2, p), 2) : uint32_t(raw.pair[p] >> 32)) ^ kFlip;
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t u[4];
            if constexpr (NK) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {  // bytes 8 q .. 8 q + 7 of the lane's sixteen
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const uint32_t src = raw.u[4 * t + 2 * q + p / 2] ^ kFlip;
                        u[p] = __builtin_amdgcn_perm(src, src, (p & 1) ? 0x0c030c02u : 0x0c010c00u);
                    }
                    b.h[q][t] = over_512(u);
                }
            } else {
#pragma unroll
                for (int p = 0; p < 4; ++p) u[p] = __builtin_amdgcn_perm(hi[p], lo[p], sel[t]);
                b.h[0][t] = over_512(u);
            }
        }
    }
    // zero what a fragment holds past K (the next row's values, which may be anything); K is even
    __device__ __forceinline__ void mask(int4v_t (&af)[kAChunks], int st, int kg) const {
#pragma unroll
        for (int q = 0; q < kAChunks; ++q) {
            const int left = k - (st * kStageK + (kg * kAChunks + q) * 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t keep = left > 2 * e ? 0xFFFFFFFFu : 0u;
                af[q][e] = int(uint32_t(af[q][e]) & keep);
            }
        }
    }
    template <typename R>
    static __device__ __forceinline__ void multiply(const int4v_t (&af)[kAChunks], const Fragments &b, float4_t (&acc)[4], R) {
#pragma unroll
        for (int q = 0; q < kAChunks; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, af[q]), b.h[q][t], acc[t], 0, 0, 0);
    }
    __device__ __forceinline__ void store(int row, int col, const float (&v)[4]) const {
        if (col >= limit()) return;
        half4_t o;
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = scaled_biased_f16(OFFSET ? v[t] : v[t] * 512.0f, float(scale4[t]), float(bias4[t]));
        _Float16 *dst = args.c + int64_t(row) * args.ldc + col;
        if (SHIFTED) {
#pragma unroll
            for (int t = 0; t < 4; t += 2)
                if (col + t < limit()) __builtin_memcpy(dst + t, reinterpret_cast<const _Float16 *>(&o) + t, 4);
        } else if (args.vector_out) {
            *reinterpret_cast<half4_t *>(dst) = o;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (col + t < args.n_out) dst[t] = o[t];
        }
    }
};

template <typename T>
struct Form {
    using type = T;
};

}  // namespace

// Per shape and row count the tile and the K split of the smallest estimated time. `limit_us`: no launch and false where that
// exceeds it - or where the operands have a form this kernel does not take.
// `n_out` <= n columns of the result are written, at a row stride of ldc.
bool mid_w8a16_launch(const void *a, const void *w, bool nk, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                      int64_t n, int64_t lda, int64_t ldw, int64_t n_out, int64_t ldc, double limit_us, const Workspace &ws, hipStream_t stream) {
    const MidW8Args args{static_cast<const _Float16 *>(scale), static_cast<const _Float16 *>(bias), static_cast<_Float16 *>(c), int(ldc), int(n_out),
                         n_out % 4 == 0 && ldc % 4 == 0 && aligned(c, 8)};
    // four columns of a lane are all inside the matrix; loads start at multiples of four bytes, and no dword of the
    // activations lies half outside their buffer (it would read as zero: K is even); what a tile reads lies within 2 GiB
    // (kMidOutside)
    constexpr int64_t kMost = (int64_t(1) << 31) - (1 << 20);
    const bool shifted = !nk && n % 4 == 2 && n_out == n;
    if ((n % 4 != 0 && !shifted) || k % 2 != 0 || lda % 2 != 0 || !aligned(a, 4) || !aligned(w, 4) || lda * 256 + k * 2 >= kMost || ldc >= kMost) return false;
    const int64_t las = lda * 2;
    if (nk) {
        if (ldw % 4 != 0 || ldw * 64 + k >= kMost) return false;
        const MidChoice c2 = mid_choose<MidW8<true>, 2, 4>({5.5, 1.4, 1.5, 0.3}, ws, m, n, k), c4 = mid_choose<MidW8<true>, 4, 2>({6.0, 1.6, 1.5, 0.4}, ws, m, n, k);
        if (std::min(c2.us, c4.us) > limit_us) return false;
        if (c2.us < c4.us) mid_launch<MidW8<true>, 2, 4>(c2, a, w, las, ldw, args, m, n, k, ws, stream);
        else mid_launch<MidW8<true>, 4, 2>(c4, a, w, las, ldw, args, m, n, k, ws, stream);
        return true;
    }
    if ((k + 64) * n >= kMost) return false;
    constexpr double kFullRound = 0.62;  // 256 pieces of 16 KiB at 6.8 TB/s
    auto run = [&](auto form, auto high) {
        using Op = typename decltype(form)::type;
        using High = typename decltype(high)::type;  // on 128 rows
        const MidChoice c2 = mid_choose<Op, 2, 6>({4.07, 0.37, 1.55, 0.077, kFullRound, 0.006}, ws, m, n, k),
                        c4 = mid_choose<Op, 4, 4>({4.85, 0.485, 1.2, 0.252, kFullRound, 0.0089}, ws, m, n, k),
                        c8 = mid_choose<High, 8, 3>({6.96, 0.765, 1.42, 0.426, kFullRound, 0.0142}, ws, m, n, k);
        const double us = std::min({c2.us, c4.us, c8.us});
        if ((us == c2.us ? c2 : us == c4.us ? c4 : c8).busy_us > limit_us) return false;
        if (us == c2.us) mid_launch<Op, 2, 6>(c2, a, w, las, n, args, m, n, k, ws, stream);
        else if (us == c4.us) mid_launch<Op, 4, 4>(c4, a, w, las, n, args, m, n, k, ws, stream);
        else mid_launch<High, 8, 3>(c8, a, w, las, n, args, m, n, k, ws, stream);
        return true;
    };
    return shifted ? run(Form<MidW8<false, true>>(), Form<MidW8<false, true>>()) : run(Form<MidW8<false>>(), Form<MidW8<false, false, true>>());
}

}  // namespace qmm
