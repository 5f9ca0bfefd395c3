// Quantization kernels: symmetric int8/int16 quantize + dequantize over a [outer, reduce, inner]
// view, group-wise signed int4 with nibble packing, and per-tensor float8 e4m3.
//
// Codes and scales match the CPU definition (IEEE division, then rounding) bit for bit. A product with the reciprocal stands in
// for a division only where it provably rounds alike (round_quotients_f32, round_quotients_16, e4m3_codes4).
#include "common.h"
#include "gemm_tiling.h"
#include "numeric.h"

namespace qmm {
namespace {


template <typename T>
__global__ void zero_kernel(T *p, int64_t n) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Nearest integer (ties to even) of v, |v| < 2^21, in the low bits of the returned word.
__device__ __forceinline__ uint32_t nearest_bits(float v) { return __float_as_uint(v + 12582912.0f); }  // 1.5 * 2^23

// code[e] = round_half_away(fl(x[e] / s[e])) as integers in the low bits, clamped to +-bound: the value IEEE division
// followed by roundf gives, with the division left out where it cannot matter. x * rcp(s) is within 2^-22 of the quotient
// (rcp is good to one unit in the last place, then two roundings), so its nearest integer is the answer unless it lies within bound * 2^-21 of a tie. |x| is at most the
// maximum the scale was made from, so that answer needs no clamp. `fast` is false for a scale whose reciprocal may be
// imprecise (zero, tiny, huge, NaN); a NaN among x fails the comparison and takes the division. 5 issue slots per element
// instead of 20: dividing every element kept the quantizers at the VALU's rate.
__device__ __forceinline__ void round_quotients_f32(const float (&x)[4], const float (&s)[4], const float (&inv)[4], bool fast, float low,
                                                    float high, uint32_t (&code)[4]) {
    const float limit = 0.5f - (high + 1.0f) * 0x1p-21f;
    bool sure = fast;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = __builtin_fmaf(x[e], inv[e], 12582912.0f);
        code[e] = __float_as_uint(t);
        sure = sure && fabsf(__builtin_fmaf(x[e], inv[e], 12582912.0f - t)) < limit;
    }
    if (__builtin_expect(!sure, 0)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) code[e] = s[e] != 0.0f ? uint32_t(int(fminf(fmaxf(roundf(x[e] / s[e]), low), high))) : 0u;
    }
}
__device__ __forceinline__ bool reciprocal_is_precise(float s) {
    const float a = fabsf(s);
    return a >= 0x1p-100f && a <= 0x1p100f;
}

// The 16-bit types: rint(rnd(fl(x[e] / s[e]))), rnd = round to the type (ties to even, as the reference's GPU lowering),
// without the division. q = x * rcp(s) is within 2^-22 of the quotient, its remainder x - q s is exact (s has at most 11
// significant bits), and one correction leaves q within 2^-24 (1 + 2^-19). A quotient of two 11-bit numbers that is not
// itself a midpoint between two numbers of the type (12 bits) is at least 2^-23 away from one, and one that is comes out
// exactly: q rounds as the quotient does. (NaN gives the lowest code, as the clamp of the division's result does.)
template <int DT>
__device__ __forceinline__ void round_quotients_16(const float (&x)[4], const float (&s)[4], const float (&inv)[4], bool fast, float low,
                                                   float high, uint32_t (&code)[4]) {
    if (__builtin_expect(fast, 1)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float q = x[e] * inv[e];
            q = __builtin_fmaf(__builtin_fmaf(-q, s[e], x[e]), inv[e], q);
            code[e] = nearest_bits(__builtin_amdgcn_fmed3f(round_to<DT>(q), low, high));
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) code[e] = s[e] != 0.0f ? uint32_t(int(fminf(fmaxf(rintf(round_to<DT>(x[e] / s[e])), low), high))) : 0u;
    }
}

// Codes of four elements, in the low bits: saturating_cast(round(rnd(w / scale))), zero where the scale is.
template <int DT, int QT>
__device__ __forceinline__ void codes4(const float (&x)[4], const float (&s)[4], const float (&inv)[4], bool fast, uint32_t (&code)[4]) {
    constexpr float low = QT == HIDET_QMM_I8 ? -128.0f : -32768.0f, high = QT == HIDET_QMM_I8 ? 127.0f : 32767.0f;
    if constexpr (DT == HIDET_QMM_F32) round_quotients_f32(x, s, inv, fast, low, high, code);
    else round_quotients_16<DT>(x, s, inv, fast, low, high, code);
}

// Scales of four columns from their maxima, and what codes4 wants to know about them.
template <int DT, int QT>
__device__ __forceinline__ bool scales4(const float (&amax)[4], float (&s)[4], float (&inv)[4]) {
    const float qmax = QT == HIDET_QMM_I8 ? 127.0f : 32767.0f;
    bool fast = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        s[e] = round_to<DT>(amax[e] / qmax);
        inv[e] = __builtin_amdgcn_rcpf(s[e]);
        fast = fast && reciprocal_is_precise(s[e]);
    }
    return fast;
}

// Largest of a wave's values, in every lane (no LDS: the six exchanges of a shuffled tree are 0.3 us of a kernel that runs for 3).
__device__ __forceinline__ float wave_max(float m) {
    auto step = [&m](auto ctrl, auto rows) {  // (lanes that the move does not reach keep their own value)
        const int v = __float_as_int(m);
        m = fmaxf(m, __int_as_float(__builtin_amdgcn_update_dpp(v, v, decltype(ctrl)::value, decltype(rows)::value, 0xF, false)));
    };
    using std::integral_constant;
    step(integral_constant<int, 0xB1>(), integral_constant<int, 0xF>());   // quads: neighbours
    step(integral_constant<int, 0x4E>(), integral_constant<int, 0xF>());   // quads: pairs
    step(integral_constant<int, 0x141>(), integral_constant<int, 0xF>());  // half rows of 16 lanes, mirrored
    step(integral_constant<int, 0x140>(), integral_constant<int, 0xF>());  // rows, mirrored
    step(integral_constant<int, 0x142>(), integral_constant<int, 0xA>());  // lane 15 of rows 0, 2 to rows 1, 3
    step(integral_constant<int, 0x143>(), integral_constant<int, 0xC>());  // lane 31 to rows 2, 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 63));
}

// Four elements at the alignment of one: rows of an odd length start anywhere (the hardware takes such accesses whole).
typedef float float4_at4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t half4_at2_t __attribute__((ext_vector_type(4), aligned(2)));

// Elements i .. i + 3, the ones from `count` on left out (read as zero, not stored).
template <int DT>
__device__ __forceinline__ void load_upto4(const void *p, int64_t i, int64_t count, float (&x)[4]) {
    if (count >= 4) {
        if constexpr (DT == HIDET_QMM_F32) {
            const float4_at4_t v = *reinterpret_cast<const float4_at4_t *>(static_cast<const float *>(p) + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = v[e];
        } else {
            const half4_at2_t v = *reinterpret_cast<const half4_at2_t *>(static_cast<const uint16_t *>(p) + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = DT == HIDET_QMM_F16 ? f16_bits_to_f32(v[e]) : bf16_bits_to_f32(v[e]);
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x[e] = 0.0f;
        if (e < count) x[e] = load_as_f32<DT>(p, i + e);
    }
}
template <int DT>
__device__ __forceinline__ void store_upto4(void *p, int64_t i, int64_t count, const float (&x)[4]) {  // values of the type
    if (count >= 4) {
        if constexpr (DT == HIDET_QMM_F32) {
            *reinterpret_cast<float4_at4_t *>(static_cast<float *>(p) + i) = float4_at4_t{x[0], x[1], x[2], x[3]};
        } else {
            half4_at2_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = DT == HIDET_QMM_F16 ? f32_to_f16_bits(x[e]) : f32_to_bf16_bits(x[e]);
            *reinterpret_cast<half4_at2_t *>(static_cast<uint16_t *>(p) + i) = v;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < count) store_from_f32<DT>(p, i + e, x[e]);
}
template <int QT>
__device__ __forceinline__ void store_codes_upto4(void *p, int64_t i, int64_t count, const uint32_t (&code)[4]) {  // low bits of each
    if constexpr (QT == HIDET_QMM_I8) {
        const uint32_t lo = __builtin_amdgcn_perm(code[1], code[0], 0x0c0c0400u), hi = __builtin_amdgcn_perm(code[3], code[2], 0x0c0c0400u);
        const uint32_t packed = lo | (hi << 16);
        int8_t *o = static_cast<int8_t *>(p) + i;
        if (count >= 4) {
            __builtin_memcpy(o, &packed, 4);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < count) o[e] = int8_t(packed >> (8 * e));
        }
    } else {
        int16_t *o = static_cast<int16_t *>(p) + i;
        if (count >= 4) {
            *reinterpret_cast<half4_at2_t *>(o) = half4_at2_t{uint16_t(code[0]), uint16_t(code[1]), uint16_t(code[2]), uint16_t(code[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < count) o[e] = int16_t(code[e]);
        }
    }
}
template <int QT>
__device__ __forceinline__ void load_codes_upto4(const void *p, int64_t i, int64_t count, float (&code)[4]) {
    if constexpr (QT == HIDET_QMM_I8) {
        uint32_t v = 0;
        const int8_t *q = static_cast<const int8_t *>(p) + i;
        if (count >= 4) {
            __builtin_memcpy(&v, q, 4);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < count) v |= uint32_t(uint8_t(q[e])) << (8 * e);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) code[e] = float(int8_t(v >> (8 * e)));
    } else {
        const int16_t *q = static_cast<const int16_t *>(p) + i;
#pragma unroll
        for (int e = 0; e < 4; ++e) code[e] = e < count ? float(q[e]) : 0.0f;
    }
}

// Maxima over the middle axis of [outer, R, inner], inner > 1 (strided reduction): 1024 / QUADS row lanes x QUADS column quads,
// 4 rows of 16 bytes (float32) in flight per thread. Block x = column block, y = row range, z = outer: the ranges of one
// column leave their maxima in rows of their own of `amax` [ranges, outer * inner], which the quantizing kernel takes
// together (one atomic per range and column instead wants the array cleared by a launch of its own). Bound by memory: K = 4096,
// N = 11008, float32 in 37 - 38 us = 4.8 TB/s, what a copy reaches (4-byte loads, 64 columns per workgroup, and the
// clearing launch in front: 40.6 us and 2 - 5 us).
constexpr int kAmaxThreads = 1024, kAmaxRows = 4;
template <int DT, int QUADS>
__global__ __launch_bounds__(kAmaxThreads) void amax_strided_kernel(const void *__restrict__ w, float *__restrict__ amax, int64_t R,
                                                                    int64_t inner, int64_t rows_per_range, int64_t nscale) {
    constexpr int kLanes = kAmaxThreads / QUADS;
    __shared__ float4_t red[kLanes][QUADS];
    const int tx = threadIdx.x % QUADS;
    const int ty = QUADS == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / QUADS) : threadIdx.x / QUADS;  // (64: a wave's row is a scalar)
    const int64_t col = int64_t(blockIdx.x) * (4 * QUADS) + 4 * tx;
    const int64_t o = blockIdx.z, count = inner - col;
    const int64_t r1 = min(R, (int64_t(blockIdx.y) + 1) * rows_per_range);
    float m[4] = {0.f, 0.f, 0.f, 0.f};
    if (count > 0) {
        const int64_t base = o * R * inner;
        int64_t r = int64_t(blockIdx.y) * rows_per_range + ty;
        for (; r + kLanes * (kAmaxRows - 1) < r1; r += kLanes * kAmaxRows) {
            float v[kAmaxRows][4];
#pragma unroll
            for (int i = 0; i < kAmaxRows; ++i) load_upto4<DT>(w, base + (r + kLanes * i) * inner + col, count, v[i]);
#pragma unroll
            for (int i = 0; i < kAmaxRows; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], fabsf(v[i][e]));
        }
        for (; r < r1; r += kLanes) {
            float v[4];
            load_upto4<DT>(w, base + r * inner + col, count, v);
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], fabsf(v[e]));
        }
    }
    red[ty][tx] = float4_t{m[0], m[1], m[2], m[3]};
    __syncthreads();
    if constexpr (kLanes > 16) {  // 16 rows of maxima are left to the first threads
        if (ty < 16) {
            for (int t = ty + 16; t < kLanes; t += 16)
#pragma unroll
                for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], red[t][tx][e]);
            red[ty][tx] = float4_t{m[0], m[1], m[2], m[3]};
        }
        __syncthreads();
    }
    if (ty == 0 && count > 0) {
#pragma unroll 4
        for (int t = 1; t < 16; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], red[t][tx][e]);
        store_upto4<HIDET_QMM_F32>(amax, int64_t(blockIdx.y) * nscale + o * inner + col, count, m);
    }
}

// The same for a short innermost axis (narrow_inner, at most 256): the threads of a workgroup take consecutive elements of
// whole rows, eight loads in flight each, so that a thread stays on one column and no lane is idle for want of columns. The
// maxima of the ranges form a tensor [outer, ranges, inner], which a second launch of this kernel takes together.
template <int DT>
__global__ __launch_bounds__(256) void amax_narrow_kernel(const void *__restrict__ w, float *__restrict__ amax, int64_t R, int64_t inner_,
                                                          int64_t rows_per_range) {
    __shared__ float red[256];
    const int t = threadIdx.x, inner = int(inner_), lanes = 256 / inner, span = lanes * inner;
    const int64_t o = blockIdx.z, r0 = int64_t(blockIdx.y) * rows_per_range;
    const int64_t base = (o * R + r0) * inner, count = (min(R, r0 + rows_per_range) - r0) * inner;
    float m = 0.0f;
    if (t < span) {
        int64_t i = t;
        for (; i + 7 * span < count; i += 8 * span) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = load_as_f32<DT>(w, base + i + j * span);
#pragma unroll
            for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
        }
        for (; i < count; i += span) m = fmaxf(m, fabsf(load_as_f32<DT>(w, base + i)));
    }
    red[t] = m;
    __syncthreads();
    int step = 1;
    while (2 * step < lanes) step *= 2;
    for (; step > 0; step >>= 1) {
        if (t < step * inner && t + step * inner < span) red[t] = fmaxf(red[t], red[t + step * inner]);
        __syncthreads();
    }
    if (t < inner) amax[(o * gridDim.y + blockIdx.y) * inner + t] = red[t];
}

// amax over the last axis of [outer, R] (inner == 1): one wave per row, 4 rows per block.
template <int DT>
__global__ __launch_bounds__(256) void amax_contig_kernel(const void *__restrict__ w, float *__restrict__ amax,
                                                          int64_t outer, int64_t R) {
    const int lane = threadIdx.x & 63;
    const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= outer) return;
    float m = 0.0f;
    for (int64_t r = lane * 4; r < R; r += 256) {
        float v[4];
        load_upto4<DT>(w, row * R + r, R - r, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(v[e]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) amax[row] = m;
}

typedef uint32_t uint2v_t __attribute__((ext_vector_type(2)));
// Four-element forms (numel a multiple of 4, 16-byte aligned input, 4-byte aligned codes). ONCE: non-temporal loads.
template <int DT, bool ONCE = false>
__device__ __forceinline__ void load4_as_f32(const void *p, int64_t i4, float (&x)[4]) {
    if (DT == HIDET_QMM_F32) {
        const float4_t *from = reinterpret_cast<const float4_t *>(p) + i4;
        const float4_t v = ONCE ? __builtin_nontemporal_load(from) : *from;
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
        const uint2v_t *from = reinterpret_cast<const uint2v_t *>(p) + i4;
        const uint2v_t v = ONCE ? __builtin_nontemporal_load(from) : *from;
        const uint16_t h[4] = {uint16_t(v.x), uint16_t(v.x >> 16), uint16_t(v.y), uint16_t(v.y >> 16)};
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = DT == HIDET_QMM_F16 ? f16_bits_to_f32(h[e]) : bf16_bits_to_f32(h[e]);
    }
}

// code = saturating_cast(round(rnd(w / scale))), scale = rnd(amax / qmax), rnd = round to w's dtype. `round` is what
// the reference's GPU lowering of round() does for the dtype: ties away from zero for float32 (roundf,
// python/hidet/ir/primitives/hip/math/float32.py:40), ties to even for float16 (hrint, hip/math/float16.py:42) and
// bfloat16 (hrint, cuda/math/bfloat16.py:29; the reference has no HIP bfloat16 math set). Its CPU half types round ties
// away instead (include/hidet/runtime/cpu/float16.h:747-750): a float16 quotient of exactly n + 0.5 - common, since
// float16 has a spacing of 1/16 between 64 and 128 - differs by one code between the two targets.
// (codes4 and scales4 above.)

// Columns of [outer, R, inner] quantized from their maxima (`ranges` <= kMaxRanges rows of them, amax_strided_kernel):
// kQuantLanes row lanes x 64 column quads. The workgroup puts its columns' maxima together, a thread works out the scales
// of its four columns once and takes TRIPS times TRIP rows, a trip's 16-byte loads in flight together (a single trip's go out before
// the maxima are read). Block x counts column blocks, then row blocks of kQuantLanes * TRIP * TRIPS; z = outer. Of a large matrix 64 rows per workgroup pay for
// the maxima and scales (16: 40 - 51 us); all eight loads of a
// thread at once cost the occupancy that hides them (16-bit types: 44 instead of 28 us). K = 4096, N = 11008: float32 35 - 36 us
// (the second read comes from the last-level cache: 6.3 TB/s), bfloat16 36 -> 28 us (the divisions).
constexpr int kQuantLanes = 8, kQuantTrip = 4, kQuantRows = 2 * kQuantLanes * kQuantTrip, kMaxRanges = 32;
template <int DT, int QT, int TRIP, int TRIPS>
__global__ __launch_bounds__(64 * kQuantLanes) void quantize_rows_kernel(const void *__restrict__ w, const float *__restrict__ amax, int ranges,
                                                                         int64_t nscale, void *__restrict__ q, void *__restrict__ scale,
                                                                         int64_t R, int64_t inner, uint32_t col_blocks) {
    __shared__ float4_t red[kQuantLanes][64];
    constexpr int kRows = kQuantLanes * TRIP * TRIPS;
    const int tx = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // a wave's row is a scalar
    const int64_t col = int64_t(blockIdx.x % col_blocks) * 256 + 4 * tx, row0 = int64_t(blockIdx.x / col_blocks) * kRows;
    const int64_t o = blockIdx.z, count = inner - col, r_end = min(R, row0 + kRows);
    int64_t r = row0 + ty;
    float x[TRIP][4];
    auto load = [&] {
#pragma unroll
        for (int j = 0; j < TRIP; ++j)
            if (count > 0 && r + kQuantLanes * j < r_end) load_upto4<DT>(w, (o * R + r + kQuantLanes * j) * inner + col, count, x[j]);
    };
    if constexpr (TRIPS == 1) load();
    float m[4] = {0.f, 0.f, 0.f, 0.f};
    if (count > 0) {
        for (int i = ty; i < ranges; i += kQuantLanes) {
            float v[4];
            load_upto4<HIDET_QMM_F32>(amax, i * nscale + o * inner + col, count, v);
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], v[e]);
        }
    }
    red[ty][tx] = float4_t{m[0], m[1], m[2], m[3]};
    __syncthreads();
#pragma unroll 4
    for (int t = 0; t < kQuantLanes; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], red[t][tx][e]);
    if (count <= 0) return;
    float s[4], inv[4];
    const bool fast = scales4<DT, QT>(m, s, inv);
    if (row0 == 0 && ty == 0) store_upto4<DT>(scale, o * inner + col, count, s);
    for (; r < r_end; r += kQuantLanes * TRIP) {
        if constexpr (TRIPS > 1) load();
#pragma unroll
        for (int j = 0; j < TRIP; ++j) {
            if (r + kQuantLanes * j >= r_end) break;
            uint32_t code[4];
            codes4<DT, QT>(x[j], s, inv, fast, code);
            store_codes_upto4<QT>(q, (o * R + r + kQuantLanes * j) * inner + col, count, code);
        }
        if constexpr (TRIPS == 1) break;
    }
}

// A weight of half of the last-level cache and more of which whole cache lines are read, and read once, passes that cache by, which then keeps what the next kernel reads and
// writes (4096 x 11008 float32, quantized and dequantized along rows 90.0 -> 74.3 us; int4 groups 40.4 -> 36.1). Smaller weights may lie in it. us, plain and non-temporal, three weights in
// turn (and weights from memory): along rows bfloat16 902 x 3712 4.5 and 5.3 (4.6 and 5.5), float16 1632 x 10624 14.4 and 17.6 (16.8 and 17.1), float32 1086 x 8640 9.4 and 10.6
// (10.7 and 10.6), 2032 x 10496 18.2 and 20.1 (19.8 and 20.1), but 1408 x 3648 6.5 and 6.2. int4, groups of 64: 3712 x 5760 18.7 and 20.8 (21.6 and 20.9), 896 x 4288 7.9 and 8.7
// (8.9 and 8.9), 3840 x 8896 31.8 and 30.1 (32.7 and 30.3). From 128 MiB on the same weight quantized again and again is the one case that plain loads serve better (float32 along rows 4096 x
// 10496 31.8 and 36.7, int4 34.3 and 38.5 of 4096 x 11008); three in turn 36.4 and 36.5, 40.1 and 37.6, and with the dequantization behind it the one weight too 80.4 and 69.2.
// quantize_meet_kernel is apart: it reads all that it holds this way (below).
constexpr int kNonTemporal = 2;
constexpr int64_t kReadOnceFrom = int64_t(128) << 20;  // bytes

// ---- maxima and codes in one pass over the weight ----------------------------------------------
//
// The two kernels above read the weight twice and are two launches. The ones here keep what they have read in registers: a workgroup of
// kStripThreads holds NV quads of columns per thread (and NL in LDS) between the maxima and the codes, rows beyond that are read again.

// A quad of columns as it lies in memory, at the alignment of one element; zeros past the end of the buffer, without a trip to memory.
template <int DT>
struct Quad {
    typedef uint4v_t type;
};
template <>
struct Quad<HIDET_QMM_F16> {
    typedef uint2v_t type;
};
template <>
struct Quad<HIDET_QMM_BF16> {
    typedef uint2v_t type;
};
template <int DT, bool ONCE = false>
__device__ __forceinline__ typename Quad<DT>::type load_quad(const __amdgpu_buffer_rsrc_t &from, int offset) {
    constexpr int kAux = ONCE ? kNonTemporal : 0;
    if constexpr (DT == HIDET_QMM_F32) return __builtin_bit_cast(uint4v_t, __builtin_amdgcn_raw_buffer_load_b128(from, offset, 0, kAux));
    else return __builtin_bit_cast(uint2v_t, __builtin_amdgcn_raw_buffer_load_b64(from, offset, 0, kAux));
}
template <int DT>
__device__ __forceinline__ void quad_to_f32(const typename Quad<DT>::type &v, float (&x)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (DT == HIDET_QMM_F32) x[e] = __uint_as_float(v[e]);
        else {
            const uint16_t h = uint16_t(v[e >> 1] >> (16 * (e & 1)));
            x[e] = DT == HIDET_QMM_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
        }
    }
}
template <int DT>
__device__ __forceinline__ void quad_max(float (&m)[4], const typename Quad<DT>::type &v) {
    float t[4];
    quad_to_f32<DT>(v, t);
#pragma unroll
    for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], fabsf(t[e]));
}
template <int DT, int QT>
__device__ __forceinline__ void store_quad_codes(const typename Quad<DT>::type &v, const float (&s)[4], const float (&inv)[4], bool fast, void *q) {
    float t[4];
    uint32_t code[4];
    quad_to_f32<DT>(v, t);
    codes4<DT, QT>(t, s, inv, fast, code);
    store_codes_upto4<QT>(q, 0, 4, code);
}
// The quads stay as they are in memory: the compiler would keep the unpacked values of the maxima for the codes.
template <int N, typename V>
__device__ __forceinline__ void keep_packed(V (&x)[N]) {
#pragma unroll
    for (int v = 0; v < N; ++v)
#pragma unroll
        for (int i = 0; i < int(sizeof(V) / 4); ++i) asm volatile("" : "+v"(x[v][i]));
}

// A strip of 4 CL columns over all rows of [R, inner] per workgroup, kStripThreads / CL rows at a time. Neighbouring strips share the cache
// lines of the codes, so an XCD has a run of them. The last quad of a row that is no multiple of four is moved back into the row: its lane and
// the one before store the same codes twice.
constexpr int kStripThreads = 512;
template <int DT, int QT, int CL, int NV, int WAVES>
__global__ __launch_bounds__(kStripThreads, WAVES) void quantize_strip_kernel(const char *__restrict__ w, char *__restrict__ q, void *__restrict__ scale, int R, int inner,
                                                                              int strips, int items, int per_xcd) {
    constexpr int kElement = DT == HIDET_QMM_F32 ? 4 : 2, kCode = QT == HIDET_QMM_I8 ? 1 : 2;
    constexpr int kLanes = kStripThreads / CL, kWaves = kStripThreads / 64, kBatch = DT == HIDET_QMM_F32 ? 4 : 8;
    typedef typename Quad<DT>::type V;
    __shared__ float4_t red[kWaves][CL];
    const int tid = threadIdx.x, tx = tid % CL, ty = tid / CL, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int item = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);
    if (item >= items || int(blockIdx.x >> 3) >= per_xcd) return;
    const int o = item / strips, place = ((item - o * strips) * CL + tx) * 4, col = min(place, inner - 4);
    const int row_bytes = inner * kElement, offset = ty * row_bytes + col * kElement;
    const int64_t step = int64_t(kLanes) * row_bytes, bytes = int64_t(R) * row_bytes;
    w += o * bytes;
    q += o * bytes / kElement * kCode;
    auto trip = [&](int v) {  // rows v kLanes and on
        const int64_t left = bytes - v * step;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w) + v * step, 0, left > 0 ? int(left) : 0, 0x00020000);
    };
    V x[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = load_quad<DT>(trip(v), offset);
    __builtin_amdgcn_sched_barrier(0);
    float m[4] = {0.f, 0.f, 0.f, 0.f};
    const int trips = (R + kLanes - 1) / kLanes;
    for (int v = NV; v < trips; v += kBatch) {
        V y[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) y[j] = load_quad<DT>(trip(v + j), offset);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) quad_max<DT>(m, y[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NV; ++v) quad_max<DT>(m, x[v]);
    keep_packed(x);
#pragma unroll
    for (int d = CL; d < 64; d <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], __shfl_xor(m[e], d));
    if ((tid & 63) < CL) red[wave][tx] = float4_t{m[0], m[1], m[2], m[3]};
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kWaves; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], red[t][tx][e]);
    if (place >= inner) return;
    float s[4], inv[4];
    const bool fast = scales4<DT, QT>(m, s, inv);
    if (ty == 0) store_upto4<DT>(scale, int64_t(o) * inner + col, 4, s);
    char *out = q + (int64_t(ty) * inner + col) * kCode;
    const int64_t out_step = int64_t(kLanes) * inner * kCode;
    auto emit = [&](int v, const V &quad) {
        if (v * kLanes + ty < R) store_quad_codes<DT, QT>(quad, s, inv, fast, out + v * out_step);
    };
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        emit(v, x[v]);
        __builtin_amdgcn_sched_barrier(0);  // (one quad's values at a time in registers)
    }
    for (int v = NV; v < trips; v += kBatch) {
        V y[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) y[j] = load_quad<DT>(trip(v + j), offset);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) emit(v + j, y[j]);
    }
}

// 256 columns x `share` rows per workgroup, all workgroups resident at once: the `ranges` workgroups of a column block (a group) leave their maxima in
// memory, count themselves in, and go on when all have. What a workgroup waits for is bounded: one that gives up reads its columns itself,
// so a launch ends with the right codes whatever else keeps workgroups of it from starting. Counters of a group lie on cache lines of their own (next to each other the atomics of all
// groups queue up: 2048 x 4096 float32 35 us instead of 16); the last to leave returns them to zero.
// What a workgroup holds passes the last-level cache by, at every size: against plain loads, 120 weights of 6 to 190 MB, that is 8 % faster from memory (7 with the dequantization behind
// it) and with three weights in turn the same (2); 2 % slower only where, besides, the codes and values go to the same memory each time.
constexpr int kMeetCounterWords = 64, kMeetGroups = kExchangeLostWord / (2 * kMeetCounterWords), kMeetSpins = 512;
template <int DT, int QT, int NV, int NL>
__global__ __launch_bounds__(kStripThreads, 4) void quantize_meet_kernel(const char *__restrict__ w, char *__restrict__ q, void *__restrict__ scale, float *partials,
                                                                         uint32_t *counters, int R, int inner, int col_blocks, int groups, int ranges, int share, int spins) {
    constexpr int kElement = DT == HIDET_QMM_F32 ? 4 : 2, kCode = QT == HIDET_QMM_I8 ? 1 : 2, kAgentScope = 1 << 4;  // sc1
    constexpr int kWaves = kStripThreads / 64, kBatch = 4, kHeld = kWaves * (NV + NL);
    typedef typename Quad<DT>::type V;
    static_assert(NL == 0 || sizeof(V) == 16, "16 bytes per lane go to LDS");
    extern __shared__ uint4 lds[];
    float4_t *red = reinterpret_cast<float4_t *>(lds + NL * kStripThreads);  // [kWaves][64], then the flag
    int *all_here = reinterpret_cast<int *>(red + kWaves * 64);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int range = int(blockIdx.x) / groups, group = int(blockIdx.x) - range * groups, o = group / col_blocks;
    const int place = (group - o * col_blocks) * 256 + 4 * lane, col = min(place, inner - 4), offset = col * kElement;
    const int first = range * share + wave, end = min(R, (range + 1) * share);
    const int64_t row_bytes = int64_t(inner) * kElement;
    w += int64_t(o) * R * row_bytes;
    q += int64_t(o) * R * inner * kCode;
    auto row = [&](int r, int past) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w) + r * row_bytes, 0, r < past ? int(row_bytes) : 0, 0x00020000); };
    V x[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = load_quad<DT, true>(row(first + kWaves * v, end), offset);
    if constexpr (NL > 0) {
#pragma unroll
        for (int l = 0; l < NL; ++l) buffer_load_to_lds_b128<kNonTemporal>(row(first + kWaves * (NV + l), end), lds + l * kStripThreads + wave * 64, offset, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    float m[4] = {0.f, 0.f, 0.f, 0.f};
    for (int r = first + kHeld; r < end; r += kWaves * kBatch) {
        V y[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) y[j] = load_quad<DT>(row(r + kWaves * j, end), offset);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) quad_max<DT>(m, y[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NV; ++v) quad_max<DT>(m, x[v]);
    keep_packed(x);
    const V *held = reinterpret_cast<const V *>(lds) + tid;  // what this lane's own loads put there
    if constexpr (NL > 0) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int l = 0; l < NL; ++l) quad_max<DT>(m, held[l * kStripThreads]);
    }
    auto waves_max = [&] {
#pragma unroll
        for (int t = 0; t < kWaves; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], red[t * 64 + lane][e]);
    };
    red[wave * 64 + lane] = float4_t{m[0], m[1], m[2], m[3]};
    __syncthreads();
    uint32_t *arrived = counters + 2 * kMeetCounterWords * group, *left = arrived + kMeetCounterWords;
    const __amdgpu_buffer_rsrc_t maxima = __builtin_amdgcn_make_buffer_rsrc(partials + int64_t(group) * ranges * 256, 0, ranges * 1024, 0x00020000);
    if (wave == 0) {
        waves_max();
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v_t, float4_t{m[0], m[1], m[2], m[3]}), maxima, (range * 64 + lane) * 16, 0, kAgentScope);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // acknowledged: they write through
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0) {
            uint32_t n = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
            for (int i = 0; i < spins && n < uint32_t(ranges); ++i) {
                __builtin_amdgcn_s_sleep(1);
                n = __hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            *all_here = n >= uint32_t(ranges);
        }
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    m[0] = m[1] = m[2] = m[3] = 0.0f;
    if (*all_here) {
        for (int i = wave; i < ranges; i += kWaves) {
            const float4_t v = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(maxima, (i * 64 + lane) * 16, 0, kAgentScope));
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], v[e]);
        }
    } else {
        for (int r = wave; r < R; r += kWaves) quad_max<DT>(m, load_quad<DT>(row(r, R), offset));
    }
    __syncthreads();  // (wave 0 may still be reading the workgroup's own maxima)
    red[wave * 64 + lane] = float4_t{m[0], m[1], m[2], m[3]};
    __syncthreads();
    waves_max();
    if (tid == 0 && __hip_atomic_fetch_add(left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == uint32_t(ranges)) {
        __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(left, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (place >= inner) return;
    float s[4], inv[4];
    const bool fast = scales4<DT, QT>(m, s, inv);
    if (range == 0 && wave == 0) store_upto4<DT>(scale, int64_t(o) * inner + col, 4, s);
    auto emit = [&](int r, const V &quad) {
        if (r < end) store_quad_codes<DT, QT>(quad, s, inv, fast, q + (int64_t(r) * inner + col) * kCode);
    };
    V y[kBatch];
    auto load_rest = [&](int r) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j) y[j] = load_quad<DT>(row(r + kWaves * j, end), offset);
    };
    load_rest(first + kHeld);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        emit(first + kWaves * v, x[v]);
        __builtin_amdgcn_sched_barrier(0);  // (one quad's values at a time in registers)
    }
    if constexpr (NL > 0) {
#pragma unroll
        for (int l = 0; l < NL; ++l) emit(first + kWaves * (NV + l), held[l * kStripThreads]);
    }
    for (int r = first + kHeld; r < end; r += kWaves * kBatch) {
#pragma unroll
        for (int j = 0; j < kBatch; ++j) emit(r + kWaves * j, y[j]);
        load_rest(r + kWaves * kBatch);
    }
}

// inner == 1, rows too long for a workgroup's registers: four (or fewer, at a row's end) elements per thread from the
// row's maximum. Block x counts blocks of 1024 elements within a row, y = row.
template <int DT, int QT>
__global__ __launch_bounds__(256) void quantize_long_row_kernel(const void *__restrict__ w, const float *__restrict__ amax, void *__restrict__ q,
                                                                void *__restrict__ scale, int64_t R, uint32_t blocks_per_row) {
    const int64_t row = blockIdx.x / blocks_per_row;
    const int64_t c = (int64_t(blockIdx.x % blocks_per_row) * 256 + threadIdx.x) * 4, count = R - c;
    if (count <= 0) return;
    const float a = amax[row];
    const float m[4] = {a, a, a, a};
    float s[4], inv[4], x[4];
    uint32_t code[4];
    const bool fast = scales4<DT, QT>(m, s, inv);
    if (c == 0) store_from_f32<DT>(scale, row, s[0]);
    load_upto4<DT>(w, row * R + c, count, x);
    codes4<DT, QT>(x, s, inv, fast, code);
    store_codes_upto4<QT>(q, row * R + c, count, code);
}

// inner == 1 (one scale per row, e.g. an embedding table): one workgroup per row keeps the whole row in registers
// between the amax pass and the quantization, so the tensor is read once. Rows of up to T * 4 * NV elements, a
// multiple of 4, 16-byte aligned. Same arithmetic as above.
template <int DT, int QT, int T, int NV, bool ONCE>
__global__ __launch_bounds__(T) void quantize_row_fused_kernel(const void *__restrict__ w, void *__restrict__ q,
                                                                 void *__restrict__ scale, int64_t R4) {
    __shared__ float red[T / 64];
    const int tid = threadIdx.x;
    const int64_t base4 = int64_t(blockIdx.x) * R4;
    float x[NV][4];
    float m = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t j = int64_t(v) * T + tid;
        x[v][0] = x[v][1] = x[v][2] = x[v][3] = 0.0f;
        if (j < R4) load4_as_f32<DT, ONCE>(w, base4 + j, x[v]);
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(x[v][e]));
    }
    m = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int i = 1; i < T / 64; ++i) m = fmaxf(m, red[i]);
    const float mm[4] = {m, m, m, m};
    float s[4], inv[4];
    const bool fast = scales4<DT, QT>(mm, s, inv);
    if (tid == 0) store_from_f32<DT>(scale, blockIdx.x, s[0]);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t j = int64_t(v) * T + tid;
        if (j >= R4) continue;
        uint32_t code[4];
        codes4<DT, QT>(x[v], s, inv, fast, code);
        store_codes_upto4<QT>(q, (base4 + j) * 4, 4, code);
    }
}

constexpr int kDequantRows = 32;
// Codes times scales. inner > 1: 256 threads = 4 row lanes x 64 column quads, a thread keeps its four columns' scales over
// kDequantRows / 4 rows (one index division per workgroup, where a thread per four elements pays two of 64 bits:
// bfloat16 4096 x 11008
// 35 -> 22 us, a row length that is no multiple of four 75 -> 31 us). Block x counts column blocks, then row blocks; z = outer.
template <int QT, int ST>
__global__ __launch_bounds__(256) void dequantize_rows_kernel(const void *__restrict__ q, const void *__restrict__ scale, void *__restrict__ w,
                                                              int64_t R, int64_t inner, uint32_t col_blocks) {
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t col = int64_t(blockIdx.x % col_blocks) * 256 + 4 * tx, row0 = int64_t(blockIdx.x / col_blocks) * kDequantRows;
    const int64_t o = blockIdx.z, count = inner - col;
    if (count <= 0) return;
    float s[4];
    load_upto4<ST>(scale, o * inner + col, count, s);
#pragma unroll
    for (int j = 0; j < kDequantRows / 4; ++j) {
        const int64_t r = row0 + 4 * j + ty;
        if (r >= R) break;
        const int64_t i = (o * R + r) * inner + col;
        float code[4], out[4];
        load_codes_upto4<QT>(q, i, count, code);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = round_to<ST>(code[e] * s[e]);
        store_upto4<ST>(w, i, count, out);
    }
}

// [outer, R, inner] with a short innermost axis, or more slices than a grid has layers: four consecutive elements
// per thread, each with the scale of its own column. The kernels above give a column quad to a lane, so of a row of 9
// elements (a 3 x 3 filter) they use 3 lanes in 64. Bound by memory and, where rows are no multiple of four, by the gathers of
// the scales. float32, element-wise kernels on 64-bit indexes -> these, us: quantize 4096 x 256 x 9 40.6 -> 28.7, 1000000 x 9 53 -> 30,
// 64 x 4096 x 32 49 -> 23, 1000000 x 64 202 -> 154; dequantize 19.1 -> 11.5, 19.0 -> 11.9, 11.6 -> 8.5, 64 -> 64.
template <typename F>
__device__ __forceinline__ void for_columns4(int64_t i, int64_t R, int64_t inner, F &&f) {  // f(e, column of the scales, row)
    int64_t row, o;
    if (((i | R | inner) >> 32) == 0) {
        row = uint32_t(i) / uint32_t(inner);
        o = uint32_t(row) / uint32_t(R);
    } else {
        row = i / inner;
        o = row / R;
    }
    int64_t r = row - o * R, c = i - row * inner;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f(e, o * inner + c, r);
        if (++c == inner) {
            c = 0;
            if (++r == R) r = 0, ++o;
        }
    }
}
// Entries of `p`, one per column, of the `count` elements from i on (four at most).
template <int DT>
__device__ __forceinline__ void load_columns4(const void *p, int64_t i, int64_t count, int64_t R, int64_t inner, float (&v)[4]) {
    if (inner % 4 == 0) {  // a quad lies in one row, and so does the last
        for_columns4(i, R, inner, [&](int e, int64_t column, int64_t) {
            if (e == 0) load_upto4<DT>(p, column, 4, v);
        });
        return;
    }
    for_columns4(i, R, inner, [&](int e, int64_t column, int64_t) { v[e] = e < count ? load_as_f32<DT>(p, column) : 0.0f; });
}
template <int DT, int QT>
__global__ __launch_bounds__(256) void quantize_flat_kernel(const void *__restrict__ w, const float *__restrict__ amax, void *__restrict__ q,
                                                            void *__restrict__ scale, int64_t R, int64_t inner, int64_t total) {
    const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4, count = total - i;
    if (count <= 0) return;
    float x[4], m[4], s[4], inv[4];
    load_upto4<DT>(w, i, count, x);
    load_columns4<HIDET_QMM_F32>(amax, i, count, R, inner, m);
    const bool fast = scales4<DT, QT>(m, s, inv);
    for_columns4(i, R, inner, [&](int e, int64_t column, int64_t r) {
        if (e < count && r == 0) store_from_f32<DT>(scale, column, s[e]);
    });
    uint32_t code[4];
    codes4<DT, QT>(x, s, inv, fast, code);
    store_codes_upto4<QT>(q, i, count, code);
}
template <int QT, int ST>
__global__ __launch_bounds__(256) void dequantize_flat_kernel(const void *__restrict__ q, const void *__restrict__ scale, void *__restrict__ w,
                                                              int64_t R, int64_t inner, int64_t total) {
    const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4, count = total - i;
    if (count <= 0) return;
    float code[4], s[4], out[4];
    if (ST == HIDET_QMM_F32 && inner % 4 == 0) {  // whole quads: no branch between the two loads
        load_codes_upto4<QT>(q, i, 4, code);
        for_columns4(i, R, inner, [&](int e, int64_t column, int64_t) {
            if (e == 0) load_upto4<ST>(scale, column, 4, s);
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = round_to<ST>(code[e] * s[e]);
        store_upto4<ST>(w, i, 4, out);
        return;
    }
    load_codes_upto4<QT>(q, i, count, code);
    load_columns4<ST>(scale, i, count, R, inner, s);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = round_to<ST>(code[e] * s[e]);
    store_upto4<ST>(w, i, count, out);
}

// inner == 1: one scale per row. Block x counts blocks of 4096 elements within a row, then rows.
template <int QT, int ST>
__global__ __launch_bounds__(256) void dequantize_long_row_kernel(const void *__restrict__ q, const void *__restrict__ scale, void *__restrict__ w,
                                                                  int64_t R, uint32_t blocks_per_row) {
    const int64_t row = blockIdx.x / blocks_per_row;
    const float s = load_as_f32<ST>(scale, row);
    const int64_t c0 = int64_t(blockIdx.x % blocks_per_row) * 4096 + threadIdx.x * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t c = c0 + j * 1024, count = R - c;
        if (count <= 0) break;
        float code[4], out[4];
        load_codes_upto4<QT>(q, row * R + c, count, code);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = round_to<ST>(code[e] * s);
        store_upto4<ST>(w, row * R + c, count, out);
    }
}

// Group-wise int4: grid (ceil(n / (4 CL)), k / group); 512 threads = 512 / CL row lanes x CL column quads.
// scale32 = amax / 7 and code = clamp(round_half_away(w / scale32), -7, 7) in float32; two codes per
// byte along n, low nibble first; the stored scale is scale32 rounded to the scale dtype.
//
// Bound by memory: 4 bytes read and half a byte written per weight. ROWS > 0 (a group of up to ROWS * 512 / CL rows): the
// workgroup keeps its columns of the group in registers between the maximum and the codes, so the weight is read once.
// Longer groups take narrower column blocks instead of more rows per thread: with 8 rows per thread (76 registers) three
// workgroups share a CU and one's loads run under another's codes (16 rows, two workgroups: 42.8 us).
// ROWS = 0, groups beyond that: the rows are read twice. K = 4096, N = 11008, groups of 128: 82 - 87 us with the group
// read twice in 8-byte loads, a division per weight and one-byte stores -> 38.3 us = 5.3 TB/s.
// ONCE (kReadOnceFrom): non-temporal loads, 4096 x 11008 40.4 -> 36.1 us = 5.6 TB/s.
template <int ST, int CL, int ROWS, bool ONCE = false>
__global__ __launch_bounds__(512, 6) void group_quantize_int4_kernel(const float *__restrict__ w, uint8_t *__restrict__ packed,
                                                                     void *__restrict__ scales, int64_t n, int group) {
    constexpr int LANES = 512 / CL;
    __shared__ float4_t red[LANES][CL];
    // a row's address is a scalar base (the wave's first row) and one per-lane offset for all rows
    const int tx = threadIdx.x % CL, ty = threadIdx.x / CL;
    const int sub = (threadIdx.x & 63) / CL, ty0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * (64 / CL);
    const int64_t b0 = int64_t(blockIdx.x) * (4 * CL), c0 = b0 + 4 * tx;
    const int64_t g = blockIdx.y;
    const int cols = c0 >= n ? 0 : (n - c0 >= 4 ? 4 : 2);  // n is even
    const float *base = w + g * group * n + b0;
    const int64_t lane_off = sub * n + 4 * tx;
    auto load = [&](int i) {  // row i * LANES + ty of the group
        float4_t v = {0.f, 0.f, 0.f, 0.f};
        const float *row = base + int64_t(i * LANES + ty0) * n;
        if (i * LANES + ty < group) {
            if (cols == 4) {
                const float4_at4_t *from = reinterpret_cast<const float4_at4_t *>(row + lane_off);
                v = ONCE ? __builtin_nontemporal_load(from) : *from;
            } else if (cols == 2) {
                v[0] = row[lane_off];
                v[1] = row[lane_off + 1];
            }
        }
        return v;
    };
    const int trips = (group + LANES - 1) / LANES;
    float4_t x[ROWS > 0 ? ROWS : 1];
    float4_t m = {0.f, 0.f, 0.f, 0.f};
    auto larger = [&](const float4_t &v) {
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = fmaxf(m[e], fabsf(v[e]));
    };
    if constexpr (ROWS > 0) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) x[i] = load(i);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) larger(x[i]);
    } else {
        for (int i = 0; i < trips; ++i) larger(load(i));
    }
    red[ty][tx] = m;
    __syncthreads();
#pragma unroll 2  // (the weights are in registers: no room for all of these at once)
    for (int t = 0; t < LANES; ++t) larger(red[t][tx]);
    if (cols == 0) return;
    float s[4], inv[4];
    bool fast = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        s[e] = m[e] / 7.0f;
        inv[e] = __builtin_amdgcn_rcpf(s[e]);
        fast = fast && reciprocal_is_precise(s[e]);
    }
    if (ty == 0) {
        for (int e = 0; e < cols; ++e) store_from_f32<ST>(scales, g * n + c0 + e, round_to<ST>(s[e]));
    }
    uint8_t *out = packed + ((g * group * n + b0) >> 1);  // n is even: every row starts on a byte
    auto emit = [&](int i, const float4_t &v) {
        if (i * LANES + ty >= group) return;
        const float x4[4] = {v[0], v[1], v[2], v[3]};
        uint32_t n4[4], code = 0;
        round_quotients_f32(x4, s, inv, fast, -7.0f, 7.0f, n4);
#pragma unroll
        for (int e = 0; e < 4; ++e) code |= (n4[e] & 0xFu) << (4 * e);
        uint8_t *o = out + ((int64_t(i * LANES + ty0) * n) >> 1) + (lane_off >> 1);
        if (cols == 4) __builtin_memcpy(o, &code, 2);
        else *o = uint8_t(code);
    };
    if constexpr (ROWS > 0) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) emit(i, x[i]);
    } else {
        for (int i = 0; i < trips; ++i) emit(i, load(i));
    }
}

// ---- per-tensor float8 e4m3 -------------------------------------------------------------------

// Elements i .. i + V - 1 (V = 16 bytes of the type) as they lie in memory, zero from `numel` on, at the alignment of one.
typedef uint32_t uint4_at4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t uint4_at2_t __attribute__((ext_vector_type(4), aligned(2)));
template <int DT>
__device__ __forceinline__ uint4v_t load_vector(const void *p, int64_t i, int64_t numel) {
    constexpr int V = DT == HIDET_QMM_F32 ? 4 : 8;
    uint4v_t v = {0u, 0u, 0u, 0u};
    if (i + V <= numel) {
        if constexpr (DT == HIDET_QMM_F32) v = *reinterpret_cast<const uint4_at4_t *>(static_cast<const uint32_t *>(p) + i);
        else v = *reinterpret_cast<const uint4_at2_t *>(static_cast<const uint16_t *>(p) + i);
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (i + e >= numel) continue;
            if constexpr (DT == HIDET_QMM_F32) v[e] = static_cast<const uint32_t *>(p)[i + e];
            else v[e >> 1] |= uint32_t(static_cast<const uint16_t *>(p)[i + e]) << (16 * (e & 1));
        }
    }
    return v;
}
template <int DT>
__device__ __forceinline__ float vector_element(const uint4v_t &v, int e) {
    if constexpr (DT == HIDET_QMM_F32) return __uint_as_float(v[e]);
    const uint16_t h = uint16_t(v[e >> 1] >> (16 * (e & 1)));
    return DT == HIDET_QMM_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
}
constexpr int kChunkLoads = 4, kChunkVectors = 256 * kChunkLoads;  // 16 KiB of 16-byte vectors: one trip of a workgroup
constexpr int kAmaxPartials = 1024;
// Vectors of 256 threads up to which a thread converts one of them (bfloat16, one and four: 512 x 4096 4.4 and 5.4 us, 2048 x 4096 5.9 and 6.1, 4096 x 8192 18.6 and 13.6).
constexpr int kFineChunks = 2048;

// Largest magnitude of each workgroup's share of a tensor, one float per workgroup (an atomic on a single word takes
// longer than the reads, and the word has to be cleared by a launch of its own).
template <int DT>
__global__ __launch_bounds__(256) void amax_all_kernel(const void *__restrict__ x, float *__restrict__ amax, int64_t numel, int64_t chunks) {
    constexpr int V = DT == HIDET_QMM_F32 ? 4 : 8;
    __shared__ float red[4];
    float m = 0.0f;
    for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        uint4v_t v[kChunkLoads];
#pragma unroll
        for (int j = 0; j < kChunkLoads; ++j) v[j] = load_vector<DT>(x, (c * kChunkVectors + j * 256 + threadIdx.x) * V, numel);
#pragma unroll
        for (int j = 0; j < kChunkLoads; ++j)
#pragma unroll
            for (int e = 0; e < V; ++e) m = fmaxf(m, fabsf(vector_element<DT>(v[j], e)));
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) amax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// e4m3 codes of four values: the quotient by the scale, clamped to +-448 (what saturation means for a format whose largest
// finite value is 448), converted by the hardware's round-to-nearest-even OCP conversion; NaN becomes NaN of the same sign.
__device__ __forceinline__ uint32_t e4m3_codes4_divided(const float (&x)[4], float s) {
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)  // (these two keep a NaN, where the median of three hides it)
        q[e] = s == 0.0f ? 0.0f : __builtin_elementwise_minimum(__builtin_elementwise_maximum(x[e] / s, -448.0f), 448.0f);
    uint32_t p = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    p = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], int(p), true);
#pragma unroll
    for (int e = 0; e < 4; ++e)  // (the conversion drops a NaN's sign)
        if (q[e] != q[e]) p = (p & ~(0xFFu << (8 * e))) | ((0x7Fu | ((__float_as_uint(q[e]) >> 24) & 0x80u)) << (8 * e));
    return p;
}

// The same without the division where its result provably converts alike; `fast`: the reciprocal of the scale is precise.
// float32: the product with the reciprocal, within 2^-22 of the quotient, converts alike unless a rounding boundary of the format lies
// between them; those have at most five significant bits, so a product whose low 19 bits are not within 8 of zero (or that is too
// small for any code but zero) needs no division. 448 is such a boundary and no quotient by a precise scale exceeds it by
// as much as 8 units in the last place, so only divided values need the clamp.
// 16-bit types: there that test fails for one element in 128 or so (448 / 2^j times a maximum of few bits, and often 3/4 of that),
// which sends nearly every wave through the division (4096 x 8192: 23 us, of which 10 for this). One correction with the remainder
// instead leaves Q (1 + h), |h| < 2^-45, rounded once. It differs from the rounded quotient Q only next to a midpoint of two
// float32 numbers, and matters only where one of those is a boundary B: where x = s T (1 + h) with T = B +- half a unit. With s = N 2^b,
// N of 24 bits, and B = beta 2^c, 16 <= beta < 32, x and s T differ by |J -+ N / 2^20| 2^(b+c) for an integer J, out of at most 2^29 2^(b+c): h would
// have to be below 2^-45, so N within 2^-16 of a multiple of 2^20. But N is (maximum / 7) times a power of two, rounded: the low bits of a
// multiple of 1/7 repeat with period three and never come near zero, and where seven divides the maximum N has at most nine bits, a
// multiple of 2^15; N / 2^20 is then an integer (x = s T would need 25 bits) or 2^-5 away from one. (tests/host/e4m3_quotients.cpp: every pair.)
template <int DT>
__device__ __forceinline__ uint32_t e4m3_codes4(const float (&x)[4], float s, float inv, bool fast) {
    float q[4];
    bool sure = fast;
    uint32_t nearest = 0xFFFFFFFFu;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        q[e] = x[e] * inv;
        if constexpr (DT == HIDET_QMM_F32) nearest = min(nearest, (__float_as_uint(fmaxf(fabsf(q[e]), 0x1.1p-12f + 0x1p-20f)) + 8u) & 0x7FFFFu);
        else q[e] = __builtin_fmaf(-__builtin_fmaf(q[e], s, -x[e]), inv, q[e]);  // (in this form a zero keeps its sign)
    }
    if constexpr (DT == HIDET_QMM_F32) sure = sure && nearest > 16u;
    sure = sure && !(__builtin_isunordered(q[0], q[1]) || __builtin_isunordered(q[2], q[3]));
    uint32_t p = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    p = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], int(p), true);
    if (__builtin_expect(!sure, 0)) p = e4m3_codes4_divided(x, s);
    return p;
}

// Small tensors (the activations of a decode step), up to 65536 elements, in one launch: a workgroup of 1024 threads looks at
// the whole tensor for its maximum and converts 4096 elements of it. One workgroup that converted all of it was bound by its
// vector ALU (bfloat16, 65536 elements 10.5 us, the two launches of larger tensors 7); looking at everything 16 times costs little
// beside that. What bounds it is the launch and code that comes from memory line by line, so the loops stay rolled up. Same
// arithmetic as fp8_quantize_kernel.
template <int DT>
__global__ __launch_bounds__(1024) void fp8_quantize_small_kernel(const void *__restrict__ x, uint32_t *__restrict__ codes,
                                                                  float *__restrict__ scale, int numel4) {
    __shared__ float red[16];
    const int tid = threadIdx.x, own = blockIdx.x * 1024 + tid, last = numel4 - 1;
    if (numel4 == 0) {
        if (tid == 0) *scale = 0.0f;
        return;
    }
    float mine[4];
    load4_as_f32<DT>(x, min(own, last), mine);
    float m = 0.0f;
#pragma unroll 1
    for (int j = tid; j < numel4; j += 4096) {
        float v[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) load4_as_f32<DT>(x, min(j + i * 1024, last), v[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(v[i][e]));
    }
    m = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int wv = 1; wv < 16; ++wv) m = fmaxf(m, red[wv]);
    const float s = m / 448.0f, inv = __builtin_amdgcn_rcpf(s);
    const bool fast = reciprocal_is_precise(s);
    if (own == 0) *scale = s;
    if (own < numel4) codes[own] = e4m3_codes4<DT>(mine, s, inv, fast);
}

// LOADS * 4 KiB per workgroup. The loads go out first; the workgroups' maxima (amax_all_kernel) are put together
// while they are under way. Chunks of 16 KiB are taken from the end of the tensor, where the maximum pass read last, each on the
// XCD that read it then: what is still in that L2 does not come from memory again. 4096 x 8192
// bfloat16: maxima 11 us (15.4 with atomics, + a clearing launch), codes 14 us (13 with no arithmetic at all). A tensor of which one
// vector per thread already fills the chip takes that: what bounds it is the launch and the code, which comes from memory line by line (4 -> 1
// vectors: 64 x 4096 5.6 -> 2.8 us, 512 x 4096 5.2 -> 4.0).
template <int DT, int LOADS>
__global__ __launch_bounds__(256) void fp8_quantize_kernel(const void *__restrict__ x, const float *__restrict__ amax, int partials,
                                                           uint8_t *__restrict__ codes, float *__restrict__ scale, int64_t numel, int64_t chunks8) {
    constexpr int V = DT == HIDET_QMM_F32 ? 4 : 8;
    __shared__ float red[4];
    const int64_t c = (chunks8 - 1 - int64_t(blockIdx.x >> 3)) * 8 + (blockIdx.x & 7);
    uint4v_t v[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) v[j] = load_vector<DT>(x, (c * (256 * LOADS) + j * 256 + threadIdx.x) * V, numel);
    float m = 0.0f;
    {
        float a[kAmaxPartials / 256];
#pragma unroll
        for (int i = 0; i < kAmaxPartials / 256; ++i) a[i] = amax[min(int(threadIdx.x) + i * 256, partials - 1)];
#pragma unroll
        for (int i = 0; i < kAmaxPartials / 256; ++i) m = fmaxf(m, a[i]);
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float s = m / 448.0f, inv = __builtin_amdgcn_rcpf(s);
    const bool fast = reciprocal_is_precise(s);
    if (blockIdx.x == 0 && threadIdx.x == 0) *scale = s;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int64_t i = (c * (256 * LOADS) + j * 256 + threadIdx.x) * V;
        if (i >= numel) continue;
        uint32_t out[V / 4];
#pragma unroll
        for (int h = 0; h < V / 4; ++h) {
            float t[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = vector_element<DT>(v[j], 4 * h + e);
            out[h] = e4m3_codes4<DT>(t, s, inv, fast);
        }
        if (i + V <= numel) {
            __builtin_memcpy(codes + i, out, V);
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (i + e < numel) codes[i + e] = uint8_t(out[e >> 2] >> (8 * (e & 3)));
        }
    }
}

// Rows of which the quantizing column-quad kernel would use less than three eighths of a wave's lanes: at 64 the flat kernel is the
// faster one for every type, at 96 float32 quantizes slower in it (2048 x 128 x 96 48.5 -> 52.5 us, bfloat16 52.0 -> 46.4).
inline bool narrow_inner(int64_t inner) { return inner < 96; }
constexpr int64_t kNarrowGroups = 1024;

// Elements of a workgroup's share of the maxima from which more than kMaxRanges row ranges pay for the launch that puts them
// together (float32, kMaxRanges -> more: 16384 x 128, 32768 elements, 12.0 -> 13.2 us; 65536 x 128, 131072 elements, 30.4 -> 20.6).
constexpr int64_t kCombineFrom = 65536;

// One pass over the weight where the matrix is of a size for it; false: nothing was launched.
//
// Strips where a CU's strip is short: 8, 16 or 32 columns, the fewest that one round of the chip covers the matrix with, up to the rows from which
// the other kernel is as fast (a thread holds 32 registers of quads; rows beyond those it holds are read twice). Two launches -> strips, us: float32 600 x 800
// 6.9 -> 4.0, 1024 x 1024 7.3 -> 5.0, 1024 x 4096 12.3 -> 8.7, 512 x 8192 11.5 -> 7.8; bfloat16 512 x 8192 10.5 -> 6.7, 1448 x 4096 12.9 -> 9.9, 1500 x 2501 12.9 -> 9.5.
// At their limits, strips and the other kernel: float32 1448 x 1024 8.5 and 8.5, 2048 x 4096 16.1 and 15.7, 1024 x 8192 14.1 and 14.4, 512 / 724 x 11008 10.9 / 15.6 and
// 12.1 / 14.7; bfloat16 2048 x 2048 11.5 and 9.5, 1448 x 8192 14.3 and 14.5, 1024 / 1448 x 11008 15.0 / 21.6 and 15.2 / 18.3.
//
// Above, workgroups that meet, all resident: two per CU, of 64 or 128 rows at least (more workgroups cost more in the meeting than they save: float32 2048 x 2048 with
// 16 / 32 / 64 rows 14.3 / 14.3 / 11.3), 64 to a column block at most, with as few quads held as the rows need (code that is not needed comes from memory all the
// same: bfloat16 2048 x 2048, 16 / 32 quads 9.5 / 11.1). Two launches -> these, us: float32 4096 x 11008 74 -> 58, 3000 x 6400 35 -> 27, 2048 x 11008 40.5 -> 31, 4096 x 4096 31 -> 26.6;
// bfloat16 4096 x 11008 50 -> 38, 4096 x 2048 15.6 -> 13.0. float32 of up to 1024 columns and less than 12 MB stays with two launches (2048 x 1024 9.5 and
// 10.1, 4096 x 512 10.3 and 11.0), and so do matrices of which the workgroups would hold less than a quarter or that are too narrow to fill the chip
// (bfloat16 65536 x 512 40 and 57).
template <int DT, typename F>
bool quantize_in_one_pass(F &&go, const void *w, void *wq, void *scale, int64_t outer, int64_t reduce, int64_t inner, const Workspace &ws) {
    using std::integral_constant;
    constexpr int kElement = DT == HIDET_QMM_F32 ? 4 : 2, kWide = 4 / kElement;  // kWide: quads of a register quad
    const int64_t cus = std::max(1, device_cus()), row_bytes = inner * kElement;
    if (reduce * row_bytes >= (int64_t(1) << 31) || row_bytes >= (int64_t(1) << 23) || outer > cus) return false;
    const char *from = static_cast<const char *>(w);
    char *to = static_cast<char *>(wq);
    auto strips = [&](auto cl, auto nv, auto waves) {
        constexpr int CL = decltype(cl)::value, NV = decltype(nv)::value, WAVES = decltype(waves)::value;
        const int64_t per_slice = cdiv(inner, 4 * CL), items = outer * per_slice, per_xcd = cdiv(items, 8);
        go(quantize_strip_kernel<DT, HIDET_QMM_I8, CL, NV, WAVES>, quantize_strip_kernel<DT, HIDET_QMM_I16, CL, NV, WAVES>, dim3(uint32_t(8 * per_xcd)), kStripThreads, 0,
           from, to, scale, int(reduce), int(inner), int(per_slice), int(items), int(per_xcd));
        return true;
    };
    auto one_round = [&](int columns) { return outer * cdiv(inner, columns) <= cus; };
    const bool f32 = DT == HIDET_QMM_F32;
    if (one_round(8)) {
        if (reduce <= (!f32 && inner <= 1024 ? 2048 : 1536)) return strips(integral_constant<int, 2>(), integral_constant<int, 4 * kWide>(), integral_constant<int, 8>());
    } else if (one_round(16)) {
        if (reduce <= (f32 ? 2048 : 1536)) return strips(integral_constant<int, 4>(), integral_constant<int, 8 * kWide>(), integral_constant<int, 6>());
    } else if (outer * cdiv(inner, 32) <= 2 * cus) {
        if (reduce <= (one_round(32) ? (f32 ? 1024 : 1536) : (f32 ? 640 : 1024))) return strips(integral_constant<int, 8>(), integral_constant<int, 8 * kWide>(), integral_constant<int, 6>());
    }
    const int64_t col_blocks = cdiv(inner, 256), groups = outer * col_blocks;
    if (ws.counters == nullptr || groups > kMeetGroups || (f32 && inner <= 1024 && outer * reduce * row_bytes < (12 << 20))) return false;
    const int64_t ranges_most = std::min<int64_t>(64, 2 * cus / groups);
    if (ranges_most < 2) return false;
    const int64_t least = f32 && reduce <= 2048 ? 64 : 128, share = cdiv(std::max(least, cdiv(reduce, ranges_most)), 8) * 8, ranges = cdiv(reduce, share);
    if (ws.scratch_bytes < groups * ranges * 1024 || (share > 256 && groups * ranges < cus)) return false;
    auto meet = [&](auto nv, auto nl) {
        constexpr int NV = decltype(nv)::value, NL = decltype(nl)::value, kLds = NL * kStripThreads * 16 + kStripThreads * 16 + 16;
        if (share > 4 * 8 * (NV + NL)) return false;
        allow_dynamic_lds(reinterpret_cast<const void *>(quantize_meet_kernel<DT, HIDET_QMM_I8, NV, NL>), kLds);
        allow_dynamic_lds(reinterpret_cast<const void *>(quantize_meet_kernel<DT, HIDET_QMM_I16, NV, NL>), kLds);
        go(quantize_meet_kernel<DT, HIDET_QMM_I8, NV, NL>, quantize_meet_kernel<DT, HIDET_QMM_I16, NV, NL>, dim3(uint32_t(groups * ranges)), kStripThreads, kLds, from, to, scale,
           reinterpret_cast<float *>(ws.scratch), ws.counters, int(reduce), int(inner), int(col_blocks), int(groups), int(ranges), int(share),
           std::min(kMeetSpins, exchange_spin_limit().load(std::memory_order_relaxed)));
        return true;
    };
    if (share <= 64 * kWide) return meet(integral_constant<int, 8 * kWide>(), integral_constant<int, 0>());
    if (share <= 128 * kWide) return meet(integral_constant<int, 16 * kWide>(), integral_constant<int, 0>());
    return meet(integral_constant<int, 20 * kWide>(), integral_constant<int, f32 ? 8 : 0>());
}

// The quantizer's launches for [outer, reduce, inner], no extent zero, outer at most quantize_slices_most(reduce, inner).
template <int DT>
void quantize_slices(const void *w, void *wq, void *scale, int64_t outer, int64_t reduce, int64_t inner, int q_dtype, const Workspace &ws, hipStream_t stream) {
    float *amax = reinterpret_cast<float *>(ws.scratch);
    const int64_t total = outer * reduce * inner, nscale = outer * inner;
    const int esize = DT == HIDET_QMM_F32 ? 4 : 2, qsize = q_dtype == HIDET_QMM_I8 ? 1 : 2;
    auto go_lds = [&](auto i8, auto i16, dim3 grid, int threads, size_t lds, auto... args) {
        if (q_dtype == HIDET_QMM_I8) launch(i8, grid, dim3(threads), lds, stream, args...);
        else launch(i16, grid, dim3(threads), lds, stream, args...);
    };
    auto go = [&](auto i8, auto i16, dim3 grid, int threads, auto... args) { go_lds(i8, i16, grid, threads, 0, args...); };
    if (inner == 1) {
        // rows that fit a workgroup's registers: one pass
        if (reduce % 4 == 0 && reduce <= 4 * 4 * 1024 && aligned(w, 4 * esize) && aligned(wq, 4 * qsize)) {
            const dim3 grid{uint32_t(outer)};
            const bool once = total * esize >= kReadOnceFrom;
            auto run = [&](auto threads, auto vectors) {
                constexpr int T = decltype(threads)::value, NV = decltype(vectors)::value;
                if (once) go(quantize_row_fused_kernel<DT, HIDET_QMM_I8, T, NV, true>, quantize_row_fused_kernel<DT, HIDET_QMM_I16, T, NV, true>, grid, T, w, wq, scale, reduce / 4);
                else go(quantize_row_fused_kernel<DT, HIDET_QMM_I8, T, NV, false>, quantize_row_fused_kernel<DT, HIDET_QMM_I16, T, NV, false>, grid, T, w, wq, scale, reduce / 4);
            };
            using std::integral_constant;
            // (four quads per thread: sixteen of 256 threads are code that comes from memory line by line; 4096 x 11008 bfloat16 40 -> 33.5 us,
            // 512 x 11008 10.2 -> 7.0, 1024 x 6144 9.6 -> 7.3; float32 56.8 -> 50, 8.2 -> 8.0, 10.8 -> 8.6)
            if (reduce <= 4 * 4 * 256) run(integral_constant<int, 256>(), integral_constant<int, 4>());
            else if (reduce <= 4 * 4 * 512) run(integral_constant<int, 512>(), integral_constant<int, 4>());
            else run(integral_constant<int, 1024>(), integral_constant<int, 4>());
            return;
        }
        launch(amax_contig_kernel<DT>, dim3(cdiv(outer, 4)), dim3(256), 0, stream, w, amax, outer, reduce);
        const int64_t blocks = cdiv(reduce, 1024);
        go(quantize_long_row_kernel<DT, HIDET_QMM_I8>, quantize_long_row_kernel<DT, HIDET_QMM_I16>, dim3(uint32_t(blocks * outer)), 256, w, amax, wq, scale,
           reduce, uint32_t(blocks));
        return;
    }
    const int64_t col_blocks = cdiv(inner, 256), row_blocks = cdiv(reduce, kQuantRows);
    QMM_CHECK(col_blocks * row_blocks < (int64_t(1) << 31), "tensor too large for one launch");
    const int64_t spare = ws.scratch_bytes / (nscale * 4) - 1;  // rows of maxima the scratch memory holds beside the final ones
    float *partials = amax + nscale;
    auto quantize = [&](int ranges) {
        auto run = [&](auto i8, auto i16, int64_t rows) {
            go(i8, i16, dim3(uint32_t(col_blocks * cdiv(reduce, rows)), 1, uint32_t(outer)), 64 * kQuantLanes, w, amax, ranges, nscale, wq, scale, reduce, inner,
               uint32_t(col_blocks));
        };
        // Small matrices: more workgroups, each a shorter chain with its loads in front of the maxima, until what every workgroup
        // spends on maxima and scales costs more (16, 32 and 64 rows, float32: 600 x 600 3.9, 4.4, 5.4 us; 1024 x 1024 4.3, 4.8, 5.8; 2048 x 4096
        // 9.8, 9.0, 8.8; bfloat16: 1500 x 2432 7.0, 6.4, 8.4; 4096 x 4096 17.6, 14.5, 12.7).
        const int64_t groups = col_blocks * row_blocks * outer;
        if (groups <= 128) run(quantize_rows_kernel<DT, HIDET_QMM_I8, 2, 1>, quantize_rows_kernel<DT, HIDET_QMM_I16, 2, 1>, 2 * kQuantLanes);
        else if (groups <= 384) run(quantize_rows_kernel<DT, HIDET_QMM_I8, 4, 1>, quantize_rows_kernel<DT, HIDET_QMM_I16, 4, 1>, 4 * kQuantLanes);
        else run(quantize_rows_kernel<DT, HIDET_QMM_I8, kQuantTrip, 2>, quantize_rows_kernel<DT, HIDET_QMM_I16, kQuantTrip, 2>, kQuantRows);
    };
    if (narrow_inner(inner)) {
        // Four workgroups per CU, of 2048 elements at least (1000000 x 9, float32: 32 workgroups and the column-quad kernel 216 us, these
        // and the flat one 30).
        int64_t ranges = std::min<int64_t>({kNarrowGroups / std::min<int64_t>(kNarrowGroups, outer), reduce * inner / 2048, spare});
        const int64_t rows_per_range = cdiv(reduce, std::max<int64_t>(1, ranges));
        ranges = cdiv(reduce, rows_per_range);
        launch(amax_narrow_kernel<DT>, dim3(1, uint32_t(ranges), uint32_t(outer)), dim3(256), 0, stream, w, ranges > 1 ? partials : amax, reduce, inner, rows_per_range);
        if (ranges > 1) launch(amax_narrow_kernel<HIDET_QMM_F32>, dim3(1, 1, uint32_t(outer)), dim3(256), 0, stream, partials, amax, ranges, inner, ranges);
        if (cdiv(total, 1024) < (int64_t(1) << 24)) {
            go(quantize_flat_kernel<DT, HIDET_QMM_I8>, quantize_flat_kernel<DT, HIDET_QMM_I16>, dim3(uint32_t(cdiv(total, 1024))), 256, w, amax, wq, scale, reduce,
               inner, total);
            return;
        }
        quantize(1);
        return;
    }
    if (quantize_in_one_pass<DT>(go_lds, w, wq, scale, outer, reduce, inner, ws)) return;
    // Workgroups of 256 columns where 16 row ranges of them are two workgroups per CU, else of 64, which need a quarter of the
    // ranges (float32, 256 -> 64: 4096 x 4096 35.3 -> 29.4 us, 16384 x 1024 42.8 -> 34.8, 65536 x 1024 150 -> 122, 65536 x 512 103 -> 56, but 16384 x 4096 106 -> 110;
    // bfloat16 65536 x 1024 120 -> 82). Ranges of 64 (128) rows at least, as many as two workgroups per CU take and the scratch memory
    // holds maxima of. Up to kMaxRanges of them are put together by the quantizing kernel; more, which a launch of its own puts together,
    // where they take that from the maxima's time.
    // (Rows that do not start on whole cache lines give short segments away: bfloat16 960 x 6410 26.3 us with 256, 29.5 with 64.)
    const int64_t blocks = col_blocks * outer;
    const bool wide = blocks >= 32 || (blocks >= 16 && inner * esize % 64 != 0);
    const int64_t amax_blocks = wide ? col_blocks : cdiv(inner, 64), groups = amax_blocks * outer;
    int64_t ranges = std::min(512 / std::min<int64_t>(512, groups), cdiv(reduce, wide ? 64 : 128));
    if (ranges > kMaxRanges && total / (kMaxRanges * groups) < kCombineFrom) ranges = kMaxRanges;
    ranges = std::max<int64_t>(1, std::min(ranges, ranges > kMaxRanges ? spare : spare + 1));
    const bool combine = ranges > kMaxRanges;
    const dim3 grid{uint32_t(amax_blocks), uint32_t(ranges), uint32_t(outer)};
    if (wide) launch(amax_strided_kernel<DT, 64>, grid, dim3(kAmaxThreads), 0, stream, w, combine ? partials : amax, reduce, inner, cdiv(reduce, ranges), nscale);
    else launch(amax_strided_kernel<DT, 16>, grid, dim3(kAmaxThreads), 0, stream, w, combine ? partials : amax, reduce, inner, cdiv(reduce, ranges), nscale);
    if (combine) {
        launch(amax_strided_kernel<HIDET_QMM_F32, 16>, dim3(uint32_t(cdiv(nscale, 64))), dim3(kAmaxThreads), 0, stream, partials, amax, ranges, nscale, ranges, nscale);
        ranges = 1;
    }
    quantize(int(ranges));
}
// Slices of a launch: a grid has 65535 layers, and 2^32 threads along x.
inline int64_t quantize_slices_most(int64_t reduce, int64_t inner) {
    return inner > 1 ? 65535 : std::max<int64_t>(1, ((int64_t(1) << 24) - 1) / cdiv(reduce, 1024));
}

template <typename F>
void dispatch_float(int dt, F &&f) {
    switch (dt) {
        case HIDET_QMM_F32: f(std::integral_constant<int, HIDET_QMM_F32>()); break;
        case HIDET_QMM_F16: f(std::integral_constant<int, HIDET_QMM_F16>()); break;
        case HIDET_QMM_BF16: f(std::integral_constant<int, HIDET_QMM_BF16>()); break;
        default: QMM_FAIL("expected a float32, float16 or bfloat16 dtype code, got " << dt);
    }
}

}  // namespace
}  // namespace qmm

using namespace qmm;

HIDET_API void hidet_symmetric_quantize(const void *w, void *wq, void *scale, int64_t outer, int64_t reduce,
                                        int64_t inner, int w_dtype, int q_dtype, void *workspace,
                                        int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(q_dtype == HIDET_QMM_I8 || q_dtype == HIDET_QMM_I16, "quant_type must be int8 or int16, got code " << q_dtype);
    QMM_CHECK(outer >= 0 && reduce >= 0 && inner >= 0, "negative extent");
    const int64_t total = outer * reduce * inner;
    const int64_t nscale = outer * inner;
    if (nscale == 0) return;
    QMM_CHECK(scale && (total == 0 || (w && wq)), "null tensor pointer");
    QMM_CHECK(inner < (int64_t(1) << 31) * 64, "extent too large");
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    QMM_CHECK(ws.scratch_bytes >= nscale * 4, "workspace too small: its scratch part (three quarters of what follows the first 64 KiB) must hold "
                                                  << nscale * 4 << " bytes, got a workspace of " << workspace_bytes);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    dispatch_float(w_dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        const int esize = DT == HIDET_QMM_F32 ? 4 : 2, qsize = q_dtype == HIDET_QMM_I8 ? 1 : 2;
        QMM_CHECK(aligned(w, esize) && aligned(wq, qsize) && aligned(scale, esize), "a tensor is not aligned to its element type");
        if (total == 0) {  // no elements (reduce is 0): the scales still have to be written
            if (DT == HIDET_QMM_F32) launch_aux(zero_kernel<uint32_t>, dim3(cdiv(nscale, 256)), dim3(256), 0, stream, static_cast<uint32_t *>(scale), nscale);
            else launch_aux(zero_kernel<uint16_t>, dim3(cdiv(nscale, 256)), dim3(256), 0, stream, static_cast<uint16_t *>(scale), nscale);
            return;
        }
        const int64_t step = quantize_slices_most(reduce, inner);
        for (int64_t o = 0; o < outer; o += step)  // (one launch after the other: they share the scratch memory)
            quantize_slices<DT>(static_cast<const char *>(w) + o * reduce * inner * esize, static_cast<char *>(wq) + o * reduce * inner * qsize,
                                static_cast<char *>(scale) + o * inner * esize, std::min(step, outer - o), reduce, inner, q_dtype, ws, stream);
    });
    QMM_ENTRY_END
}

HIDET_API void hidet_symmetric_dequantize(const void *wq, const void *scale, void *w, int64_t outer, int64_t reduce,
                                          int64_t inner, int q_dtype, int s_dtype, void *stream_) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(q_dtype == HIDET_QMM_I8 || q_dtype == HIDET_QMM_I16, "quantized dtype must be int8 or int16, got code " << q_dtype);
    const int64_t total = outer * reduce * inner;
    if (total == 0) return;
    QMM_CHECK(w && wq && scale, "null tensor pointer");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    dispatch_float(s_dtype, [&](auto dt) {
        constexpr int ST = decltype(dt)::value;
        const int esize = ST == HIDET_QMM_F32 ? 4 : 2, qsize = q_dtype == HIDET_QMM_I8 ? 1 : 2;
        QMM_CHECK(aligned(w, esize) && aligned(wq, qsize) && aligned(scale, esize), "a tensor is not aligned to its element type");
        if (inner == 1) {
            const int64_t blocks = cdiv(reduce, 4096);
            QMM_CHECK(blocks * outer < (int64_t(1) << 31), "tensor too large for one launch");
            const dim3 grid{uint32_t(blocks * outer)};
            if (q_dtype == HIDET_QMM_I8) launch(dequantize_long_row_kernel<HIDET_QMM_I8, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, uint32_t(blocks));
            else launch(dequantize_long_row_kernel<HIDET_QMM_I16, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, uint32_t(blocks));
            return;
        }
        // The kernel that gives a column quad to a lane where nine tenths of its lanes have one and there are workgroups enough: a
        // thread's eight rows are a chain, in float32 for four rounds of the chip's at a time. us, flat against that: float32 400000 x 192 76 and 77, 200000 x 384
        // 76 and 90, 4096 x 4096 13.5 and 16.2, 250000 x 256 64 and 55, 4096 x 11008 42 and 37; bfloat16 500000 x 128 50 and 64,
        // 200000 x 320 50 and 59, 250000 x 256 50 and 39, 4096 x 4096 13.6 and 9.6, 2048 x 4096 8.2 and 7.7, 1500 x 2432 4.9 and 5.4,
        // 1024 x 1024 2.8 and 5.0.
        const int64_t lanes = cdiv(inner, 256) * 256, groups = cdiv(inner, 256) * cdiv(reduce, kDequantRows) * outer;
        if (outer > 65535 || ((inner * 10 < lanes * 9 || (inner % 4 == 0 && groups < (ST == HIDET_QMM_F32 ? 4096 : 512))) && cdiv(total, 1024) < (int64_t(1) << 24))) {
            QMM_CHECK(cdiv(total, 1024) < (int64_t(1) << 31), "tensor too large for one launch");
            const dim3 grid{uint32_t(cdiv(total, 1024))};
            if (q_dtype == HIDET_QMM_I8) launch(dequantize_flat_kernel<HIDET_QMM_I8, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, inner, total);
            else launch(dequantize_flat_kernel<HIDET_QMM_I16, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, inner, total);
            return;
        }
        const int64_t col_blocks = cdiv(inner, 256), row_blocks = cdiv(reduce, kDequantRows);
        QMM_CHECK(col_blocks * row_blocks < (int64_t(1) << 31), "tensor too large for one launch");
        const dim3 grid(uint32_t(col_blocks * row_blocks), 1, uint32_t(outer));
        if (q_dtype == HIDET_QMM_I8) launch(dequantize_rows_kernel<HIDET_QMM_I8, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, inner, uint32_t(col_blocks));
        else launch(dequantize_rows_kernel<HIDET_QMM_I16, ST>, grid, dim3(256), 0, stream, wq, scale, w, reduce, inner, uint32_t(col_blocks));
    });
    QMM_ENTRY_END
}

HIDET_API void hidet_group_quantize_int4(const void *w, void *packed, void *scales, int64_t k, int64_t n, int group_size,
                                         int w_dtype, int s_dtype, void *stream_) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(w_dtype == HIDET_QMM_F32, "group_quantize_int4 expects float32 weights, got dtype code " << w_dtype);
    QMM_CHECK(group_size > 0 && k % group_size == 0, "K (" << k << ") must be a multiple of the group size (" << group_size << ")");
    QMM_CHECK(n % 2 == 0, "N (" << n << ") must be even: two codes are packed per byte");
    if (k == 0 || n == 0) return;
    QMM_CHECK(w && packed && scales, "null tensor pointer");
    QMM_CHECK(aligned(w, 8), "weight pointer must be 8-byte aligned");
    QMM_CHECK(k / group_size <= 65535, "too many groups");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    dispatch_float(s_dtype, [&](auto dt) {
        constexpr int ST = decltype(dt)::value;
        auto go = [&](auto kern, int cl) {
            launch(kern, dim3(cdiv(n, 4 * cl), k / group_size), dim3(512), 0, stream, static_cast<const float *>(w),
                   static_cast<uint8_t *>(packed), scales, n, group_size);
        };
        const bool once = k * n * 4 >= kReadOnceFrom && n % 32 == 0;  // (rows of whole cache lines)
        if (group_size <= 32) go(group_quantize_int4_kernel<ST, 64, 4>, 64);
        else if (group_size <= 64 && once) go(group_quantize_int4_kernel<ST, 64, 8, true>, 64);
        else if (group_size <= 64) go(group_quantize_int4_kernel<ST, 64, 8>, 64);
        else if (group_size <= 128 && once) go(group_quantize_int4_kernel<ST, 32, 8, true>, 32);
        else if (group_size <= 128) go(group_quantize_int4_kernel<ST, 32, 8>, 32);
        else if (group_size <= 256) go(group_quantize_int4_kernel<ST, 16, 8>, 16);
        else go(group_quantize_int4_kernel<ST, 64, 0>, 64);
    });
    QMM_ENTRY_END
}

HIDET_API void hidet_fp8_quantize_per_tensor(const void *x, void *codes, void *scale, int64_t numel, int x_dtype,
                                             void *workspace, int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(scale, "null scale pointer");
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    QMM_CHECK(ws.scratch_bytes >= 4, "workspace too small");
    QMM_CHECK(numel == 0 || (x && codes), "null tensor pointer");
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    float *amax = reinterpret_cast<float *>(ws.scratch);
    dispatch_float(x_dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        const int esize = DT == HIDET_QMM_F32 ? 4 : 2;
        QMM_CHECK(aligned(x, esize), "the tensor is not aligned to its element type");
        if (numel <= 65536 && numel % 4 == 0 && aligned(x, 4 * esize) && aligned(codes, 4)) {
            launch(fp8_quantize_small_kernel<DT>, dim3(uint32_t(std::max<int64_t>(1, cdiv(numel / 4, 1024)))), dim3(1024), 0, stream, x, static_cast<uint32_t *>(codes),
                   static_cast<float *>(scale), int(numel / 4));
            return;
        }
        const int64_t chunks = cdiv(numel, int64_t(kChunkVectors) * (16 / esize)), chunks8 = cdiv(chunks, 8);
        QMM_CHECK(chunks8 * 8 < (int64_t(1) << 31), "tensor too large for one launch");
        // four workgroups per CU, a multiple of the XCDs (a chunk is then converted on the XCD that looked at it); fewer where the
        // scratch memory holds fewer maxima
        const int64_t partials = std::min<int64_t>({chunks, kAmaxPartials, ws.scratch_bytes / 4});
        launch(amax_all_kernel<DT>, dim3(uint32_t(partials)), dim3(256), 0, stream, x, amax, numel, chunks);
        const int64_t fine8 = cdiv(cdiv(numel, int64_t(256) * (16 / esize)), 8);
        if (fine8 * 8 <= kFineChunks) launch(fp8_quantize_kernel<DT, 1>, dim3(uint32_t(fine8 * 8)), dim3(256), 0, stream, x, amax, int(partials), static_cast<uint8_t *>(codes),
                                      static_cast<float *>(scale), numel, fine8);
        else launch(fp8_quantize_kernel<DT, kChunkLoads>, dim3(uint32_t(chunks8 * 8)), dim3(256), 0, stream, x, amax, int(partials), static_cast<uint8_t *>(codes),
                    static_cast<float *>(scale), numel, chunks8);
    });
    QMM_ENTRY_END
}
