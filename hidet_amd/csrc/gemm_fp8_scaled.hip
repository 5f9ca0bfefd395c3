// Block-scaled FP8 e4m3 GEMM (DeepSeek-style): for every K block of 128
//   c[m, n] += (sum_{k in block} a[m, k] * b[n, k]) * scale_a[kb, m] * scale_b[n / 128, kb]
// with scale_a float32 [K/128, M] (M contiguous) and scale_b float32 [N/128, K/128].
//
// Each k block is multiplied into a scratch accumulator (one 16x16x128 MFMA per 16 x 16 block, C = 0) and folded into
// the running sum with its two scales on the vector ALU: one fma per accumulator element and k block, which the MFMA
// cannot absorb (its built-in block scales are powers of two).
//
// gemm_fp8_kernel8 (tensors below 1 GiB, 16-byte aligned): workgroup tile 256 x 128 (one scale_b entry per k block), eight
// waves of 64 x 64, two per SIMD, operand tiles and the block's row scales straight into a three-slot LDS ring
// (buffer_load ... lds) three k blocks ahead, one barrier per k block in the middle of its MFMAs, fragments fetched half a block
// ahead, the scratch accumulator double-buffered per row block so that the fold of row block i - 1 runs behind the MFMAs of row
// block i. The running sums live in VGPRs (the VALU cannot read accumulation registers). What bounds it: on real operands the
// power limit (16384 x 7168 x 1536 179 us, on zeros 150, all of these in one session, in others 192 to 204 in a graph of calls: before the
// scales came through the LDS, the barrier moved and the layout weighed bytes 188 and 163; 2048 x 7168 x 4096 62.0 -> 58.6, 8192 x 2048 x 1024
// 28.4 -> 23.3; without scales 16384 x 7168 x 1536 151 -> 142, 1536 x 4096 x 4096 28.6 -> 27.2, 8192 x 2048 x 1024 27.0 -> 19.9). Matrix and vector instructions of a SIMD hardly overlap, also between its two
// waves. Measured and dropped: single MFMAs alternating with their folds (fewer cycles but 226 us: the clock falls), 32 x 32 x 64
// MFMAs (on zeros 139, on real operands 180; without scales 149), raised priority during the MFMAs (180; 150).
// gemm_fp8_scaled_kernel (128 x 128 tile, register-staged double-buffered LDS) takes the rest.
#include "common.h"
#include "gemm_fp8_plan.h"
#include "gemm_tiling.h"
#include "numeric.h"

namespace qmm {
namespace {

constexpr int kT = 128;  // tile rows, tile columns and k-step bytes
constexpr int kThreads = 256;
constexpr int kStageChunks = 2 * kT * 8;
constexpr int kChunksPerThread = kStageChunks / kThreads;  // 8
constexpr int kLdsBytes = 2 * kStageChunks * 16;           // 64 KiB

template <int OUT>
__device__ __forceinline__ void store4_scaled(void *c, int64_t o, float4_t v) {
    if (OUT == HIDET_QMM_F32) {
        *reinterpret_cast<float4_t *>(static_cast<float *>(c) + o) = v;
    } else if (OUT == HIDET_QMM_BF16) {
        uint2 w2;
        w2.x = uint32_t(f32_to_bf16_bits(v[0])) | (uint32_t(f32_to_bf16_bits(v[1])) << 16);
        w2.y = uint32_t(f32_to_bf16_bits(v[2])) | (uint32_t(f32_to_bf16_bits(v[3])) << 16);
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(c) + o) = w2;
    } else if (OUT == HIDET_QMM_F16) {
        uint2 w2;
        w2.x = uint32_t(f32_to_f16_bits(v[0])) | (uint32_t(f32_to_f16_bits(v[1])) << 16);
        w2.y = uint32_t(f32_to_f16_bits(v[2])) | (uint32_t(f32_to_f16_bits(v[3])) << 16);
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(c) + o) = w2;
    } else if (OUT == HIDET_QMM_E5M2) {
        *reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(c) + o) =
            uint32_t(f32_to_e5m2(v[0])) | (uint32_t(f32_to_e5m2(v[1])) << 8) | (uint32_t(f32_to_e5m2(v[2])) << 16) |
            (uint32_t(f32_to_e5m2(v[3])) << 24);
    } else {
        *reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(c) + o) =
            uint32_t(f32_to_e4m3(v[0])) | (uint32_t(f32_to_e4m3(v[1])) << 8) | (uint32_t(f32_to_e4m3(v[2])) << 16) |
            (uint32_t(f32_to_e4m3(v[3])) << 24);
    }
}

// FMT: operand format of the MFMA, 0 = float8 e4m3, 1 = float8 e5m2 (both operands the same).
template <int OUT, int FMT = 0>
__global__ __launch_bounds__(kThreads, 1) void gemm_fp8_scaled_kernel(const uint8_t *__restrict__ a, const uint8_t *__restrict__ b,
                                                                      const float *__restrict__ scale_a,
                                                                      const float *__restrict__ scale_b, void *__restrict__ c,
                                                                      int m, int n, int k, int tiles_m) {
    extern __shared__ uint4 lds[];
    const int m0 = (blockIdx.x % tiles_m) * kT;
    const int nb = blockIdx.x / tiles_m;
    const int n0 = nb * kT;
    const int kblocks = k / 128;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int kg = lane >> 4, ls = lane & 15;

    float4_t total[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) total[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    uint4 stage[kChunksPerThread];
    auto load_stage = [&](int kbase) {
#pragma unroll
        for (int j = 0; j < kChunksPerThread; ++j) {
            const int id = j * kThreads + tid;
            const int row = id >> 3, pos = id & 7;
            const int kb = kbase + (pos ^ (row & 7)) * 16;
            stage[j] = uint4{0u, 0u, 0u, 0u};
            if (j < kChunksPerThread / 2) {
                if (m0 + row < m) stage[j] = *reinterpret_cast<const uint4 *>(a + int64_t(m0 + row) * k + kb);
            } else {
                if (n0 + row - kT < n) stage[j] = *reinterpret_cast<const uint4 *>(b + int64_t(n0 + row - kT) * k + kb);
            }
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int j = 0; j < kChunksPerThread; ++j) lds[buf * kStageChunks + j * kThreads + tid] = stage[j];
    };

    load_stage(0);
    store_stage(0);
    __syncthreads();

    for (int s = 0; s < kblocks; ++s) {
        const int buf = s & 1;
        const bool more = s + 1 < kblocks;
        if (more) load_stage((s + 1) * 128);
        // scale of this k block for the lane's 4 rows (one per row block) and the tile's column block
        const float sb = scale_b[int64_t(nb) * kblocks + s];
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = m0 + wm * 64 + i * 16 + ls;
            f[i] = row < m ? scale_a[int64_t(s) * m + row] * sb : 0.f;
        }
        const uint4 *la = lds + buf * kStageChunks;
        const uint4 *lb = la + kT * 8;
        uint4 bf[4][2];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = wn * 64 + j * 16 + ls;
            bf[j][0] = lb[r * 8 + ((2 * kg) ^ (r & 7))];
            bf[j][1] = lb[r * 8 + ((2 * kg + 1) ^ (r & 7))];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = wm * 64 + i * 16 + ls;
            const uint4 a0 = la[r * 8 + ((2 * kg) ^ (r & 7))];
            const uint4 a1 = la[r * 8 + ((2 * kg + 1) ^ (r & 7))];
            int8v_t cv;
            cv[0] = int(a0.x); cv[1] = int(a0.y); cv[2] = int(a0.z); cv[3] = int(a0.w);
            cv[4] = int(a1.x); cv[5] = int(a1.y); cv[6] = int(a1.z); cv[7] = int(a1.w);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int8v_t rv;
                rv[0] = int(bf[j][0].x); rv[1] = int(bf[j][0].y); rv[2] = int(bf[j][0].z); rv[3] = int(bf[j][0].w);
                rv[4] = int(bf[j][1].x); rv[5] = int(bf[j][1].y); rv[6] = int(bf[j][1].z); rv[7] = int(bf[j][1].w);
                const float4_t part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    rv, cv, float4_t{0.f, 0.f, 0.f, 0.f}, FMT, FMT, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
#pragma unroll
                for (int v = 0; v < 4; ++v) total[i][j][v] += part[v] * f[i];
            }
        }
        if (more) store_stage(buf ^ 1);
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * 64 + i * 16 + ls;
        if (row >= m) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + wn * 64 + j * 16 + 4 * kg;
            if (col >= n) continue;
            const int64_t o = int64_t(row) * n + col;
            const float4_t v = total[i][j];
            store4_scaled<OUT>(c, o, v);
        }
    }
}


// ---- fast path ---------------------------------------------------------------------------------------------------------

constexpr int kThreads8 = 512;
constexpr int kOperandChunks8 = (kM8 + kN8) * 8;       // 16-byte chunks of one k block: A rows then B rows
constexpr int kSlotChunks8 = kOperandChunks8 + kM8 / 4;  // + the block's scales of the rows
constexpr int kLoads8 = kOperandChunks8 / kThreads8;  // 6 direct-to-LDS loads per thread and k block
constexpr int kRingBytes8 = 3 * kSlotChunks8 * 16;  // 147 KiB
constexpr int kLdsBytes8 = kRingBytes8 + 16;       // + the K-split fix-up's flag; the ring must start at LDS address 0

template <int FMT>
__device__ __forceinline__ float4_t mfma_fp8_k128(const int4v_t (&r)[2], const int4v_t (&c)[2], const float4_t &acc) {
    const int8v_t rv = __builtin_shufflevector(r[0], r[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const int8v_t cv = __builtin_shufflevector(c[0], c[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(rv, cv, acc, FMT, FMT, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
}

// sum += part * factor, at its place among the instructions around it.
__device__ __forceinline__ void fold_row_block(float4_t (&part)[4], float4_t (&sum)[4], float factor) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        asm volatile("" : "+v"(part[j]));
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[j][v] = __builtin_fmaf(part[j][v], factor, sum[j][v]);
        asm volatile("" : "+v"(sum[j]));
    }
}

// SCALED: scale_a / scale_b are the block scales described at the top of the file. !SCALED: plain a x b^T with optional
// per-tensor scales (one float each, may be null), applied to the sums in the epilogue.
template <int OUT, bool SCALED, int FMT = 0>
__global__ __launch_bounds__(kThreads8, 1) void gemm_fp8_kernel8(const uint8_t *__restrict__ a, int64_t lda,
                                                                 const uint8_t *__restrict__ b, int64_t ldb,
                                                                 const float *__restrict__ scale_a,
                                                                 const float *__restrict__ scale_b, void *__restrict__ c,
                                                                 int m, int n, int k, int tiles_m, int tiles_n, int xm, int xn,
                                                                 int tail_parts, int tail_stride, int panel, float *__restrict__ partials,
                                                                 uint32_t *__restrict__ counters) {
    extern __shared__ uint4 lds[];  // [3][kSlotChunks8]; no static LDS: fragment reads address the ring from 0
    int &s_last = *reinterpret_cast<int *>(lds + kRingBytes8 / 16);
    GemmWorkItem item;
    if (!gemm_work_item(tiles_m, tiles_n, xm, xn, kConcurrent8, tail_parts, tail_stride, &item, panel)) return;
    const int tile_m = item.tile_m, tile_n = item.tile_n;
    const int m0 = tile_m * kM8, n0 = tile_n * kN8;
    const int kblocks = k / 128;
    // this workgroup's K range (the whole of K unless the launch splits tail tiles)
    const int kb_begin = (kblocks * item.part) / item.parts, kb_end = (kblocks * (item.part + 1)) / item.parts;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int kg = lane >> 4, ls = lane & 15;

    float4_t total[4][4];  // [row block][column block] of this wave's 64 x 64
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) total[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a), 0, int(int64_t(m - 1) * lda + k), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(b), 0, int(int64_t(n - 1) * ldb + k), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_sa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(scale_a), 0, SCALED ? int(int64_t(kblocks) * m * 4) : 0, 0x00020000);

    // Load instruction j of a wave fills chunk slots j * 512 + wave * 64 .. + 63 of a k block: tile row j * 64 + tid / 8
    // (A rows for j < 4, B rows after), position tid % 8, which holds chunk (tid % 8) ^ key(row). Rows past the end of a
    // tensor get an offset outside the buffer and read as zero.
    constexpr int kOutside = 0x7FFFFFF0;
    const int chunk = (tid & 7) ^ lds_swizzle_key_step2(tid >> 3);
    int voff[kLoads8];
#pragma unroll
    for (int j = 0; j < kLoads8; ++j) {
        const int r = j * 64 + (tid >> 3);
        if (j < 4) voff[j] = m0 + r < m ? int(int64_t(m0 + r) * lda) + chunk * 16 : kOutside;
        else voff[j] = n0 + r - kM8 < n ? int(int64_t(n0 + r - kM8) * ldb) + chunk * 16 : kOutside;
    }
    // The row scales of a k block lie next to each other: one more direct-to-LDS load per wave (64 rows, four waves would do; the
    // same number of loads in every wave keeps the waits alike). Fetched per lane and block instead, four rows and the column
    // factor, they took the vector memory path about as long as the operands: 174 against 134 us with the MFMAs left out.
    const int sa_row = m0 + (wave & 3) * 64 + lane, sa_off = sa_row < m ? sa_row * 4 : kOutside;
    // A short matrix leaves most of the 256 tile rows empty: load instructions whose 64 rows all lie past M are left
    // out (a_cnt of the 4 stay; the same for every wave), and a wave whose 64 output rows do skips its fragment reads
    // and MFMAs. That takes a plainer loop, in which a tile of 129 to 192 rows would take a quarter longer than a full one (924 x 4096 x 4096 with block
    // scales 38.5 us, a full matrix 32.6): such a tile is computed as a full one, its last loads answered with zeros.
    int a_cnt = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) a_cnt += int(m0 + j * 64 < m);
    if (a_cnt == 3) a_cnt = 4;
    const bool wave_active = m0 + wm * 64 < m;
    constexpr int kBlockLoads = kLoads8 + (SCALED ? 1 : 0);
    auto load_one = [&](auto j_tag, int kb, int slot) {  // one of the kBlockLoads instructions of a k block
        constexpr int J = decltype(j_tag)::value;
        // the scalar offset is not part of the buffer's range check: a prefetch past the end of K re-reads the last block
        const int kbc = kb < kblocks ? kb : kblocks - 1;
        uint4 *dst = lds + slot * kSlotChunks8;
        if constexpr (J < kLoads8) buffer_load_to_lds_b128(J < 4 ? rsrc_a : rsrc_b, dst + wave * 64 + J * kThreads8, voff[J], kbc * 128);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_sa, (__attribute__((address_space(3))) void *)(dst + kOperandChunks8 + (wave & 3) * 16), 4,
                                                     sa_off, kbc * m * 4, 0, 0);
    };
    using i0 = std::integral_constant<int, 0>;
    using i1 = std::integral_constant<int, 1>;
    using i2 = std::integral_constant<int, 2>;
    using i3 = std::integral_constant<int, 3>;
    using i4 = std::integral_constant<int, 4>;
    using i5 = std::integral_constant<int, 5>;
    using i6 = std::integral_constant<int, 6>;
    using i7 = std::integral_constant<int, 7>;
    auto load_tiles = [&](int kb, int slot) {
        load_one(i0(), kb, slot);
        if (a_cnt > 1) load_one(i1(), kb, slot);
        if (a_cnt == 4) load_one(i2(), kb, slot), load_one(i3(), kb, slot);
        load_one(i4(), kb, slot);
        load_one(i5(), kb, slot);
        if constexpr (SCALED) load_one(i6(), kb, slot);
    };
    auto wait_older_tiles = [&]() {  // everything but the loads of the last load_tiles has landed
        if (a_cnt == 1) __builtin_amdgcn_s_waitcnt(waitcnt_vm(kBlockLoads - 3));
        else __builtin_amdgcn_s_waitcnt(waitcnt_vm(kBlockLoads - 2));
    };
    // The column factor of 64 k blocks at a time, one per lane (lane s % 64 that of block s).
    const float *const col_scale = SCALED ? scale_b + int64_t(tile_n) * kblocks : nullptr;
    float sb_lane = 1.0f;
    auto column_factors_at = [&](int kb) {
        const int at = (kb & ~63) + lane;
        return col_scale + (at < kblocks ? at : kblocks - 1);
    };
    auto fetch_column_factors = [&](int kb) {  // (load and wait by hand: a load that the compiler knows of would be waited for in every block)
        asm volatile("global_load_dword %0, %1, off\n\ts_waitcnt vmcnt(0)" : "=v"(sb_lane) : "v"(column_factors_at(kb)) : "memory");
    };
    auto column_factor = [&](int kb) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sb_lane), kb & 63)); };
    if constexpr (SCALED) sb_lane = *column_factors_at(kb_begin);
    __builtin_amdgcn_sched_barrier(0);  // (in front of the tiles' loads: it is waited for together with the first of them)

    // LDS byte addresses of this lane's two 16-byte fragment halves in block 0 of its wave, ring slot 0; block i adds
    // i * 16 rows = i * 2048 bytes
    uint32_t a_addr[2], b_addr[2];
    {
        const int ra = wm * 64 + ls, rb = kM8 + wn * 64 + ls;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            a_addr[h] = uint32_t((ra * 8 + ((2 * kg + h) ^ lds_swizzle_key_step2(ra))) * 16);
            b_addr[h] = uint32_t((rb * 8 + ((2 * kg + h) ^ lds_swizzle_key_step2(rb))) * 16);
        }
    }
    const uint32_t sa_addr = uint32_t(kOperandChunks8 * 16 + (wm * 64 + ls) * 4);
    constexpr uint32_t kSlotBytes = kSlotChunks8 * 16;
    int4v_t af[4][2], bf[4][2];        // [16-row or 16-column block][half]
    uint64_t sa_pair[2] = {0, 0};      // factors of this lane's rows, blocks 0 and 1, 2 and 3
    auto read_a = [&](auto i_tag, uint32_t so) {
        constexpr int I = decltype(i_tag)::value;
        af[I][0] = lds_read_b128_early<I * 2048>(a_addr[0] + so);
        af[I][1] = lds_read_b128_early<I * 2048>(a_addr[1] + so);
    };
    auto read_b = [&](auto j_tag, uint32_t so) {
        constexpr int J = decltype(j_tag)::value;
        bf[J][0] = lds_read_b128_early<J * 2048>(b_addr[0] + so);
        bf[J][1] = lds_read_b128_early<J * 2048>(b_addr[1] + so);
    };
    auto read_row_factors = [&](uint32_t so) {
        if constexpr (!SCALED) return;
        asm volatile("ds_read2_b32 %0, %1 offset0:0 offset1:16" : "=v"(sa_pair[0]) : "v"(sa_addr + so));
        asm volatile("ds_read2_b32 %0, %1 offset0:32 offset1:48" : "=v"(sa_pair[1]) : "v"(sa_addr + so));
    };
    float f[4] = {0.f, 0.f, 0.f, 0.f};  // factors of the k block at hand, per row block
    auto take_factors = [&](int kb) {   // (behind the wait for sa_pair)
        asm volatile("" : "+v"(sa_pair[0]), "+v"(sa_pair[1]));
        const float sb = column_factor(kb);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = __builtin_bit_cast(float, uint32_t(sa_pair[i >> 1] >> (32 * (i & 1)))) * sb;
    };
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};

    if (a_cnt == 4) {
        // Full tiles. One barrier per k block, in the middle of its MFMAs: in front of it everything of this block has been
        // read (its slot is free for block s + 3) and every wave's loads of block s + 1 have landed, behind it the fragments
        // of block s + 1 are fetched as those of this block have had their last use. The four MFMAs of a row block run as one
        // burst and the sums of the row block before are folded behind them. `keep` fixes that order: left to itself the
        // compiler folds a row block right behind its own MFMAs, which then wait for one another.
        float4_t part[2][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) part[0][j] = zero, part[1][j] = zero;
        auto keep = [](auto &v) { asm volatile("" : "+v"(v)); };
        load_tiles(kb_begin, 0);
        load_tiles(kb_begin + 1, 1);
        load_tiles(kb_begin + 2, 2);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kBlockLoads));
        asm volatile("" : "+v"(sb_lane) :: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_a(i0(), 0);
        read_a(i1(), 0);
        read_row_factors(0);
        read_a(i2(), 0);
        lds_wait_keep_newer<2>(af[0][0], af[1][0]);  // (no more than 15 reads can be counted)
        read_b(i0(), 0);
        read_b(i1(), 0);
        read_b(i2(), 0);
        read_b(i3(), 0);
        read_a(i3(), 0);
        __builtin_amdgcn_sched_barrier(0);
        int slot = 0;
        for (int s = kb_begin; s < kb_end; ++s) {
            const int next = slot == 2 ? 0 : slot + 1;
            const uint32_t so = uint32_t(next) * kSlotBytes;
            auto row_block = [&](auto i_tag) {
                constexpr int I = decltype(i_tag)::value, O = (I + 3) % 4;
                // reads in flight, oldest first: a0 a1 factors a2 | b0 b1 b2 b3 a3, two each
                if constexpr (I == 0) {
                    lds_wait_keep_newer<8>(af[0][0], af[0][1]);
                    lds_wait_keep_newer<8>(bf[0][0], bf[0][1]);
                }
                auto mm = [&](auto j_tag) {
                    constexpr int J = decltype(j_tag)::value;
                    if constexpr (I == 0 && J > 0) lds_wait_keep_newer<8 - 2 * J>(bf[J][0], bf[J][1]);
                    else keep(af[I][0]);
                    if constexpr (SCALED) {
                        part[I & 1][J] = mfma_fp8_k128<FMT>(bf[J], af[I], zero);
                        keep(part[I & 1][J]);
                    } else {
                        total[I][J] = mfma_fp8_k128<FMT>(bf[J], af[I], total[I][J]);
                        keep(total[I][J]);
                    }
                };
                mm(i0());
                mm(i1());
                mm(i2());
                mm(i3());
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (I == 1) {
                    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kBlockLoads));
                    lds_wait_keep_newer<0>(af[2][0], af[2][1]);
                    lds_wait_keep_newer<0>(af[3][0], af[3][1]);
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    read_a(i0(), so);
                    read_a(i1(), so);
                    read_row_factors(so);
                    load_one(i0(), s + 3, slot), load_one(i1(), s + 3, slot);
                }
                if constexpr (I == 2) {
                    read_a(i2(), so);
                    load_one(i2(), s + 3, slot), load_one(i3(), s + 3, slot), load_one(i4(), s + 3, slot);
                }
                if constexpr (I == 3) {
                    lds_wait_keep_newer<2>(af[0][0], af[1][0]);
                    read_b(i0(), so);
                    read_b(i1(), so);
                    read_b(i2(), so);
                    read_b(i3(), so);
                    read_a(i3(), so);
                    load_one(i5(), s + 3, slot);
                    if constexpr (SCALED) load_one(i6(), s + 3, slot);
                }
                if constexpr (SCALED) {
                    fold_row_block(part[O & 1], total[O], f[O]);
                    if constexpr (I == 0) {
                        take_factors(s);
                        keep(f[0]), keep(f[1]), keep(f[2]), keep(f[3]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            row_block(i0());
            row_block(i1());
            row_block(i2());
            row_block(i3());
            slot = next;
            if constexpr (SCALED)
                if (((s + 1) & 63) == 0) fetch_column_factors(s + 1);
        }
        if constexpr (SCALED) fold_row_block(part[1], total[3], f[3]);
        // the fragments of a block past the end must not land in registers that have another use by then
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lds_wait_keep_newer<0>(af[i][0], af[i][1]);
            lds_wait_keep_newer<0>(bf[i][0], bf[i][1]);
        }
        asm volatile("" : "+v"(sa_pair[0]), "+v"(sa_pair[1]));
    } else {
        load_tiles(kb_begin, 0);
        load_tiles(kb_begin + 1, 1);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        asm volatile("" : "+v"(sb_lane) :: "memory");
        __builtin_amdgcn_s_barrier();
        for (int s = kb_begin, slot = 0; s < kb_end; ++s) {
            load_tiles(s + 2, slot >= 1 ? slot - 1 : 2);  // slot (s + 2) % 3 was last read in k block s - 1
            if (wave_active) {
                const uint32_t so = uint32_t(slot) * kSlotBytes;
                read_row_factors(so);
                read_b(i0(), so);
                read_a(i0(), so);
                read_b(i1(), so);
                read_b(i2(), so);
                read_b(i3(), so);
                lds_wait_keep_newer<6>(af[0][0], bf[0][0]);  // (no more than 15 reads can be counted)
                read_a(i1(), so);
                read_a(i2(), so);
                read_a(i3(), so);
                __builtin_amdgcn_sched_barrier(0);
                lds_wait_keep_newer<12>(af[0][0], af[0][1]);
                lds_wait_keep_newer<12>(bf[0][0], bf[0][1]);
                if constexpr (SCALED) take_factors(s);
                lds_wait_keep_newer<6>(bf[1][0], bf[1][1]);
                lds_wait_keep_newer<6>(bf[2][0], bf[2][1]);
                lds_wait_keep_newer<6>(bf[3][0], bf[3][1]);
                auto row_block = [&](auto i_tag) {
                    constexpr int I = decltype(i_tag)::value;
                    if constexpr (I > 0) lds_wait_keep_newer<2 * (3 - I)>(af[I][0], af[I][1]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if constexpr (SCALED) {
                            const float4_t sum = mfma_fp8_k128<FMT>(bf[j], af[I], zero);
#pragma unroll
                            for (int v = 0; v < 4; ++v) total[I][j][v] = __builtin_fmaf(sum[v], f[I], total[I][j][v]);
                        } else {
                            total[I][j] = mfma_fp8_k128<FMT>(bf[j], af[I], total[I][j]);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                row_block(i0());
                row_block(i1());
                row_block(i2());
                row_block(i3());
            }
            if constexpr (SCALED)
                if (((s + 1) & 63) == 0) fetch_column_factors(s + 1);
            // the tiles of k block s + 1 (issued one block ago) must have landed before anyone reads them; the loads issued
            // in this block may stay in flight
            wait_older_tiles();
            __builtin_amdgcn_s_barrier();
            slot = slot == 2 ? 0 : slot + 1;
        }
    }
    // LDS must not be released with tile loads in flight
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));

    if (item.parts > 1) {
        uint32_t rows_valid = 0;  // row blocks of this wave that reach into the matrix
#pragma unroll
        for (int i = 0; i < 4; ++i) rows_valid |= uint32_t(m0 + wm * 64 + i * 16 < m) << i;
        if (!gemm_k_split_fixup<kThreads8>(total, item, partials, counters, &s_last, rows_valid)) return;
    }

    float alpha = 1.0f;
    if constexpr (!SCALED) {
        if (scale_a != nullptr) alpha *= *scale_a;
        if (scale_b != nullptr) alpha *= *scale_b;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * 64 + i * 16 + ls;
        if (row >= m) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + wn * 64 + j * 16 + 4 * kg;
            if (col >= n) continue;  // n % 4 == 0
            float4_t v = total[i][j];
            if constexpr (!SCALED) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] *= alpha;
            }
            store4_scaled<OUT>(c, int64_t(row) * n + col, v);
        }
    }
}

}  // namespace

// Estimated time in microseconds of the tiled kernels, for the choice between them and the narrow tiles of gemm_mid.h: the plan's time and a fixed part
// with which that choice is right (one microsecond more or less changes it for 3 of 427 shapes of 17 to 1100 rows); where K is no multiple of 128 (the register-staged 256 x 256
// kernel) 3.5 us per k block and round.
double gemm_fp8_estimate_us(int64_t m, int64_t n, int64_t k, bool scaled, void *workspace, int64_t workspace_bytes) {
    if (k % 128 != 0) return 8.0 + double(cdiv(cdiv(m, 256) * cdiv(n, 256), 256)) * 3.5 * double(cdiv(k, 128));
    return (scaled ? 7.3 : 9.1) + make_fp8_plan(m, n, k, scaled, split_workspace(workspace, workspace_bytes)).us;
}

// Launch of the 8-wave kernel; SCALED selects block scales (scale_a [K/128, M], scale_b [N/128, K/128]) or optional
// per-tensor scales.
template <bool SCALED, int FMT = 0>
static void launch_kernel8(const void *a, int64_t lda, const void *b, int64_t ldb, const void *scale_a, const void *scale_b,
                           void *c, int64_t m, int64_t n, int64_t k, int out_dtype, void *workspace, int64_t workspace_bytes,
                           hipStream_t stream) {
    const int tiles_m = int(cdiv(m, kM8)), tiles_n = int(cdiv(n, kN8));
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    const Fp8Plan plan = make_fp8_plan(m, n, k, SCALED, ws);
    const GemmTiling &tiling = plan.tiling;
    const GemmTail &tail = plan.tail;
    const int64_t grid = gemm_grid_with_tail(tiling, kConcurrent8, tail);
    QMM_CHECK(grid < (int64_t(1) << 31), "problem too large for one launch");
    auto go = [&](auto kern) {
        allow_dynamic_lds(reinterpret_cast<const void *>(kern), kLdsBytes8);
        launch(kern, dim3(uint32_t(grid)), dim3(kThreads8), size_t(kLdsBytes8), stream, static_cast<const uint8_t *>(a), lda,
               static_cast<const uint8_t *>(b), ldb, static_cast<const float *>(scale_a), static_cast<const float *>(scale_b), c,
               int(m), int(n), int(k), tiles_m, tiles_n, tiling.xm, tiling.xn, tail.parts, tail.max_tiles, tiling.panel,
               reinterpret_cast<float *>(ws.scratch), ws.counters);
    };
    constexpr int kOut8 = FMT == 1 ? HIDET_QMM_E5M2 : HIDET_QMM_E4M3;  // the 8-bit output type is the operands' own
    if (out_dtype == HIDET_QMM_F32) go(gemm_fp8_kernel8<HIDET_QMM_F32, SCALED, FMT>);
    else if (out_dtype == HIDET_QMM_F16) go(gemm_fp8_kernel8<HIDET_QMM_F16, SCALED, FMT>);
    else if (out_dtype == HIDET_QMM_BF16) go(gemm_fp8_kernel8<HIDET_QMM_BF16, SCALED, FMT>);
    else if (out_dtype == kOut8) go(gemm_fp8_kernel8<kOut8, SCALED, FMT>);
    else QMM_FAIL("unsupported output dtype code " << out_dtype);
}

// a x b^T with optional per-tensor scales on the 256 x 128, 8-wave kernel. The caller has checked: K a multiple of 128,
// 16-byte aligned rows and pointers, N a multiple of 4, tensors below 1 GiB.
void gemm_fp8_kernel8_launch(const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                             int out_dtype, const void *scale_a, const void *scale_b, void *workspace, int64_t workspace_bytes,
                             hipStream_t stream) {
    launch_kernel8<false>(a, lda, b, ldb, scale_a, scale_b, c, m, n, k, out_dtype, workspace, workspace_bytes, stream);
}

template <int FMT>
static void scaled_launch(const void *a, const void *b, const void *scale_a, const void *scale_b, void *c, int64_t m, int64_t n,
                          int64_t k, int out_dtype, void *workspace, int64_t workspace_bytes, hipStream_t stream) {
    const bool fast = m * k <= (int64_t(1) << 30) && n * k <= (int64_t(1) << 30) && (k / 128) * m * 4 < (int64_t(1) << 31) &&
                      aligned(a, 16) && aligned(b, 16) && aligned(c, 16);
    if (fast) {
        launch_kernel8<true, FMT>(a, k, b, k, scale_a, scale_b, c, m, n, k, out_dtype, workspace, workspace_bytes, stream);
        return;
    }
    const int tiles_m = int(cdiv(m, kT)), tiles_n = int(n / 128);
    const int64_t grid = int64_t(tiles_m) * tiles_n;
    QMM_CHECK(grid < (int64_t(1) << 31), "problem too large for one launch");
    auto go = [&](auto kern) {
        launch(kern, dim3(uint32_t(grid)), dim3(kThreads), size_t(kLdsBytes), stream, static_cast<const uint8_t *>(a),
               static_cast<const uint8_t *>(b), static_cast<const float *>(scale_a), static_cast<const float *>(scale_b), c,
               int(m), int(n), int(k), tiles_m);
    };
    constexpr int kOut8 = FMT == 1 ? HIDET_QMM_E5M2 : HIDET_QMM_E4M3;
    if (out_dtype == HIDET_QMM_F32) go(gemm_fp8_scaled_kernel<HIDET_QMM_F32, FMT>);
    else if (out_dtype == HIDET_QMM_F16) go(gemm_fp8_scaled_kernel<HIDET_QMM_F16, FMT>);
    else if (out_dtype == HIDET_QMM_BF16) go(gemm_fp8_scaled_kernel<HIDET_QMM_BF16, FMT>);
    else if (out_dtype == kOut8) go(gemm_fp8_scaled_kernel<kOut8, FMT>);
    else QMM_FAIL("unsupported output dtype code " << out_dtype);
}

// `e5m2`: both operands are float8_e5m2 (the 8-bit output type is then e5m2 as well), else e4m3.
void gemm_fp8_scaled_launch(const void *a, const void *b, const void *scale_a, const void *scale_b, void *c, int64_t m,
                            int64_t n, int64_t k, int out_dtype, bool e5m2, void *workspace, int64_t workspace_bytes,
                            hipStream_t stream) {
    if (e5m2) scaled_launch<1>(a, b, scale_a, scale_b, c, m, n, k, out_dtype, workspace, workspace_bytes, stream);
    else scaled_launch<0>(a, b, scale_a, scale_b, c, m, n, k, out_dtype, workspace, workspace_bytes, stream);
}

}  // namespace qmm
