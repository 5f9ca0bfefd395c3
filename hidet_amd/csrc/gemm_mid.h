// GEMMs of a few dozen to a few hundred activation rows: more than the one pass of the bandwidth-bound kernels, too few
// for the large tiles of the prefill GEMMs to fill the chip.
//
// What bounds these sizes is neither memory nor MFMAs but how few workgroups there are and what it costs to bring the pieces
// of K together again. A workgroup of eight waves owns a tile of 16 RB rows x 64 or 128 columns; the K stages of the tile go in
// turn to groups of one or two waves, each with its part of the tile in its own accumulators and a ring of operand slices in
// LDS (filled by direct-to-LDS loads), and the groups meet once, at the end, in LDS. So K is cut eight ways inside a
// workgroup before it is cut between workgroups, and the partial results that cross memory stay small: 64 rows x 4096 columns x
// 4096 deep run as 32 tiles in four pieces of 32 KiB, where the 128 x 256 tiles of the prefill GEMM gave 16 tiles in eight pieces of
// 64 KiB and used 128 of 256 CUs. int8, K = 4096, N = 4096: 49 / 128 / 256 / 512 rows 17.4 / 27.5 / 28.3 / 32.7 -> 12.3 / 15.0 / 19.2 /
// 26.7 us; K = 11008, N = 4096: 49 / 128 / 256 rows 27.6 / 49.4 / 49.9 -> 20.9 / 26.6 / 36.1 us.
//
// An operand policy `Op` says how a stage of weights is loaded, widened and multiplied and how four results of a row are
// stored; everything else - the ring, the K tail, the meeting of the waves, the exchange of the pieces - is here.
#pragma once
#include "common.h"
#include "gemm_tiling.h"

namespace qmm {

constexpr int kMidWaves = 8;
constexpr int kMidThreads = kMidWaves * 64;

// The work of a launch: item (tile, piece), the pieces of a tile being `parts` equal runs of its K stages. XCD x takes the
// items from `items` x / 8 on, in an order that keeps the row tiles of a column next to each other (they read the same
// weights). All of it is 32-bit arithmetic with divisions by host-made reciprocals: what stands before a workgroup's
// first load delays the whole launch. One piece per workgroup: everything after the K loop - the groups' meeting, the
// exchange - costs a workgroup about 4 us, whatever the size of the piece, and runs across tile boundaries, which use every
// CU, pay that twice.
struct MidPlan {
    int m, n;
    int tiles_m, tiles_n, stages, parts, share;  // share: stages of a piece, the last one's may be fewer
    uint32_t tiles_m_magic, parts_magic;
    float *partials;
    uint32_t *counters;
};

__host__ __device__ __forceinline__ uint32_t mid_magic(int d) { return d <= 1 ? 0xFFFFFFFFu : uint32_t((uint64_t(1) << 32) / uint32_t(d)); }
__host__ __device__ __forceinline__ int mid_div(int n, int d, uint32_t magic) {
    const uint32_t q = uint32_t((uint64_t(uint32_t(n)) * magic) >> 32);  // one too small at most
    return int((q + 1) * uint32_t(d) <= uint32_t(n) ? q + 1 : q);
}

struct MidItem {
    int tile_m, tile_n, tile;  // `tile`: number of the tile, for its counter and its partial results
    int part, s_begin, s_end;
};
// Item of workgroup `block` (of 8 ceil(items / 8)); false: it has none.
__host__ __device__ __forceinline__ bool mid_item(const MidPlan &p, int block, MidItem *r) {
    const uint32_t items = uint32_t(p.tiles_m) * p.tiles_n * p.parts, xcd = block & 7;
    const int at = int((items * xcd) >> 3) + (block >> 3);
    if (at >= int((items * (xcd + 1)) >> 3)) return false;
    const int rest = mid_div(at, p.tiles_m, p.tiles_m_magic);
    r->tile_m = at - rest * p.tiles_m;
    r->tile_n = mid_div(rest, p.parts, p.parts_magic);
    r->part = rest - r->tile_n * p.parts;
    r->tile = r->tile_n * p.tiles_m + r->tile_m;
    r->s_begin = r->part * p.share;
    r->s_end = r->s_begin + p.share < p.stages ? r->s_begin + p.share : p.stages;
    return true;
}

// Added to a lane's offset it leads past the end of every buffer here (each below 2 GiB, as are the offsets).
constexpr uint32_t kMidOutside = 0x80000000u;

template <int N>
struct MidStatic {
    static constexpr int value = N;
};
template <int B, int E, typename F>
__device__ __forceinline__ void mid_for(F &&f) {
    if constexpr (B < E) {
        f(MidStatic<B>());
        mid_for<B + 1, E>(f);
    }
}

// Row key of the 16-byte chunk swizzle of a slot with rows of 128 (eight chunks, two consecutive ones read per lane) or 64
// bytes (four chunks, one read per lane): both keep the 16 lanes that ds_read_b128 serves at a time on 16 different bank
// groups (see lds_swizzle_key_step1; for four chunks a group sees rows 0-3 and 12-15 at chunk g and rows 4-11 at chunk
// g ^ 1, hence the keys 0, 2, 3, 1 of the four row quarters).
template <int ROW_BYTES>
__device__ __forceinline__ int mid_key(int row) {
    if constexpr (ROW_BYTES == 64) return (0x78 >> (((row >> 2) & 3) * 2)) & 3;
    else return (row & 7) ^ ((row >> 3) & 1);
}

// Where Op::kKeep: the fragments are computed here and not further down. The compiler moves the widening of every other round to where
// the fragments are used, behind the MFMAs that it is meant to run beside. int4, whose widening is long, gains by having it back (256 x 4096 x
// 4096 23.3 -> 21.9 us, 384 x 11008 x 4096 72.5 -> 67.8), int8 does not (512 x 4096 x 4096 24.6 -> 25.4) and FP8 with block scales loses (600 x 5376 x
// 1408 19.4 -> 21.5).
template <typename F>
__device__ __forceinline__ void mid_keep(F &f) {
    static_assert(sizeof(F) % 4 == 0, "registers");
    uint32_t r[sizeof(F) / 4];
    __builtin_memcpy(r, &f, sizeof(F));
#pragma unroll
    for (int i = 0; i < int(sizeof(F) / 4); ++i) asm volatile("" : "+v"(r[i]));
    __builtin_memcpy(&f, r, sizeof(F));
}

template <class Op, int RB, int DEPTH>
struct MidCfg {
    static constexpr int kGroupWaves = Op::kGroupWaves;        // waves side by side on one K stage,
    static constexpr int kFrags = Op::kFrags;                  // each with so many 16-column blocks, kFrags columns to a lane
    static constexpr int kGroups = kMidWaves / kGroupWaves;
    static constexpr int kWaveCols = kFrags * 16;
    static constexpr int kCols = kGroupWaves * kWaveCols;
    static constexpr int kPitch = kCols - Op::kSpare;          // columns from one tile to the next
    static constexpr int kRowBytes = Op::kRowBytes;            // bytes of an activation row per stage
    static constexpr int kChunks = kRowBytes / 16;
    static constexpr int kABytes = RB * 16 * kRowBytes;
    static constexpr int kALoads = kABytes / 1024 / kGroupWaves;  // direct-to-LDS instructions of a wave and stage
    static constexpr int kSlotBytes = kABytes + Op::kWLdsBytes;
    static constexpr int kLoads = kALoads + Op::kWLoads;
    static constexpr int kRingBytes = kGroups * DEPTH * kSlotBytes;
    static constexpr int kHalfRows = RB * kGroupWaves <= kMidWaves ? (RB < 4 ? RB : 4) : kMidWaves / kGroupWaves;  // row blocks that meet in LDS at a time
    static constexpr int kHalves = RB / kHalfRows;
    static constexpr int kPlanes = kMidWaves / (kHalfRows * kGroupWaves);
    static constexpr int kWidth = 4 / kPlanes;                 // accumulator rows a thread sums
    static constexpr int kMeetBytes = kGroups * kHalfRows * kGroupWaves * kFrags * 1024;
    static constexpr int kVecs = kFrags * kWidth / 4;          // float4 sums of a thread and half
    static constexpr int kLdsMain = kRingBytes > kMeetBytes ? kRingBytes : kMeetBytes;
    static constexpr int kLdsBytes = kLdsMain + 16;            // + the exchange's flag
    static constexpr int kTileFloats = RB * 16 * kCols;
    static_assert(kALoads * 1024 * kGroupWaves == kABytes, "whole load instructions");
    static_assert(kVecs * 4 == kFrags * kWidth, "whole float4 sums");
    static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");
    static_assert(kLoads * (DEPTH - 1) <= 63, "vmcnt range");
};

template <class Op, int RB, int DEPTH>
__global__ __launch_bounds__(kMidThreads) void gemm_mid_kernel(const char *a, const char *w, int a_stride, int w_stride, int k, int m, int n,
                                                               int tiles_m, int tiles_n, int stages, int parts, int share,
                                                               uint32_t tiles_m_magic, uint32_t parts_magic, float *partials,
                                                               uint32_t *counters, typename Op::Args args) {
    // (the sixteen words up to the last reciprocal arrive in scalar registers)
    const MidPlan plan{m, n, tiles_m, tiles_n, stages, parts, share, tiles_m_magic, parts_magic, partials, counters};
    using Cfg = MidCfg<Op, RB, DEPTH>;
    extern __shared__ uint4 lds[];  // no static LDS in this kernel: fragment reads address the rings from 0
    int *flag = reinterpret_cast<int *>(lds + Cfg::kLdsMain / 16);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = lane >> 4, ns = lane & 15;
    const int group = wave / Cfg::kGroupWaves, side = wave % Cfg::kGroupWaves;

    MidItem item;
    if (!mid_item(plan, int(blockIdx.x), &item)) return;
    const int m0 = item.tile_m * (RB * 16), n0 = item.tile_n * Cfg::kPitch;
    const int rows = plan.m - m0 < RB * 16 ? plan.m - m0 : RB * 16;

    // ---- main loop ----------------------------------------------------------------------------------------------
    Op op(args, w, w_stride, k, m, n, m0, n0, side, lane);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(a) + int64_t(m0) * a_stride, 0, (rows - 1) * a_stride + k * Op::kElementBytes, 0x00020000);
    int a_off[Cfg::kALoads];
#pragma unroll
    for (int i = 0; i < Cfg::kALoads; ++i) {
        const int id = (side * Cfg::kALoads + i) * 64 + lane, r = id / Cfg::kChunks;
        a_off[i] = r * a_stride + ((id % Cfg::kChunks) ^ mid_key<Cfg::kRowBytes>(r)) * 16;
    }
    const uint32_t ring = uint32_t(group * DEPTH * Cfg::kSlotBytes);
    uint32_t af_addr[Op::kAChunks];  // chunks of a fragment: kg (64-byte rows), 2 kg and 2 kg + 1 (128-byte rows)
#pragma unroll
    for (int q = 0; q < Op::kAChunks; ++q)
        af_addr[q] = ring + uint32_t(ns * Cfg::kRowBytes + (((kg * Op::kAChunks + q) ^ mid_key<Cfg::kRowBytes>(ns)) * 16));

    float4_t acc[RB][Cfg::kFrags];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int t = 0; t < Cfg::kFrags; ++t) acc[rb][t] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Every load of a stage past the end of the piece goes past the end of its buffer: it returns zeros without touching
    // memory, so the number of loads in flight is always the same. Activation rows past the matrix read as zeros. (All
    // offsets sit in the per-lane register, the only one that is range-checked.)
    auto issue = [&](uint32_t slot_bytes, int st, auto &&load_w) {
        const bool on = st < item.s_end;
        const uint32_t at = on ? uint32_t(st) * Cfg::kRowBytes : kMidOutside;
#pragma unroll
        for (int i = 0; i < Cfg::kALoads; ++i)
            buffer_load_to_lds_b128(rsrc_a, lds + (ring + slot_bytes + (side * Cfg::kALoads + i) * 1024) / 16, int(uint32_t(a_off[i]) + at), 0);
        load_w(on ? uint32_t(st) * uint32_t(op.w_stage) : kMidOutside, st);
    };
    auto multiply_all = [&](auto &af, auto &bf, int st) {
        mid_for<0, RB>([&](auto r) {
            constexpr int R = decltype(r)::value, NEWER = (RB - 1 - R) * Op::kAChunks;
            if constexpr (Op::kAChunks == 1) lds_wait_keep_newer<NEWER>(af[R][0]);
            else lds_wait_keep_newer<NEWER>(af[R][0], af[R][1]);
            if (st * Op::kStageK + Op::kStageK > k) op.mask(af[R], st, kg);  // the stage that K ends in
            op.multiply(af[R], bf, acc[R], r);
        });
    };
    if constexpr (Cfg::kGroupWaves == 1) {
        // weights in registers, activations in a ring of the wave's own: no barrier
        typename Op::Weights wr[DEPTH];
        int s = item.s_begin + group;
        mid_for<0, DEPTH>([&](auto d) {
            constexpr int D = decltype(d)::value;
            issue(D * Cfg::kSlotBytes, s + D * Cfg::kGroups, [&](uint32_t at, int) { op.load(wr[D], at); });
        });
        for (; s < item.s_end; s += DEPTH * Cfg::kGroups) {
            mid_for<0, DEPTH>([&](auto d_tag) {
                constexpr int D = decltype(d_tag)::value;
                const int st = s + D * Cfg::kGroups;
                if (st < item.s_end) {
                    __builtin_amdgcn_s_waitcnt(waitcnt_vm((DEPTH - 1) * Cfg::kLoads));
                    __builtin_amdgcn_sched_barrier(0);
                    int4v_t af[RB][Op::kAChunks];
                    mid_for<0, RB>([&](auto r) {
                        mid_for<0, Op::kAChunks>([&](auto q) {
                            constexpr int R = decltype(r)::value, Q = decltype(q)::value;
                            af[R][Q] = lds_read_b128_early<D * Cfg::kSlotBytes + R * 16 * Cfg::kRowBytes>(af_addr[Q]);
                        });
                    });
                    typename Op::Fragments bf;
                    op.widen(wr[D], bf, st);
                    multiply_all(af, bf, st);
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    issue(D * Cfg::kSlotBytes, st + DEPTH * Cfg::kGroups, [&](uint32_t at, int) { op.load(wr[D], at); });
                }
            });
        }
    } else {
        // Both operands in a ring that the waves of a group share, one barrier per stage. While a stage is multiplied the
        // next one is read from LDS and widened between the MFMAs: the waves of a workgroup run in step, so neither the
        // LDS's latency nor the widening hides behind another wave. (A stage past the end multiplies zeros.)
        const int rounds = (item.s_end - item.s_begin + Cfg::kGroups - 1) / Cfg::kGroups;
        int st = item.s_begin + group;
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            issue(d * Cfg::kSlotBytes, st + d * Cfg::kGroups, [&](uint32_t at, int nst) { op.load(lds, ring + d * Cfg::kSlotBytes + Cfg::kABytes, at, nst); });
        typename Op::Fragments bf[2];
        int4v_t af[2][RB][Op::kAChunks];
        typename Op::Weights raw;
        uint32_t slot = 0;
        // the loads of the oldest stage in flight have landed: this wave's by its own count, the others' behind the barrier
        auto arrive = [&](auto newer_tag) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(decltype(newer_tag)::value * Cfg::kLoads));
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto read_a = [&](auto &dst, uint32_t at) {
            mid_for<0, RB>([&](auto r) {
                mid_for<0, Op::kAChunks>([&](auto q) {
                    constexpr int R = decltype(r)::value, Q = decltype(q)::value;
                    dst[R][Q] = lds_read_b128_early<R * 16 * Cfg::kRowBytes>(af_addr[Q] + at);
                });
            });
        };
        auto settle_a = [&](auto &dst, int stage) {
            mid_for<0, RB>([&](auto r) {
                constexpr int R = decltype(r)::value;
                if constexpr (Op::kAChunks == 1) lds_wait_keep_newer<0>(dst[R][0]);
                else lds_wait_keep_newer<0>(dst[R][0], dst[R][1]);
            });
            if (stage * Op::kStageK + Op::kStageK > k)  // the stage that K ends in
                mid_for<0, RB>([&](auto r) { op.mask(dst[decltype(r)::value], stage, kg); });
        };
        arrive(MidStatic<DEPTH - 1>());
        op.read(raw, ring + Cfg::kABytes);
        read_a(af[0], 0);
        op.template settle<RB * Op::kAChunks>(raw);
        op.widen(raw, bf[0], st);
        settle_a(af[0], st);
        auto round = [&](auto b_tag) {
            constexpr int B = decltype(b_tag)::value;
            arrive(MidStatic<DEPTH - 2>());
            issue(slot, st + DEPTH * Cfg::kGroups, [&](uint32_t at, int nst) { op.load(lds, ring + slot + Cfg::kABytes, at, nst); });
            slot = slot + Cfg::kSlotBytes == DEPTH * Cfg::kSlotBytes ? 0 : slot + Cfg::kSlotBytes;
            st += Cfg::kGroups;
            op.read(raw, ring + slot + Cfg::kABytes);
            read_a(af[B ^ 1], slot);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int kAhead = RB / 4 > 0 ? RB / 4 : 1;  // row blocks whose MFMAs cover the reads' latency
            mid_for<0, kAhead>([&](auto r) { op.multiply(af[B][decltype(r)::value], bf[B], acc[decltype(r)::value], r); });
            __builtin_amdgcn_sched_barrier(0);
            op.template settle<RB * Op::kAChunks>(raw);
            op.widen(raw, bf[B ^ 1], st);
            mid_for<kAhead, RB>([&](auto r) { op.multiply(af[B][decltype(r)::value], bf[B], acc[decltype(r)::value], r); });
            constexpr int kLeft = (RB - kAhead) * Op::kMfmas;
            mid_for<0, kLeft>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (Op::kWidenOps + kLeft - 1) / kLeft, 0);
            });
            if constexpr (Op::kKeep) mid_keep(bf[B ^ 1]);
            settle_a(af[B ^ 1], st);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int i = 0; i < rounds; i += 2) {
            round(MidStatic<0>());
            if (i + 1 < rounds) round(MidStatic<1>());
        }
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // nothing may land in LDS past this point
    asm volatile("" ::: "memory");

    op.factors(n0 + (wave / Cfg::kPlanes % Cfg::kGroupWaves) * Cfg::kWaveCols + ns * Cfg::kFrags);  // on their way while the sums come together

    // ---- the groups meet: thread (unit, lane) sums kFrags columns x kWidth rows of a row block ------------------------
    float4_t sum[Cfg::kHalves][Cfg::kVecs];  // [half][.]: flat index t * kWidth + row
    float *meet = reinterpret_cast<float *>(lds);
    const int plane = wave % Cfg::kPlanes, side_u = wave / Cfg::kPlanes % Cfg::kGroupWaves, rbu = wave / (Cfg::kPlanes * Cfg::kGroupWaves);
    typedef float width_t __attribute__((ext_vector_type(Cfg::kWidth)));
    static_assert(Cfg::kHalfRows * Cfg::kGroupWaves * Cfg::kPlanes == kMidWaves, "one unit per wave");
    // [group][side][plane][row block][t][lane]
    auto meet_at = [&](int g, int sd, int p, int f) {
        return reinterpret_cast<width_t *>(meet + ((((g * Cfg::kGroupWaves + sd) * Cfg::kPlanes + p) * (Cfg::kHalfRows * Cfg::kFrags) + f) * 64 + lane) * Cfg::kWidth);
    };
    mid_for<0, Cfg::kHalves>([&](auto h_tag) {
        constexpr int H = decltype(h_tag)::value;
        __syncthreads();
        mid_for<0, Cfg::kHalfRows * Cfg::kFrags>([&](auto f_tag) {
            constexpr int F = decltype(f_tag)::value;
            const float4_t v = acc[H * Cfg::kHalfRows + F / Cfg::kFrags][F % Cfg::kFrags];
#pragma unroll
            for (int p = 0; p < Cfg::kPlanes; ++p) {
                width_t part;
#pragma unroll
                for (int e = 0; e < Cfg::kWidth; ++e) part[e] = v[p * Cfg::kWidth + e];
                *meet_at(group, side, p, F) = part;
            }
        });
        __syncthreads();
        float total[Cfg::kFrags * Cfg::kWidth];
#pragma unroll
        for (int e = 0; e < Cfg::kFrags * Cfg::kWidth; ++e) total[e] = 0.f;
#pragma unroll
        for (int g = 0; g < Cfg::kGroups; ++g)
#pragma unroll
            for (int t = 0; t < Cfg::kFrags; ++t) {
                const width_t part = *meet_at(g, side_u, plane, rbu * Cfg::kFrags + t);
#pragma unroll
                for (int e = 0; e < Cfg::kWidth; ++e) total[t * Cfg::kWidth + e] += part[e];
            }
#pragma unroll
        for (int e = 0; e < Cfg::kFrags * Cfg::kWidth; ++e) sum[H][e / 4][e % 4] = total[e];
    });

    // ---- the pieces of a tile meet: the last to arrive adds them in the order of K --------------------------------
    bool finish = true;
    if (parts > 1) {
        constexpr int kAgentScope = 1 << 4;  // sc1
        constexpr int kVec = Cfg::kHalves * Cfg::kVecs;
        constexpr int kOutside = 0x7FFFFFF0;
        auto store_of = [&](int p) {
            return partials + int64_t(item.tile * parts + p) * Cfg::kTileFloats;
        };
        const __amdgpu_buffer_rsrc_t own = __builtin_amdgcn_make_buffer_rsrc(store_of(item.part), 0, Cfg::kTileFloats * 4, 0x00020000);
#pragma unroll
        for (int h = 0; h < Cfg::kHalves; ++h) {
            const int off = (h * Cfg::kHalfRows + rbu) * 16 < rows ? tid * 16 : kOutside;
#pragma unroll
            for (int e = 0; e < Cfg::kVecs; ++e)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v_t, sum[h][e]), own, off, (h * Cfg::kVecs + e) * (kMidThreads * 16), kAgentScope);
        }
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // every store of this lane has been acknowledged (they write through)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        uint32_t *counter = counters + item.tile * kCounterWords;
        if (tid == 0) {
            const uint32_t old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = (old == uint32_t(parts - 1));
            if (*flag) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        finish = *flag != 0;
        if (finish) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            // 16 loads of a thread in flight at a time (pieces past the last read a buffer of no bytes)
            constexpr int kBatch = 16 / kVec;
#pragma unroll
            for (int h = 0; h < Cfg::kHalves; ++h)
#pragma unroll
                for (int e = 0; e < Cfg::kVecs; ++e) sum[h][e] = float4_t{0.f, 0.f, 0.f, 0.f};
            for (int p0 = 0; p0 < parts; p0 += kBatch) {
                uint4v_t v[kBatch][kVec];
#pragma unroll
                for (int b = 0; b < kBatch; ++b) {
                    const bool in = p0 + b < parts;
                    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(store_of(in ? p0 + b : item.part), 0, in ? Cfg::kTileFloats * 4 : 0, 0x00020000);
#pragma unroll
                    for (int h = 0; h < Cfg::kHalves; ++h) {
                        const int off = in && (h * Cfg::kHalfRows + rbu) * 16 < rows ? tid * 16 : kOutside;
#pragma unroll
                        for (int e = 0; e < Cfg::kVecs; ++e)
                            v[b][h * Cfg::kVecs + e] = __builtin_amdgcn_raw_buffer_load_b128(from, off, (h * Cfg::kVecs + e) * (kMidThreads * 16), kAgentScope);
                    }
                }
#pragma unroll
                for (int b = 0; b < kBatch; ++b)
#pragma unroll
                    for (int h = 0; h < Cfg::kHalves; ++h)
#pragma unroll
                        for (int e = 0; e < Cfg::kVecs; ++e) sum[h][e] += __builtin_bit_cast(float4_t, v[b][h * Cfg::kVecs + e]);
            }
        }
    }
    if (finish) {
#pragma unroll
        for (int h = 0; h < Cfg::kHalves; ++h)
#pragma unroll
            for (int r = 0; r < Cfg::kWidth; ++r) {
                const int row = (h * Cfg::kHalfRows + rbu) * 16 + 4 * kg + plane * Cfg::kWidth + r;
                float out[Cfg::kFrags];
#pragma unroll
                for (int t = 0; t < Cfg::kFrags; ++t) out[t] = sum[h][(t * Cfg::kWidth + r) / 4][(t * Cfg::kWidth + r) % 4];
                if (row < rows) op.store(m0 + row, n0 + side_u * Cfg::kWaveCols + ns * Cfg::kFrags, out);
            }
    }
}

// What a launch costs in microseconds: the workgroups of a CU one after the other, each with its fixed part and its rounds of
// the groups, and, where K is cut, once the exchange of `parts` partial tiles: that of the first workgroups of a CU runs beside the next ones (counted with
// each of them, pieces that take two and three turns were estimated 25 and 50 % too high: 1900 splits of two turns of int8 and int4 take 0.95 to 0.98 of this, 890 of three 0.93 to 0.94. int4
// 171 x 9600 x 6016, in one and in three pieces, 55.6 and 50.5 us). The coefficients are fits to the times of every tile height and
// number of pieces (430 to 1700 each) on 100 to 430 shapes of 17 to 1100 rows, K and N of 1024 to 11008 (FP8 8192), of which they leave 3 to 8 %;
// not those of K-contiguous int8 and of int4 in groups of odd multiples of 32, which are older and stand for a slower exchange (the former 17 % too high).
// The choices they make cost over the best tile and split, from the last-level cache and from memory: int8 0.4 and 1.6 % in the mean of 333 shapes, int4 0.3 and 0.3 of
// 202, FP8 0.6 and 0.4 of 427, block-scaled 0.5 and 0.7 of 424.
// `full_round` (0: not known) is the least a round takes with every CU at work: the weights of a round then come at the
// rate of the memory, once for all row tiles of a column tile (up to eight are in step). `exchange_piece` (0: in the others): what every piece of the launch adds to an exchange, all of them meeting at the same time.
struct MidCost {
    double fixed, round, exchange, exchange_part, full_round, exchange_piece;
};

struct MidChoice {
    int64_t parts = 0, share = 0;
    double us = 1e30;
    double busy_us = 1e30;  // the same with full_round, for the comparison with another kernel
};
// The K split of the smallest cost. Without a workspace (or too little of it) the tiles are computed whole.
template <class Op, int RB, int DEPTH>
MidChoice mid_choose(const MidCost &cost, const Workspace &ws, int64_t m, int64_t n, int64_t k) {
    using Cfg = MidCfg<Op, RB, DEPTH>;
    const int64_t row_tiles = cdiv(m, RB * 16), tiles = row_tiles * cdiv(n, Cfg::kPitch), stages = cdiv(k, Op::kStageK), cus = std::max(1, device_cus());
    int64_t most = 8;
    if (ws.counters == nullptr || tiles > cus) most = 1;
    else most = std::min(most, ws.scratch_bytes / (tiles * Cfg::kTileFloats * 4));
    MidChoice best;
    for (int64_t p = 1; p <= std::max<int64_t>(1, most); ++p) {
        const int64_t rounds = cdiv(cdiv(stages, p), Cfg::kGroups), share = rounds * Cfg::kGroups, parts = cdiv(stages, share);
        const double exchange = parts > 1 ? cost.exchange + double(parts) * (cost.exchange_part + double(tiles) * cost.exchange_piece) : 0.0;
        const double us = double(cdiv(tiles * parts, cus)) * (cost.fixed + double(rounds) * cost.round) + exchange;
        if (us >= best.us) continue;
        const auto batch = [&](int64_t active) {  // workgroups side by side
            return active == 0 ? 0.0 : cost.fixed + double(rounds) * std::max(cost.round, cost.full_round * double(active) / double(cus * std::min<int64_t>(8, row_tiles)));
        };
        best = MidChoice{parts, share, us, double(tiles * parts / cus) * batch(cus) + batch(tiles * parts % cus) + exchange};
    }
    return best;
}

template <class Op, int RB, int DEPTH>
void mid_launch(const MidChoice &choice, const void *a, const void *w, int64_t a_stride, int64_t w_stride, const typename Op::Args &args,
                int64_t m, int64_t n, int64_t k, const Workspace &ws, hipStream_t stream) {
    using Cfg = MidCfg<Op, RB, DEPTH>;
    const int64_t tiles_m = cdiv(m, RB * 16), tiles_n = cdiv(n, Cfg::kPitch), items = tiles_m * tiles_n * choice.parts;
    QMM_CHECK(items < (int64_t(1) << 28), "problem too large for one launch");
    static_assert(256 * kCounterWords <= kExchangeLostWord, "one counter per tile that is cut");
    allow_dynamic_lds(reinterpret_cast<const void *>(gemm_mid_kernel<Op, RB, DEPTH>), Cfg::kLdsBytes);
    launch(gemm_mid_kernel<Op, RB, DEPTH>, dim3(uint32_t(8 * cdiv(items, 8))), dim3(kMidThreads), size_t(Cfg::kLdsBytes), stream,
           static_cast<const char *>(a), static_cast<const char *>(w), int(a_stride), int(w_stride), int(k), int(m), int(n), int(tiles_m),
           int(tiles_n), int(cdiv(k, Op::kStageK)), int(choice.parts), int(choice.share), mid_magic(int(tiles_m)), mid_magic(int(choice.parts)),
           reinterpret_cast<float *>(ws.scratch), ws.counters, args);
}

}  // namespace qmm
