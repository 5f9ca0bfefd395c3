// Measurement and test hooks of libhidet_qmm.so (include/hidet_qmm_bench.h): events and the per-launch timing hook,
// kernels that only read, and the host-side switch of the exchange's give-up limit. Nothing an operator call needs.
#include "common.h"
#include "skinny_fp8_tall.h"
#include "skinny_w4a16_small.h"
#include "skinny_w8a16_nk_tall.h"
#include "skinny_w8a16_small.h"
#include "../../include/hidet_qmm_bench.h"

HIDET_API void *hidet_qmm_event_create(void) {
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) {
        hidet_set_last_error("hipEventCreate failed");
        return nullptr;
    }
    return e;
}

HIDET_API void hidet_qmm_event_destroy(void *event) {
    if (event) (void)hipEventDestroy(static_cast<hipEvent_t>(event));
}

HIDET_API void hidet_qmm_event_record(void *event, void *stream) {
    QMM_ENTRY_BEGIN
    QMM_HIP(hipEventRecord(static_cast<hipEvent_t>(event), static_cast<hipStream_t>(stream)));
    QMM_ENTRY_END
}

HIDET_API void hidet_qmm_event_synchronize(void *event) {
    QMM_ENTRY_BEGIN
    QMM_HIP(hipEventSynchronize(static_cast<hipEvent_t>(event)));
    QMM_ENTRY_END
}

HIDET_API float hidet_qmm_event_elapsed_ms(void *start, void *stop) {
    float ms = -1.0f;
    hipError_t e = hipEventElapsedTime(&ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop));
    if (e != hipSuccess) {
        hidet_set_last_error(hipGetErrorString(e));
        return -1.0f;
    }
    return ms;
}

HIDET_API void hidet_qmm_arm_timing(void *start_event, void *stop_event) {
    qmm::TimingSlot &ts = qmm::timing_slot();
    ts.start = static_cast<hipEvent_t>(start_event);
    ts.stop = static_cast<hipEvent_t>(stop_event);
}

HIDET_API void hidet_qmm_gemv_ring_timed(const void *a, const void *const *weights, const void *const *scales, void *const *outs,
                                         int ring, int launches, int64_t m, int64_t k, int64_t n, int64_t lda, void *workspace,
                                         int64_t workspace_bytes, void *const *start_events, void *const *stop_events,
                                         void *stream) {
    if (a == nullptr || weights == nullptr || scales == nullptr || outs == nullptr || ring <= 0 || launches < 0) {
        hidet_set_last_error("hidet_qmm_gemv_ring_timed: null array or empty ring");
        return;
    }
    for (int i = 0; i < launches; ++i) {
        if (start_events != nullptr && stop_events != nullptr) hidet_qmm_arm_timing(start_events[i], stop_events[i]);
        const int r = i % ring;
        // the operator's own entry point, called in a loop without the host interpreter between two launches; an error
        // (last-error string set) ends the loop
        hidet_symmetric_quant_matmul_f16_i8(a, weights[r], scales[r], outs[r], m, k, n, lda, 0, workspace, workspace_bytes, stream);
        if (qmm::error_pending()) return;
    }
}

HIDET_API void hidet_qmm_set_exchange_spin_limit(int limit) {
    qmm::exchange_spin_limit().store(limit < 0 ? qmm::kExchangeSpinLimit : limit, std::memory_order_relaxed);
}

// ---- which kernel a call took, and the kernels of strips by their variant ---------------------------------------------
HIDET_API const char *hidet_qmm_last_launch(int64_t *workgroups, int64_t *threads) {
    const qmm::TimingSlot &ts = qmm::timing_slot();
    if (workgroups != nullptr) *workgroups = ts.workgroups;
    if (threads != nullptr) *threads = ts.threads;
    const char *name = ts.kernel != nullptr ? hipKernelNameRefByPtr(ts.kernel, nullptr) : nullptr;
    return name != nullptr ? name : "";
}

namespace {
void check_strip(int row_blocks, bool columns, int64_t m, int64_t k, int64_t n) {
    QMM_CHECK(row_blocks >= 1 && row_blocks <= 4 && columns, "there is no such variant of the kernel");
    QMM_CHECK(m > 0 && k > 0 && n > 0 && m < (int64_t(1) << 24) && k < (int64_t(1) << 24) && n < (int64_t(1) << 24), "extents out of range");
}
}  // namespace

HIDET_API void hidet_qmm_strips_f16_i8(int row_blocks, int columns, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                                       int64_t n, int64_t lda, void *stream) {
    QMM_ENTRY_BEGIN
    check_strip(row_blocks, columns == 2 || columns == 4, m, k, n);
    QMM_CHECK(a && w && scale && c && lda >= k && qmm::skinny_w8a16_small_supported(a, n, k, lda), "not a form that the kernel takes");
    qmm::SkinnySmallPlan plan;
    plan.rb = row_blocks;
    plan.cb = columns;
    qmm::skinny_w8a16_small_launch(plan, a, w, scale, bias, c, m, k, n, lda, static_cast<hipStream_t>(stream));
    QMM_ENTRY_END
}

HIDET_API void hidet_qmm_strips_f16_i8_nk(int row_blocks, int groups, const void *a, const void *w_nk, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                                          int64_t n, int64_t lda, int64_t ldw, void *stream) {
    QMM_ENTRY_BEGIN
    check_strip(row_blocks, groups == 1 || groups == 2, m, k, n);
    QMM_CHECK(a && w_nk && scale && c && lda >= k && ldw >= k && k % 16 == 0 && ldw % 16 == 0 && lda % 8 == 0 && qmm::aligned(a, 16) && qmm::aligned(w_nk, 16),
              "not a form that the kernel takes");
    qmm::SkinnyNkTallPlan plan;
    plan.rb = row_blocks;
    plan.cg = groups;
    qmm::skinny_w8a16_nk_tall_launch(plan, a, w_nk, scale, bias, c, m, k, n, lda, ldw, static_cast<hipStream_t>(stream));
    QMM_ENTRY_END
}

HIDET_API void hidet_qmm_strips_w4a16(int row_blocks, int columns, int waves, const void *a, const void *w, const void *scales, const void *bias, void *c, int64_t m,
                                      int64_t k, int64_t n, int64_t lda, int group_size, int dtype, void *stream) {
    QMM_ENTRY_BEGIN
    check_strip(row_blocks, (columns == 2 || columns == 4) && (waves == 8 || (waves == 16 && row_blocks == 1 && columns == 2)), m, k, n);
    QMM_CHECK(a && w && scales && c && lda >= k && (dtype == HIDET_QMM_BF16 || dtype == HIDET_QMM_F16) && group_size > 0 && k % group_size == 0 &&
                  qmm::skinny_w4a16_small_supported(a, scales, n, k, lda, group_size),
              "not a form that the kernel takes");
    qmm::SkinnyW4SmallPlan plan;
    plan.rb = row_blocks;
    plan.cb = columns;
    plan.waves = waves;
    qmm::skinny_w4a16_small_launch(plan, a, w, scales, bias, c, m, k, n, lda, group_size, dtype, static_cast<hipStream_t>(stream));
    QMM_ENTRY_END
}

HIDET_API void hidet_qmm_strips_f8(int row_blocks, int groups, int block_scaled, const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k, int64_t lda,
                                   int64_t ldb, int out_dtype, const void *scale_a, const void *scale_b, void *stream) {
    QMM_ENTRY_BEGIN
    check_strip(row_blocks, groups == 1 || groups == 2, m, k, n);
    QMM_CHECK(a && b && c && lda >= k && ldb >= k && k % 16 == 0 && lda % 16 == 0 && ldb % 16 == 0 && qmm::aligned(a, 16) && qmm::aligned(b, 16) &&
                  (out_dtype == HIDET_QMM_F32 || out_dtype == HIDET_QMM_F16 || out_dtype == HIDET_QMM_BF16 || out_dtype == HIDET_QMM_E4M3) &&
                  (!block_scaled || (scale_a && scale_b && k % 128 == 0 && n % 128 == 0)),
              "not a form that the kernel takes");
    qmm::SkinnyFp8TallPlan plan;
    plan.rb = row_blocks;
    plan.cg = groups;
    qmm::skinny_fp8_tall_launch(plan, block_scaled != 0, a, b, c, m, n, k, lda, ldb, out_dtype, scale_a, scale_b, static_cast<hipStream_t>(stream));
    QMM_ENTRY_END
}

// ---- what a kernel that only reads can get out of the memory system ------------------------------------------------
namespace {
constexpr int kProbeBlockBytes = 32768;  // 256 threads x 8 loads x 16 bytes, contiguous per workgroup
constexpr int kNonTemporal = 2;          // cache policy bits of a buffer load: sc0 = 1, nt = 2, sc1 = 16

__global__ __launch_bounds__(256) void read_probe_kernel(const uint4 *__restrict__ src, uint32_t *__restrict__ sink) {
    const uint4 *p = src + int64_t(blockIdx.x) * (kProbeBlockBytes / 16) + threadIdx.x;
    uint4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = p[j * 256];
    uint32_t acc = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += v[j].x ^ v[j].y ^ v[j].z ^ v[j].w;
    if (acc == 0x9E3779B9u) sink[0] = acc;  // practically never true; keeps the loads alive
}

// The loads of the decode kernel over an int8 matrix w[k, n] and nothing else: the (256-column tile, row) space is cut
// into `workgroups` x 8 equal runs, one per wave; a wave walks its run in steps of 32 rows, a lane fetching 16 bytes of
// each of 8 rows per step (a wave instruction covers four 256-byte row segments n bytes apart), one step in flight.
// `contiguous`: the same bytes per wave, but as one 1 KiB piece per wave instruction.
__global__ __launch_bounds__(512) void pattern_probe_kernel(const char *__restrict__ w, int n, int k, int tiles, int contiguous,
                                                           uint32_t *__restrict__ sink) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lg = lane >> 4, cl = lane & 15;
    const int64_t space = int64_t(tiles) * k, runs = int64_t(gridDim.x) * 8;
    const int64_t me = int64_t(blockIdx.x) * 8 + wave;
    int64_t f0 = me * space / runs;
    const int64_t f1 = (me + 1) * space / runs;
    uint32_t acc = 0;
    if (contiguous) {
        const int64_t b0 = f0 * 256, b1 = f1 * 256;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w + b0), 0, int(b1 - b0), 0x00020000);
        const int loads = int((b1 - b0 + 1023) / 1024);
        uint32_t off = lane * 16;
        for (int s = 0; s < loads; s += 8) {
            qmm::uint4v_t v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + j * 1024, 0, kNonTemporal);
            off += 8 * 1024;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc += v[j][0] ^ v[j][1] ^ v[j][2] ^ v[j][3];
        }
    } else {
        while (f0 < f1) {
            const int tile = int(f0 / k);
            const int r0 = int(f0 - int64_t(tile) * k);
            const int64_t fend = f1 < int64_t(tile + 1) * k ? f1 : int64_t(tile + 1) * k;
            const int rows = int(fend - f0);
            // rows of the run, from the tile's first column: what lies behind reads as zero without going to memory
            const int64_t bytes = int64_t(rows) * n - tile * 256;
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(w + int64_t(r0) * n + tile * 256), 0, int(bytes), 0x00020000);
            uint32_t off = uint32_t(8 * lg) * uint32_t(n) + cl * 16;
            const int steps = (rows + 31) >> 5;
            for (int s = 0; s < steps; ++s) {
                qmm::uint4v_t v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + uint32_t(j) * uint32_t(n), 0, kNonTemporal);
                off += 32u * uint32_t(n);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc += v[j][0] ^ v[j][1] ^ v[j][2] ^ v[j][3];
            }
            f0 = fend;
        }
    }
    if (acc == 0x9E3779B9u) sink[0] = acc;
}
}  // namespace

HIDET_API void hidet_qmm_read_probe(const void *src, int64_t bytes, void *sink, void *stream) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(src && sink && qmm::aligned(src, 16), "null or misaligned pointer");
    QMM_CHECK(bytes > 0 && bytes % kProbeBlockBytes == 0 && bytes / kProbeBlockBytes < (int64_t(1) << 31),
              "the size must be a positive multiple of " << kProbeBlockBytes << " bytes, got " << bytes);
    qmm::launch(read_probe_kernel, dim3(uint32_t(bytes / kProbeBlockBytes)), dim3(256), 0, static_cast<hipStream_t>(stream),
                static_cast<const uint4 *>(src), static_cast<uint32_t *>(sink));
    QMM_ENTRY_END
}

HIDET_API void hidet_qmm_pattern_probe(const void *w, int64_t k, int64_t n, int workgroups, int contiguous, void *sink,
                                       void *stream) {
    QMM_ENTRY_BEGIN
    QMM_CHECK(w && sink && qmm::aligned(w, 16), "null or misaligned pointer");
    QMM_CHECK(k > 0 && n > 0 && n % 256 == 0 && k % 32 == 0, "the probe takes K a multiple of 32 and N a multiple of 256, got " << k << " x " << n);
    QMM_CHECK(workgroups > 0 && workgroups <= 65536, "workgroups must be in [1, 65536], got " << workgroups);
    // a wave's run is addressed with 31-bit offsets
    QMM_CHECK((k * (n / 256) / (int64_t(workgroups) * 8) + 64) * n < (int64_t(1) << 31), "too few workgroups for a matrix of " << k << " x " << n);
    qmm::launch(pattern_probe_kernel, dim3(uint32_t(workgroups)), dim3(512), 0, static_cast<hipStream_t>(stream),
                static_cast<const char *>(w), int(n), int(k), int(n / 256), contiguous, static_cast<uint32_t *>(sink));
    QMM_ENTRY_END
}
