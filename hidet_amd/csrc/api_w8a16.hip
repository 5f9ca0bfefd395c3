// Entry point of the W8A16 matmul: argument checks and the choice of kernel family.
#include "common.h"
#include "skinny_common.h"
#include "skinny_w8a16_nk_tall.h"
#include "skinny_w8a16_small.h"

namespace qmm {
bool skinny_w8a16_supported(const void *w, const void *scale, const void *bias, int64_t k, int64_t n);
void skinny_w8a16_launch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                         int64_t n, int64_t lda, int64_t n_out, int parallel_k_parts, const Workspace &ws, bool strict_workspace,
                         hipStream_t stream);
bool gemm_w8a16_supported(const void *a, const void *w, const void *c, int64_t m, int64_t k, int64_t n, int64_t lda);
void gemm_w8a16_launch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                       int64_t n, int64_t lda, int64_t n_out, int64_t ldc, const Workspace &ws, hipStream_t stream);
bool skinny_w8a16_nk_supported(const void *w, int64_t k, int64_t ldw);
void skinny_w8a16_nk_launch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                            int64_t n, int64_t lda, int64_t ldw, hipStream_t stream);
bool gemm_w8a16_nk_supported(const void *a, const void *w, const void *c, int64_t m, int64_t k, int64_t n, int64_t lda,
                             int64_t ldw);
bool mid_w8a16_launch(const void *a, const void *w, bool nk, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                      int64_t n, int64_t lda, int64_t ldw, int64_t n_out, int64_t ldc, double limit_us, const Workspace &ws, hipStream_t stream);
double gemm_w8a16_estimate_us(int64_t m, int64_t k, int64_t n, const Workspace &ws);
double gemm_w8a16_nk_estimate_us(int64_t m, int64_t k, int64_t n, const Workspace &ws);
void gemm_w8a16_nk_launch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                          int64_t n, int64_t lda, int64_t ldw, const Workspace &ws, hipStream_t stream);
}

using namespace qmm;

namespace {

constexpr int64_t kPanelK = 256;    // from this depth on panels of a padded weight beat the element-wise kernel on few rows
constexpr int64_t kElementWise = int64_t(1) << 20;  // products up to which a matrix is tiny
constexpr int64_t kMidRows = 1024;  // above, the prefill GEMM's tiles fill the chip on every shape

// ---- operands of sizes or alignments the matrix kernels do not take --------------------------------------------------
//
// Copies of the operands with rows of whole 16 (weight, factors) and 64 (activations) elements, zero past the originals,
// in the scratch memory: columns [n0, n0 + cols) of w[k, n] as [kp, np], the float16 activations [m, k] as [m, kp], the
// column factors as [np]. One thread per 16 bytes written. For odd N or K, and for N = 4 i + 2 above kMidRows: 203 rows x 4100 x 4098 took 29 us
// in all this way (18 us of them the GEMM; 20 as they lie on the narrow tiles), element by element 1815.
struct PadArgs {
    const int8_t *w;
    const _Float16 *a, *scale, *bias;
    int8_t *wp;
    _Float16 *ap, *scalep, *biasp;
    int64_t n, lda;
    int k, kp, n0, cols, np, m;
    uint32_t w_chunks, a_chunks;  // 16-byte pieces of the copies (none: that operand is left alone)
};
__global__ __launch_bounds__(256) void pad_operands_kernel(PadArgs p) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < p.w_chunks) {
        const uint32_t per_row = uint32_t(p.np) / 16, row = i / per_row, col = (i - row * per_row) * 16;
        uint4 v = {0u, 0u, 0u, 0u};
        if (int(row) < p.k) {
            const int8_t *src = p.w + int64_t(row) * p.n + p.n0 + col;
            if (int(col) + 16 <= p.cols) {
                __builtin_memcpy(&v, src, 16);
            } else {
                uint32_t word[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (int(col) + e < p.cols) word[e >> 2] |= uint32_t(uint8_t(src[e])) << (8 * (e & 3));
                v = uint4{word[0], word[1], word[2], word[3]};
            }
        }
        reinterpret_cast<uint4 *>(p.wp)[i] = v;
        return;
    }
    i -= p.w_chunks;
    if (i < p.a_chunks) {
        const uint32_t per_row = uint32_t(p.kp) / 8, row = i / per_row, kk = (i - row * per_row) * 8;
        half8_t v;
        const _Float16 *src = p.a + int64_t(row) * p.lda + kk;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = int(kk) + e < p.k ? src[e] : _Float16(0.0f);
        reinterpret_cast<half8_t *>(p.ap)[i] = v;
        return;
    }
    i -= p.a_chunks;
    if (p.w_chunks > 0 && i < uint32_t(p.np)) {
        const bool in = int(i) < p.cols;
        p.scalep[i] = in ? p.scale[p.n0 + i] : _Float16(0.0f);
        if (p.bias != nullptr) p.biasp[i] = in ? p.bias[p.n0 + i] : _Float16(0.0f);
    }
}

// Where the copies go: panels of `cols` columns and `rows` rows, at the end of the scratch memory (offsets from its beginning).
struct PadPlan {
    int64_t kp, rows, cols, a_bytes;
    int64_t a_at, bias_at, scale_at, w_at;
    bool copy_a;
};
// False: there is not enough scratch memory for a panel.
bool padded_plan(bool gemm, const void *a, int64_t m, int64_t k, int64_t n, int64_t lda, const Workspace &ws, PadPlan *plan) {
    PadPlan p{};
    p.kp = gemm ? cdiv(k, 64) * 64 : k;
    p.copy_a = gemm && (p.kp != k || lda % 8 != 0 || !aligned(a, 16) || (m * lda + k) * 2 >= (int64_t(1) << 31) - (1 << 20));
    const int64_t room = ws.scratch_bytes / 4 * 3;  // a quarter stays for partial tiles
    p.rows = p.copy_a ? std::min<int64_t>(m, room / 3 / (p.kp * 2) / 128 * 128) : m;
    if (p.rows <= 0) return false;
    p.a_bytes = p.copy_a ? cdiv(p.rows * p.kp * 2, 256) * 256 : 0;
    p.cols = cdiv(n, 16) * 16;  // per panel
    const int64_t per_col = p.kp + 4, fixed = p.a_bytes + 1024;
    const int64_t most = std::min<int64_t>(room - fixed, int64_t(1) << 30) / per_col;
    if (p.cols > most) p.cols = most / 256 * 256;
    if (p.cols <= 0) return false;
    // the bandwidth-bound kernel writes whole rows (one panel) and addresses a wave's rows with 31-bit offsets
    if (!gemm && (p.cols < n || (k + 192) * p.cols >= (int64_t(1) << 31) - (1 << 20))) return false;
    p.a_at = ws.scratch_bytes / 256 * 256 - p.a_bytes;
    p.bias_at = p.a_at - cdiv(p.cols * 2, 256) * 256;
    p.scale_at = p.bias_at - cdiv(p.cols * 2, 256) * 256;
    p.w_at = p.scale_at - cdiv(p.kp * p.cols, 256) * 256;
    *plan = p;
    return p.w_at >= 0;
}

// The matmul on padded copies, in panels of columns and rows that fit the scratch memory (the GEMM; without `gemm`, for up to 16 rows,
// the bandwidth-bound kernel, which reads activations of any alignment, on one panel): the copies lie at its end, what is before them is left to the GEMM's partial tiles. False: there
// is not enough of it for a panel.
bool w8a16_padded(bool gemm, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                  int64_t lda, const Workspace &ws, hipStream_t stream) {
    PadPlan plan;
    if (!padded_plan(gemm, a, m, k, n, lda, ws, &plan)) return false;
    const int64_t kp = plan.kp, rows = plan.rows, cols = plan.cols;
    const bool copy_a = plan.copy_a;
    PadArgs p{};
    p.w = static_cast<const int8_t *>(w);
    p.scale = static_cast<const _Float16 *>(scale);
    p.bias = static_cast<const _Float16 *>(bias);
    p.ap = reinterpret_cast<_Float16 *>(ws.scratch + plan.a_at);
    p.biasp = reinterpret_cast<_Float16 *>(ws.scratch + plan.bias_at);
    p.scalep = reinterpret_cast<_Float16 *>(ws.scratch + plan.scale_at);
    p.wp = reinterpret_cast<int8_t *>(ws.scratch + plan.w_at);
    p.n = n;
    p.lda = lda;
    p.k = int(k);
    p.kp = int(kp);
    Workspace left = ws;
    left.scratch_bytes = plan.w_at;
    for (int64_t n0 = 0; n0 < n; n0 += cols) {
        p.n0 = int(n0);
        p.cols = int(std::min(cols, n - n0));
        p.np = int(cdiv(p.cols, 16) * 16);
        for (int64_t m0 = 0; m0 < m; m0 += rows) {
            p.m = int(std::min(rows, m - m0));
            p.a = static_cast<const _Float16 *>(a) + m0 * lda;
            p.w_chunks = m0 == 0 ? uint32_t(kp * p.np / 16) : 0;
            p.a_chunks = copy_a ? uint32_t(p.m * kp / 8) : 0;
            const uint64_t threads = uint64_t(p.w_chunks) + p.a_chunks + (p.w_chunks > 0 ? p.np : 0);
            if (threads > 0) launch_aux(pad_operands_kernel, dim3(uint32_t((threads + 255) / 256)), dim3(256), 0, stream, p);
            const void *ap = copy_a ? static_cast<const void *>(p.ap) : static_cast<const void *>(p.a);
            _Float16 *cp = static_cast<_Float16 *>(c) + m0 * n + n0;
            const void *bp = bias != nullptr ? p.biasp : nullptr;
            if (gemm && p.m <= kMidRows &&
                mid_w8a16_launch(ap, p.wp, false, p.scalep, bp, cp, p.m, kp, p.np, copy_a ? kp : lda, p.np, p.cols, n,
                                 gemm_w8a16_estimate_us(p.m, kp, p.np, left), left, stream))
                continue;
            if (gemm) gemm_w8a16_launch(ap, p.wp, p.scalep, bp, cp, p.m, kp, p.np, copy_a ? kp : lda, p.cols, n, left, stream);
            else skinny_w8a16_launch(ap, p.wp, p.scalep, bp, cp, p.m, k, p.np, lda, p.cols, 0, left, false, stream);
        }
    }
    return true;
}

// What the copy and the prefill tiles take together (the copy: 4100 x 4098 10.9 us, 1026 x 2050 4.0). No limit where no copy would be made, because
// the matrix is tiny or the scratch memory holds no panel of it, and the call would run element by element.
double padded_estimate_us(const void *a, int64_t m, int64_t k, int64_t n, int64_t lda, const Workspace &ws) {
    PadPlan plan;
    if (m * k * n <= kElementWise || !((m <= 16 && padded_plan(false, a, m, k, n, lda, ws, &plan)) ||
                                       ((m > 16 || k >= kPanelK) && padded_plan(true, a, m, k, n, lda, ws, &plan))))
        return 1e29;
    return 3.0 + double(k) * double(n) / 2.15e6 + gemm_w8a16_estimate_us(m, cdiv(k, 64) * 64, cdiv(n, 16) * 16, ws);
}

// Checks and kernel choice shared by the two row-major entry points. `strict_workspace`: a bandwidth-bound launch whose
// K split does not fit the scratch memory is an error instead of a launch with fewer K slices.
void w8a16_dispatch(const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                    int64_t lda, int parallel_k_parts, void *workspace, int64_t workspace_bytes, bool strict_workspace,
                    hipStream_t stream) {
    QMM_CHECK(m >= 0 && k >= 0 && n >= 0, "negative extent: m=" << m << " k=" << k << " n=" << n);
    QMM_CHECK(lda >= k, "row stride of a (" << lda << ") is smaller than K (" << k << ")");
    QMM_CHECK(k < (int64_t(1) << 31) && n < (int64_t(1) << 31) && m < (int64_t(1) << 31), "extent exceeds 2^31");
    QMM_CHECK(parallel_k_parts >= 0, "parallel_k_parts must be >= 0");
    if (m == 0 || n == 0) return;
    QMM_CHECK(a && w && scale && c, "null tensor pointer");
    QMM_CHECK(aligned(a, 2) && aligned(scale, 2) && aligned(c, 2) && aligned(bias, 2), "float16 tensors must be 2-byte aligned");
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    // Up to 16 rows one pass of the bandwidth-bound kernel serves; beyond that every 16 rows would cost another pass
    // over the weights, and the GEMMs take over: narrow tiles (gemm_mid.h) or the prefill tiles, whichever is estimated to be
    // the faster (K=4096, N=11008, weights from HBM: narrow 14.6 / 18.3 / 24.1 / 34.6 us at M=17 / 64 / 128 / 256, prefill tiles 17.0 /
    // 20.6 / 29.2 / 39.1; at M=512 64 against 57; a wide weight, 4096 x 57344: narrow 54 / 65 us at M=17 / 64, prefill tiles 46 / 52). For 9 to 16 rows the bandwidth-bound kernel is
    // ahead of the prefill tiles on every shape measured (4096 x 11008: 13.5 - 14.1 against 16.5 us; 8192 x 8192: 16.9 - 18.2
    // against 22.4; 8192 x 28672: 42.6 - 43.8 against 49), but not of the narrow ones (below).
    // Small weights take a kernel without an exchange where it is ahead of the others by 8 % (skinny_w8a16_small.hip).
    const SkinnySmallPlan small = m <= kMidRows && parallel_k_parts == 0 ? skinny_w8a16_small_plan(a, m, n, k, lda) : SkinnySmallPlan();
    const double small_us = 1.08 * small.us;
    const auto small_launch = [&](double limit) {
        if (small_us > limit) return false;
        skinny_w8a16_small_launch(small, a, w, scale, bias, c, m, k, n, lda, stream);
        return true;
    };
    if (m > 16 && k > 0 && n % 4 != 2) {
        const bool gemm = gemm_w8a16_supported(a, w, c, m, k, n, lda);
        const double limit = gemm ? gemm_w8a16_estimate_us(m, k, n, ws) : 1e29;
        if (m <= kMidRows && mid_w8a16_launch(a, w, false, scale, bias, c, m, k, n, lda, n, n, n, std::min(limit, small_us), ws, stream)) return;
        if (small_launch(limit)) return;
        if (gemm) {
            gemm_w8a16_launch(a, w, scale, bias, c, m, k, n, lda, n, n, ws, stream);
            return;
        }
    }
    // A decode batch that the narrow tiles serve sooner: ahead by 3 % (of 512 shapes 246 go there, 17 % faster in the mean, 13 on weights from memory; 5 and 20 of them
    // are more than 3 % slower).
    if (m <= 16 && parallel_k_parts == 0 && k > 0 && n % 4 == 0 && skinny_w8a16_supported(w, scale, bias, k, n)) {
        const double limit = skinny_estimate_us(true, m, k, n) / 1.03;
        if (k >= kSkinnyEstimateK && mid_w8a16_launch(a, w, false, scale, bias, c, m, k, n, lda, n, n, n, std::min(limit, small_us), ws, stream)) return;
        if (small_launch(limit)) return;
    }
    // N = 4 i + 2 on the narrow tiles as it lies, also for one pass of 16 rows (which the bandwidth-bound kernel takes on a copy only),
    // unless the copy and the prefill tiles are estimated to take less. us, on copies against that: 1 x 1026 x 2050 14.0 and 7.6, 16 x 4096 x 4098
    // 21.3 and 11.1, 203 x 4096 x 4098 27.9 and 20.4, 600 x 4096 x 4098 45 and 37, 16 x 8192 x 8190 35 and 18; 1 x 2002 x 514 element by element 193
    // and 7.7 (0.1 us per k whatever else).
    if (n % 4 != 0 && k > 0 && m <= kMidRows && (k >= 64 || m * k * n > kElementWise)) {
        const double limit = padded_estimate_us(a, m, k, n, lda, ws);
        if (n % 4 == 2 && mid_w8a16_launch(a, w, false, scale, bias, c, m, k, n, lda, n, n, n, std::min(limit, small_us), ws, stream)) return;
        if (small_launch(limit)) return;
    }
    // Sizes the GEMM does not take (K no multiple of 64, N of 4): up to 32 rows two passes of the bandwidth-bound kernel,
    // which takes any K and N a multiple of 4, cost less than a copy of the weight and a GEMM; more rows and other N take the
    // copy. Tiny matrices are left to the element-wise kernel.
    const bool skinny = skinny_w8a16_supported(w, scale, bias, k, n);
    if (k > 0 && (!skinny || m > 32) && m * k * n > kElementWise) {
        if (m <= 16 && w8a16_padded(false, a, w, scale, bias, c, m, k, n, lda, ws, stream)) return;
        // Up to 16 rows of a weight whose copy does not fit the scratch memory whole: panels for the GEMM (8192 x 8190, one row: 52 us,
        // element by element 3037; 256 x 300002 60 and 101; at a depth of 64 such a weight has threads enough for the latter).
        if ((m > 16 || k >= kPanelK) && w8a16_padded(true, a, w, scale, bias, c, m, k, n, lda, ws, stream)) return;
    }
    skinny_w8a16_launch(a, w, scale, bias, c, m, k, n, lda, n, parallel_k_parts, ws, strict_workspace, stream);
}

// Checks and kernel choice shared by the two entry points for K-contiguous weights.
void w8a16_nk_dispatch(const void *a, const void *w_nk, const void *scale, const void *bias, void *c, int64_t m, int64_t k,
                       int64_t n, int64_t lda, int64_t ldw, void *workspace, int64_t workspace_bytes, hipStream_t stream) {
    QMM_CHECK(m >= 0 && k >= 0 && n >= 0, "negative extent: m=" << m << " k=" << k << " n=" << n);
    QMM_CHECK(lda >= k && ldw >= k, "row strides (" << lda << ", " << ldw << ") must be at least K (" << k << ")");
    QMM_CHECK(k < (int64_t(1) << 31) && n < (int64_t(1) << 31) && m < (int64_t(1) << 31), "extent exceeds 2^31");
    QMM_CHECK(workspace_bytes >= 0 && (workspace == nullptr || aligned(workspace, 16)),
              "the workspace must be 16-byte aligned (or NULL: no tile is computed in K ranges)");
    if (m == 0 || n == 0) return;
    QMM_CHECK(a && w_nk && scale && c, "null tensor pointer");
    QMM_CHECK(aligned(a, 2) && aligned(scale, 2) && aligned(c, 2) && aligned(bias, 2), "float16 tensors must be 2-byte aligned");
    QMM_CHECK(skinny_w8a16_nk_supported(w_nk, k, ldw),
              "K-contiguous weights need K and the row stride to be multiples of 16 and a 16-byte aligned pointer, got K=" << k
                                                                                                                         << " ldw=" << ldw);
    // More than one pass of 16 rows: up to 64 the kernel without an exchange for small weights or the narrow tiles reading the same layout (4096 x 4096, 49 rows: 12.3 us, the prefill
    // tiles 19.9) unless they are estimated to take longer, which they do on very wide weights (1024 x 131072, 33 rows: 61 us
    // against 47; 4096 x 57344, 64 rows: 84 against 78); else the prefill tiles, where their conditions hold.
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    const bool gemm = m > 16 && gemm_w8a16_nk_supported(a, w_nk, c, m, k, n, lda, ldw);
    if (m > 16 && m <= 64 && k > 0) {
        const double gemm_us = gemm ? gemm_w8a16_nk_estimate_us(m, k, n, ws) : 1e29;
        const SkinnyNkTallPlan tall = skinny_w8a16_nk_tall_plan(a, m, n, k, lda);
        if (mid_w8a16_launch(a, w_nk, true, scale, bias, c, m, k, n, lda, ldw, n, n, std::min(gemm_us, 1.2 * tall.us), ws, stream)) return;
        if (1.2 * tall.us <= gemm_us) {
            skinny_w8a16_nk_tall_launch(tall, a, w_nk, scale, bias, c, m, k, n, lda, ldw, stream);
            return;
        }
    }
    if (gemm) gemm_w8a16_nk_launch(a, w_nk, scale, bias, c, m, k, n, lda, ldw, ws, stream);
    else
        skinny_w8a16_nk_launch(a, w_nk, scale, bias, c, m, k, n, lda, ldw, stream);
}

// Scratch memory of hidet_symmetric_quant_matmul_f16_i8_static, used exactly like a caller's workspace of that size
// (counters, mailbox, scratch). One copy per GPU, loaded with the library's code object (zero-filled then; the kernels
// return every counter and every mailbox word they used to zero).
constexpr int64_t kStaticScratchBytes = HIDET_QMM_STATIC_SCRATCH_BYTES;
static_assert(kStaticScratchBytes > kCounterBytes && kStaticScratchBytes % 256 == 0, "counters plus partial tiles");
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each GPU, looked up on the first call there
std::mutex g_scratch_mu;

// The device address of this GPU's copy of `scratch`. In host code the array's name is only a handle for the runtime's
// symbol lookup, never a pointer a kernel may be given.
void *static_scratch_of_current_device() {
    int device = -1;
    QMM_HIP(hipGetDevice(&device));
    QMM_CHECK(device >= 0 && device < kMaxDevices, "device ordinal " << device << " out of range");
    std::lock_guard<std::mutex> guard(g_scratch_mu);
    if (g_scratch_ptr[device] == nullptr) {
        void *ptr = nullptr;
        QMM_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        QMM_CHECK(ptr != nullptr && aligned(ptr, 256), "the runtime returned no usable address for the static scratch array");
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

}  // namespace

HIDET_API void hidet_symmetric_quant_matmul_f16_i8(const void *a, const void *w, const void *scale, void *c, int64_t m,
                                                   int64_t k, int64_t n, int64_t lda, int parallel_k_parts,
                                                   void *workspace, int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    w8a16_dispatch(a, w, scale, nullptr, c, m, k, n, lda, parallel_k_parts, workspace, workspace_bytes, false,
                   static_cast<hipStream_t>(stream_));
    QMM_ENTRY_END
}

HIDET_API int64_t hidet_qmm_static_scratch_bytes(void) { return kStaticScratchBytes; }

namespace {
__global__ __launch_bounds__(256) void zero_fill_kernel(uint4 *__restrict__ dst, int64_t count) {
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < count; i += int64_t(gridDim.x) * 256) dst[i] = uint4{0u, 0u, 0u, 0u};
}
}  // namespace

HIDET_API int hidet_qmm_exchange_status(const void *workspace, int64_t workspace_bytes, void *stream_) {
    try {
        const void *base = workspace;
        if (base == nullptr) {
            base = static_scratch_of_current_device();
            workspace_bytes = kStaticScratchBytes;
        }
        hipStream_t stream = static_cast<hipStream_t>(stream_);
        uint32_t word = 0;
        if (workspace_bytes >= kCounterBytes)  // else: no counter block, no exchange ever ran on it
            QMM_HIP(hipMemcpyAsync(&word, static_cast<const uint32_t *>(base) + kExchangeLostWord, sizeof(word), hipMemcpyDeviceToHost, stream));
        QMM_HIP(hipStreamSynchronize(stream));
        return word != 0u ? 1 : 0;
    } catch (const std::exception &e) {
        hidet_set_last_error(e.what());
    } catch (...) {
        hidet_set_last_error("unknown error");
    }
    return -1;
}

HIDET_API void hidet_qmm_exchange_reset(void *workspace, int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    if (workspace == nullptr) {
        workspace = static_scratch_of_current_device();
        workspace_bytes = kStaticScratchBytes;
    }
    QMM_CHECK(aligned(workspace, 16), "the workspace must be 16-byte aligned");
    const Workspace ws = split_workspace(workspace, workspace_bytes);
    if (ws.counters == nullptr) return;
    // a fill kernel, not a memset node: callers may capture this into a graph
    const int64_t count = (kCounterBytes + ws.mailbox_bytes) / 16;
    launch_aux(zero_fill_kernel, dim3(uint32_t(std::min<int64_t>(2048, cdiv(count, 256)))), dim3(256), 0, static_cast<hipStream_t>(stream_),
               static_cast<uint4 *>(workspace), count);
    QMM_ENTRY_END
}

HIDET_API void hidet_symmetric_quant_matmul_f16_i8_static(const void *a, const void *w, const void *scale, void *c, int64_t m,
                                                          int64_t k, int64_t n, int64_t lda, int parallel_k_parts,
                                                          void *stream_) {
    QMM_ENTRY_BEGIN
    void *ptr = static_scratch_of_current_device();
    w8a16_dispatch(a, w, scale, nullptr, c, m, k, n, lda, parallel_k_parts, ptr, kStaticScratchBytes, true,
                   static_cast<hipStream_t>(stream_));
    QMM_ENTRY_END
}

HIDET_API void hidet_symmetric_quant_matmul_f16_i8_bias(const void *a, const void *w, const void *scale, const void *bias,
                                                        void *c, int64_t m, int64_t k, int64_t n, int64_t lda,
                                                        int parallel_k_parts, void *workspace, int64_t workspace_bytes,
                                                        void *stream_) {
    QMM_ENTRY_BEGIN
    w8a16_dispatch(a, w, scale, bias, c, m, k, n, lda, parallel_k_parts, workspace, workspace_bytes, false,
                   static_cast<hipStream_t>(stream_));
    QMM_ENTRY_END
}

HIDET_API void hidet_symmetric_quant_matmul_f16_i8_nk(const void *a, const void *w_nk, const void *scale, void *c, int64_t m,
                                                      int64_t k, int64_t n, int64_t lda, int64_t ldw, void *workspace,
                                                      int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    w8a16_nk_dispatch(a, w_nk, scale, nullptr, c, m, k, n, lda, ldw, workspace, workspace_bytes, static_cast<hipStream_t>(stream_));
    QMM_ENTRY_END
}

HIDET_API void hidet_symmetric_quant_matmul_f16_i8_nk_bias(const void *a, const void *w_nk, const void *scale, const void *bias,
                                                           void *c, int64_t m, int64_t k, int64_t n, int64_t lda, int64_t ldw,
                                                           void *workspace, int64_t workspace_bytes, void *stream_) {
    QMM_ENTRY_BEGIN
    w8a16_nk_dispatch(a, w_nk, scale, bias, c, m, k, n, lda, ldw, workspace, workspace_bytes, static_cast<hipStream_t>(stream_));
    QMM_ENTRY_END
}
