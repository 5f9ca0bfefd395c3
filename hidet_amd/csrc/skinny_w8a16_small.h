// Launch plan of the int8 kernel for small row-major weights (skinny_w8a16_small.hip).
#pragma once
#include "common.h"

namespace qmm {

struct SkinnySmallPlan {
    double us = 1e30;
    int rb = 1, cb = 2;  // 16-row blocks of a workgroup, columns of a lane
};
// What the kernel takes: K and the row stride of a even, a aligned to 4 bytes, N of 4 at least, offsets of 31 bits.
bool skinny_w8a16_small_supported(const void *a, int64_t n, int64_t k, int64_t lda);
// 1e30 where the kernel does not take the operands or is not for their size.
SkinnySmallPlan skinny_w8a16_small_plan(const void *a, int64_t m, int64_t n, int64_t k, int64_t lda);
void skinny_w8a16_small_launch(const SkinnySmallPlan &plan, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                               int64_t lda, hipStream_t stream);

}  // namespace qmm
