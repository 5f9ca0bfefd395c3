// Launch plan of the int4 kernel for small weights (skinny_w4a16_small.hip).
#pragma once
#include "common.h"

namespace qmm {

struct SkinnyW4SmallPlan {
    double us = 1e30;
    int rb = 1, cb = 2, waves = 8;  // 16-row blocks of a workgroup, columns of a lane, waves that cut K
};
// What the kernel takes: K a multiple of 128, groups of 64, N of 8, a and the scales aligned to 4 bytes, offsets of 31 bits.
bool skinny_w4a16_small_supported(const void *a, const void *scales, int64_t n, int64_t k, int64_t lda, int group);
// 1e30 where the kernel does not take the operands or is not for their size.
SkinnyW4SmallPlan skinny_w4a16_small_plan(const void *a, const void *scales, int64_t m, int64_t n, int64_t k, int64_t lda, int group);
void skinny_w4a16_small_launch(const SkinnyW4SmallPlan &plan, const void *a, const void *w, const void *scales, const void *bias, void *c, int64_t m, int64_t k, int64_t n, int64_t lda,
                               int group, int dtype, hipStream_t stream);

}  // namespace qmm
