// Launch plan of the FP8 kernel for 17 rows and more of small matrices (skinny_fp8.hip).
#pragma once
#include "common.h"

namespace qmm {

struct SkinnyFp8TallPlan {
    double us = 1e30;
    int rb = 1, cg = 1;  // 16-row blocks and 16-column groups of a workgroup
};
// K a multiple of 16 and not zero, a and b with 16-byte aligned rows; scaled: K and N multiples of 128, scale_a [K / 128, M], scale_b [N / 128, K / 128].
SkinnyFp8TallPlan skinny_fp8_tall_plan(bool scaled, int64_t m, int64_t n, int64_t k);
void skinny_fp8_tall_launch(const SkinnyFp8TallPlan &plan, bool scaled, const void *a, const void *b, void *c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
                            int out_dtype, const void *scale_a, const void *scale_b, hipStream_t stream);

}  // namespace qmm
