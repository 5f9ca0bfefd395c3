// Launch plan of the K-contiguous int8 kernel for 17 rows and more of small weights (skinny_w8a16_nk.hip).
#pragma once
#include "common.h"

namespace qmm {

struct SkinnyNkTallPlan {
    double us = 1e30;
    int rb = 1, cg = 1;  // 16-row blocks and 16-column groups of a workgroup
};
// Operands that skinny_w8a16_nk_supported accepts; 1e30 where the activations' rows are not 16-byte aligned.
SkinnyNkTallPlan skinny_w8a16_nk_tall_plan(const void *a, int64_t m, int64_t n, int64_t k, int64_t lda);
void skinny_w8a16_nk_tall_launch(const SkinnyNkTallPlan &plan, const void *a, const void *w, const void *scale, const void *bias, void *c, int64_t m, int64_t k, int64_t n,
                                 int64_t lda, int64_t ldw, hipStream_t stream);

}  // namespace qmm
