// Host interface of the kernel whose workgroups walk all of K (q8_gemm_deep.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "q8_gemm_wide.h"

namespace lhip {

// 16 mt activation rows x 32 nt weight rows a workgroup.
struct DeepPlan {
    int mt = 0, nt = 0;  // 0: not by this kernel
};
bool q8_gemm_deep_supports(int64_t k, const void *x);
// The form that ends first for a product of K >= 128 if it takes less than `limit` us (else mt = 0).
DeepPlan q8_gemm_deep_plan(int64_t m, int64_t n, int64_t k, double limit);
lhip_status q8_gemm_deep_launch(const int8_t *qs, const __half *ds, const void *x, WdType type, void *y, int m, int n, int k,
                                int out, DeepPlan plan, hipStream_t s);

}  // namespace lhip
