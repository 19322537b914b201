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
// What its estimates, of weights in the memory-side cache, are short of from memory against a kernel that is estimated from there: some
// 0.1 us per MB, which shows for a large or long matrix; no more beyond some 160 MB, which no cache holds for the estimates either (f16 at 8 rows
// 27324 x 10368 82.8 there, 96.3 as slices, at 6 rows 16272 x 30336 141 and 155; 39 x 5210 x 12800 the other way 41.5 and 33.0, 25 x 16486 x 20992 146 and
// 127).
static inline double q8_gemm_deep_from_memory_us(int64_t n, int64_t k) {
    const double large = static_cast<double>(n) * static_cast<double>(k) * 1e-6 - (k < 8192 ? 16.0 : 0.0);
    return 0.12 * (large < 0.0 ? 0.0 : large < 160.0 ? large : 160.0);
}
lhip_status q8_gemm_deep_launch(const int8_t *qs, const __half *ds, const void *x, WdType type, void *y, int m, int n, int k,
                                int out, DeepPlan plan, hipStream_t s);

}  // namespace lhip
