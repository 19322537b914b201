// Host interface of the tile kernel for many activation rows (q8_gemm_wide.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace lhip {

enum WdType { kWdBf16, kWdF16 };  // activations
// Results; the numbers are those of the output forms in q8_gemm.hip and q8_gemm_skinny.hip.
enum { kWdOutBf16 = 0, kWdOutF32 = 1, kWdOutSwiglu = 2, kWdOutF16 = 4 };

constexpr int64_t kWdMaxK = int64_t{1} << 22;  // offsets inside a tile (255 rows of 2 k bytes) are 32-bit

bool q8_gemm_wide_supports(int64_t k);
// y (m, n), or with slices > 1 that many f32 planes of it (out must be kWdOutF32).  ldy > 0: row pitch of y in weight
// rows, for a product that fills the leading columns of a wider one.
lhip_status q8_gemm_wide_launch(const int8_t *qs, const __half *ds, const void *x, WdType type, void *y, int m, int n, int k,
                                int out, hipStream_t s, int slices = 1, int ldy = 0);
// When a launch of that product ends, in half units of a 128x256 tile's time over all of K (1.3 us per 64 of K).
double q8_gemm_wide_ends(int64_t m, int64_t n);
// 192 or 224 where a launch over all of K takes tiles of so many rows for its last or only round, else 0.
int q8_gemm_wide_special_height(int64_t m, int64_t n);

}  // namespace lhip
