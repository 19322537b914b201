// Host interface of the f32 / f16 kernel for several activation rows (q8_gemm_rows.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace lhip {

// Blocks of K per slice (whole groups of four).
int q8_gemm_rows_slice_blocks(int64_t k, int slices);
// y (m, n) = x (m, k) W^T for f32 or f16 x and y (x 16-byte aligned), any k that is a multiple of 32, any m and n; ldy = row
// pitch of y; width = weight rows of a tile (256, 224, 192 or 128).  slices > 1: that many f32 planes of (m, n) at `part`, added in slice order; none may be empty.
lhip_status q8_gemm_rows_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, bool f16, int width,
                                int slices, float *part, int ldy, hipStream_t s);

}  // namespace lhip
