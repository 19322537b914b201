// Host interface of the f32 / f16 kernel for several activation rows (q8_gemm_rows.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "q8_gemm_deep.h"

namespace lhip {

// How a product is run: by passes of 64 rows of q8_gemm_skinny_device.h (kStream), by q8_gemm_rows.hip (kRows: `n_main` leading
// weight rows in whole rounds of workgroups, the others over `slices` K slices; n_main = 0: all of them), by the
// tiles of q8_gemm_wide.hip (kWide), or by q8_gemm_deep.hip (kDeep, f16 only).
struct RowsPlan {
    enum Kind { kStream, kRows, kWide, kDeep, kNone } kind = kStream;
    int n_main = 0, slices = 1, width = 256;  // width = weight rows of a tile (of the n_main: 256)
    size_t floats = 0;  // of partial planes
    DeepPlan deep;
};
// Floats of partial planes the plan of (m, n, k) uses when it has the library's own scratch array to itself: what a caller's workspace
// must hold for the same plan (and the same bits) with either activation type.  plans[0], plans[1]: those of f32 and f16.
size_t q8_gemm_split_workspace_floats(int64_t m, int n, int k, RowsPlan *plans = nullptr);
// Whether the streaming kernel takes the product; the product of any m rows by its plan (`known`: that of
// q8_gemm_split_workspace_floats, not for a shape that the streaming kernel takes where aligned).
bool q8_gemm_split_supports(int n, int k, const void *x, const void *y, bool f16);
lhip_status q8_gemm_split_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int64_t m, int n, int k, bool f16,
                                 hipStream_t s, bool own_workspace = false, float *ws = nullptr, size_t ws_floats = 0,
                                 const RowsPlan *known = nullptr);

// lhip_q8_0_matmul_plan's answers: for f32 / f16 on the matrix cores within `room` floats of planes; for bf16 (room SIZE_MAX: the plain
// call; q8_gemm.hip), of which the weight-streaming kernel's.
void q8_gemm_split_describe(int64_t m, int n, int k, bool f16, size_t room, int32_t plan[3]);
void q8_gemm_describe(int64_t m, int64_t n, int64_t k, size_t room, int32_t plan[3]);
void q8_gemm_skinny_describe(int m, int n, int k, size_t room, int32_t plan[3]);

// Blocks of K per slice (whole groups of four).
int q8_gemm_rows_slice_blocks(int64_t k, int slices);
// y (m, n) = x (m, k) W^T for f32 or f16 x and y (x 16-byte aligned), any k that is a multiple of 32, any m and n; ldy = row
// pitch of y; width = weight rows of a tile (256, 224, 192 or 128).  slices > 1: that many f32 planes of (m, n) at `part`, added in slice order; none may be empty.
lhip_status q8_gemm_rows_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, bool f16, int width,
                                int slices, float *part, int ldy, hipStream_t s);

}  // namespace lhip
