// Host interface of the matvec kernel for several activation rows and any K (q8_gemv_rows.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace lhip {

// Activation rows of a K that one pass over the weights takes (0: not even one row's activations fit a CU's LDS).
int q8_gemv_rows_per_pass(int64_t k, bool f16);
// Whether a product that goes to matvecs ends sooner with this kernel than with one matvec (q8_gemv_device.h) per row.
bool q8_gemv_rows_pays(int64_t m, int64_t n, int64_t k, bool f16);
// Whether its passes run side by side: a wave for every row group of all of them.
bool q8_gemv_rows_one_round(int64_t m, int64_t n, int64_t k, bool f16);
// Activation rows of a pass of the launch for that product.
int q8_gemv_rows_of_pass(int64_t m, int64_t n, int64_t k, bool f16);
// y (m, n) = x (m, k) W^T for f32 (x 16-byte aligned) or f16 (8-byte) x and y, m up to 65535: bit for bit the matvec kernels' result for each row.
lhip_status q8_gemv_rows_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, bool f16, hipStream_t s);

}  // namespace lhip
