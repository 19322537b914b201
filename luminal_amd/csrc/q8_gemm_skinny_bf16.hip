// Weight-streaming kernel (q8_gemm_skinny_device.h), bf16 activations with K in steps of 512, strips of 128 and 112 weight rows: its forms
// and their launches.
#include "q8_gemm_skinny_device.h"

namespace lhip {

lhip_status sk_launch_bf16(int cw, int out, const int8_t *qs, const __half *ds, const __bf16 *x, void *y, float *part, int m, int n, int k,
                           int splits, hipStream_t s) {
    return cw == 7 ? sk_launch_rows<7, false>(out, qs, ds, x, y, part, m, n, k, splits, s)
                   : sk_launch_rows<8, false>(out, qs, ds, x, y, part, m, n, k, splits, s);
}

}  // namespace lhip
