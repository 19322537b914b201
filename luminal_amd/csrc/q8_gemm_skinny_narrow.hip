// Weight-streaming kernel (q8_gemm_skinny_device.h), bf16 activations with K in steps of 512, strips of 64, 48 and 32 weight rows: its
// forms and their launches.
#include "q8_gemm_skinny_device.h"

namespace lhip {

lhip_status sk_launch_bf16_narrow(int cw, int out, const int8_t *qs, const __half *ds, const __bf16 *x, void *y, float *part, int m, int n,
                                  int k, int splits, hipStream_t s) {
    switch (cw) {
        case 2: return sk_launch_rows<2, false>(out, qs, ds, x, y, part, m, n, k, splits, s);
        case 3: return sk_launch_rows<3, false>(out, qs, ds, x, y, part, m, n, k, splits, s);
        default: return sk_launch_rows<4, false>(out, qs, ds, x, y, part, m, n, k, splits, s);
    }
}

}  // namespace lhip
