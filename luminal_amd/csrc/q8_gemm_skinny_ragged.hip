// Weight-streaming kernel (q8_gemm_skinny_device.h), bf16 activations with any K in steps of 64 that is none of 512: its forms and
// their launches.
#include "q8_gemm_skinny_device.h"

namespace lhip {

lhip_status sk_launch_bf16_ragged(int cw, int out, const int8_t *qs, const __half *ds, const __bf16 *x, void *y, float *part, int m, int n,
                                  int k, int splits, hipStream_t s) {
    switch (cw) {
        case 2: return sk_launch_rows<2, true>(out, qs, ds, x, y, part, m, n, k, splits, s);
        case 4: return sk_launch_rows<4, true>(out, qs, ds, x, y, part, m, n, k, splits, s);
        default: return sk_launch_rows<8, true>(out, qs, ds, x, y, part, m, n, k, splits, s);
    }
}

}  // namespace lhip
