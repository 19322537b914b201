// Weight-streaming kernel (q8_gemm_skinny_device.h), f32 and f16 activations as three or two bf16 limbs: its forms and their launches.
#include "q8_gemm_skinny_device.h"

namespace lhip {

// m rows in all; passes of 64 rows (one: the tile height follows m).
template <typename XT, int OUT, int CW>
static lhip_status sk_launch_split_strips(const int8_t *qs, const __half *ds, const XT *x, void *y, float *part, int m, int n,
                                          int k, int splits, int passes, hipStream_t s) {
    if (splits > 1) {
        if (passes == 1 && m <= 16) return sk_launch_t<1, kSkOutPartial, XT, CW>(qs, ds, x, y, part, m, n, k, splits, 1, s);
        if (passes == 1 && m <= 32) return sk_launch_t<2, kSkOutPartial, XT, CW>(qs, ds, x, y, part, m, n, k, splits, 1, s);
        return sk_launch_t<4, kSkOutPartial, XT, CW>(qs, ds, x, y, part, m, n, k, splits, passes, s);
    }
    if (passes == 1 && m <= 16) return sk_launch_t<1, OUT, XT, CW>(qs, ds, x, y, part, m, n, k, 1, 1, s);
    if (passes == 1 && m <= 32) return sk_launch_t<2, OUT, XT, CW>(qs, ds, x, y, part, m, n, k, 1, 1, s);
    return sk_launch_t<4, OUT, XT, CW>(qs, ds, x, y, part, m, n, k, 1, passes, s);
}
template <typename XT, int OUT>
static lhip_status sk_launch_split_rows(int cw, const int8_t *qs, const __half *ds, const XT *x, void *y, float *part, int m,
                                        int n, int k, int splits, int passes, hipStream_t s) {
    switch (cw) {
        case 2: return sk_launch_split_strips<XT, OUT, 2>(qs, ds, x, y, part, m, n, k, splits, passes, s);
        case 3: return sk_launch_split_strips<XT, OUT, 3>(qs, ds, x, y, part, m, n, k, splits, passes, s);
        case 4: return sk_launch_split_strips<XT, OUT, 4>(qs, ds, x, y, part, m, n, k, splits, passes, s);
        default: return sk_launch_split_strips<XT, OUT, 8>(qs, ds, x, y, part, m, n, k, splits, passes, s);
    }
}

lhip_status sk_launch_f32(int cw, const int8_t *qs, const __half *ds, const float *x, void *y, float *part, int m, int n, int k,
                          int splits, int passes, hipStream_t s) {
    return sk_launch_split_rows<float, kSkOutF32>(cw, qs, ds, x, y, part, m, n, k, splits, passes, s);
}
lhip_status sk_launch_f16(int cw, const int8_t *qs, const __half *ds, const __half *x, void *y, float *part, int m, int n, int k,
                          int splits, int passes, hipStream_t s) {
    return sk_launch_split_rows<__half, kSkOutF16>(cw, qs, ds, x, y, part, m, n, k, splits, passes, s);
}

}  // namespace lhip
