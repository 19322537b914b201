// Q8_0 matvecs of a few activation rows and of any K (the kernel: q8_gemv_rows_device.h): launch shapes and launches.
#include "q8_gemv_rows.h"
#include "q8_gemv_rows_device.h"

namespace lhip {

constexpr int kRowsWaves = 8, kRowsMax = 5;           // waves of a workgroup; activation rows of a pass
constexpr size_t kRowsLds = size_t{160} * 1024;       // of a CU

// The launch shape: weight rows and slices of 1024 of K a step, activation rows of a pass, workgroups a CU.
struct GemvRowsShape {
    int r, s, mr, bpc;
    size_t lds;
};

static int rows_slices(int64_t k) { return static_cast<int>((k + 1023) / 1024); }
static size_t lds_of(int64_t k, int s, int mr, bool f16) {
    return static_cast<size_t>(mr) * ((rows_slices(k) + s - 1) / s * s) * 1024 * (f16 ? 2 : 4);
}

// Slices a step: two where K is an even number of them from four on, so that no wave reads past K for half a step.
static int rows_step(int64_t k) { return rows_slices(k) % 2 == 0 && rows_slices(k) >= 4 ? 2 : 1; }

int q8_gemv_rows_per_pass(int64_t k, bool f16) {
    if (k > (int64_t{1} << 16)) return 0;
    const size_t rows = kRowsLds / lds_of(k, rows_step(k), 1, f16);
    return rows < kRowsMax ? static_cast<int>(rows) : kRowsMax;
}

// Two weight rows a wave for a ragged K of up to three slices (a step is short there and reads past K cost most: 2880 x 2880 f32 at three
// rows 6.3 -> 5.9 us), else one.  Two workgroups a CU where their activations fit and a wave has several row groups even so; with f32 and
// 4096 weight rows one is better, which stages half as much (4096 x 4096 at three rows 7.7 -> 7.1 us).
static GemvRowsShape rows_shape(int64_t m, int64_t n, int64_t k, bool f16) {
    GemvRowsShape p;
    p.r = k % 1024 != 0 && rows_slices(k) <= 3 ? 2 : 1;
    p.s = rows_step(k);
    const int most = q8_gemv_rows_per_pass(k, f16);
    int64_t passes = (m + most - 1) / most;
    // further passes while all of them together have a wave for each row group: 300 x 8000 at five rows, one row a pass, 5.3 us, all
    // five in one 7.1
    const int64_t groups = (n + p.r - 1) / p.r;
    while (passes < m && (passes + 1) * groups <= 256 * kRowsWaves) ++passes;
    p.mr = static_cast<int>((m + passes - 1) / passes);
    p.lds = lds_of(k, p.s, p.mr, f16);
    p.bpc = (n > 4096 || f16) && 2 * p.lds <= kRowsLds ? 2 : 1;
    return p;
}

// The staging of the activations costs half a microsecond over a matvec a row, which further activation rows earn back by what is read
// beyond the first one's weight rows or by the results there are, later for halves of a short ragged K, which the other kernel reads in
// half the time; a ragged K from 3072 on it walks without a load ahead and is behind for any size, as it is for any K beyond 12288
// (848 x 16384 f32 at two rows 11.2 -> 8.7 us, 280 x 14336 f16 at four 10.1 -> 7.2, 360 x 40960 at two 25 -> 14; at 12288 804 rows of f16 at
// two 6.9 -> 6.5, 167 of f32 at three 6.1 <- 6.5).  Drawn over 10000 random sizes of K up to 14336 and of up to 512 rows: 0.3 (f32) and 0.5 % (f16)
// behind the faster kernel on average, weights from memory, 0.4 and 0.7 % with those from the cache among them.  (Lines by (m - 1) n k and for
// every long ragged K: 1.2 to 1.4 %, and up to 30 % for small products, which matvecs a row take in, us, 24 x 256 x 2880 f16 4.4 <- 5.6, 12 x 213 x
// 4096 4.5 <- 5.2, 2 x 2240 x 4096 4.6 <- 5.5.)  A short f32 K whose weight rows fill the waves by themselves needs more further rows: 3 x 5195 x
// 416 5.1 <- 6.1, 4 x 8020 x 512 7.9 -> 6.5; 4 x 2862 x 1024 5.5 -> 4.6.
// One row: where K is long, or its weight rows fill the chip twice or do not once: 14336 x 4128 f32 19.7 -> 15.0, 644 x 13696 9.7 -> 6.7, 14168 x
// 8640 f16 30.7 -> 26.0, 1920 x 3936 f32 4.9 -> 4.5, 4000 x 4608 f32 8.2 -> 7.5, 8316 x 3904 f16 14.5 -> 9.1; the other way 2380 x 5088 f32 6.6 <- 7.2,
// 3576 x 4704 f16 6.2 <- 6.7, 7084 x 3840 f16 7.6 <- 8.5.
bool q8_gemv_rows_pays(int64_t m, int64_t n, int64_t k, bool f16) {
    if (q8_gemv_rows_per_pass(k, f16) == 0) return false;
    const bool ragged = k % 1024 != 0;
    if (m == 1) {
        const int long_k = f16 ? 4096 : 3072;
        return ragged && k > 1024 && (k > 5120 || n > (k <= long_k ? 8192 : f16 ? 4100 : 3000) || (k > long_k && n <= 256 * kRowsWaves));
    }
    const int64_t further = (m - 1) * n;
    if (f16 && ragged && k <= 3072) return static_cast<double>(further) * static_cast<double>(k < 640 ? 640 : k) > (k <= 1024 ? 18e6 : 11e6);
    if (k <= 1024) return further > (f16 ? 7000 : k >= 640 ? 8000 : n > 4096 ? 20000 : 10000);
    return (ragged && k > 3072) || k > 12288 || m * n > (ragged ? 3100 : k >= 12288 ? 1200 : 2400);
}

bool q8_gemv_rows_one_round(int64_t m, int64_t n, int64_t k, bool f16) {
    const GemvRowsShape p = rows_shape(m, n, k, f16);
    return (m + p.mr - 1) / p.mr * ((n + p.r - 1) / p.r) <= 256 * kRowsWaves;
}

int q8_gemv_rows_of_pass(int64_t m, int64_t n, int64_t k, bool f16) { return rows_shape(m, n, k, f16).mr; }

template <int R, int S, int MR, bool RAG, typename XT>
static lhip_status rows_launch(const GemvRowsShape &p, const int8_t *qs, const __half *ds, const XT *x, XT *y, int m, int n, int k,
                               hipStream_t s) {
    constexpr int W = kRowsWaves;
    int grid = ((n + R - 1) / R + W - 1) / W;
    if (grid > 256 * p.bpc) grid = 256 * p.bpc;
    const unsigned row_groups = static_cast<unsigned>((rows_slices(k) + S - 1) / S * S * RowsX<XT>::kPer);
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(q8_gemv_rows_kernel<R, S, W, MR, RAG, XT>), p.lds)) return st;
    hipLaunchKernelGGL((q8_gemv_rows_kernel<R, S, W, MR, RAG, XT>), dim3(static_cast<unsigned>(grid), static_cast<unsigned>((m + MR - 1) / MR)),
                       dim3(W * 64), p.lds, s, qs, reinterpret_cast<const unsigned short *>(ds), x, y, m, n, k, grid, 65536u / row_groups + 1);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

template <int R, int S, bool RAG, typename XT>
static lhip_status rows_launch_mr(const GemvRowsShape &p, const int8_t *qs, const __half *ds, const XT *x, XT *y, int m, int n, int k,
                                  hipStream_t s) {
    switch (p.mr) {
        case 1: return rows_launch<R, S, 1, RAG>(p, qs, ds, x, y, m, n, k, s);
        case 2: return rows_launch<R, S, 2, RAG>(p, qs, ds, x, y, m, n, k, s);
        case 3: return rows_launch<R, S, 3, RAG>(p, qs, ds, x, y, m, n, k, s);
        case 4: return rows_launch<R, S, 4, RAG>(p, qs, ds, x, y, m, n, k, s);
        default: return rows_launch<R, S, 5, RAG>(p, qs, ds, x, y, m, n, k, s);
    }
}

template <typename XT>
static lhip_status rows_launch_any(const int8_t *qs, const __half *ds, const XT *x, XT *y, int m, int n, int k, hipStream_t s) {
    const GemvRowsShape p = rows_shape(m, n, k, sizeof(XT) == 2);
    if (p.r == 2) return rows_launch_mr<2, 1, true>(p, qs, ds, x, y, m, n, k, s);
    if (p.s == 2)
        return k % 2048 != 0 ? rows_launch_mr<1, 2, true>(p, qs, ds, x, y, m, n, k, s) : rows_launch_mr<1, 2, false>(p, qs, ds, x, y, m, n, k, s);
    return k % 1024 != 0 ? rows_launch_mr<1, 1, true>(p, qs, ds, x, y, m, n, k, s) : rows_launch_mr<1, 1, false>(p, qs, ds, x, y, m, n, k, s);
}

lhip_status q8_gemv_rows_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, bool f16, hipStream_t s) {
    if (f16) return rows_launch_any(qs, ds, static_cast<const __half *>(x), static_cast<__half *>(y), m, n, k, s);
    return rows_launch_any(qs, ds, static_cast<const float *>(x), static_cast<float *>(y), m, n, k, s);
}

}  // namespace lhip
