// The weight-streaming kernel's host side (the kernel: q8_gemm_skinny_device.h): the sum of its K slices, the strips and slices of a
// product, and which kernel an f32 or f16 product of several rows takes.
#include <algorithm>
#include <cmath>

#include "q8_gemm_rows.h"
#include "q8_gemm_skinny_device.h"
#include "q8_gemm_wide.h"

namespace lhip {

constexpr size_t kSkScratchFloats = size_t{8} << 20;  // 32 MiB of partial sums

static __device__ __align__(256) float sk_scratch[kSkScratchFloats];

// Sum of the K slices in slice order, then the output form.  One thread per four weight rows.  ldy = row pitch of y
// in weight rows (N, or more when the planes are the trailing columns of a wider output).  A small result is a chain of
// loads: six in flight instead of one, 60 values over 19 slices 3.9 to 6.2 us (by where the planes lie) -> 2.3.
template <int OUT>
__global__ __launch_bounds__(256) void q8_gemm_skinny_reduce_kernel(const float *__restrict__ part, void *__restrict__ y,
                                                                    int M, int N, int splits, int ldy) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    const size_t quads = static_cast<size_t>(M) * (N >> 2);
    if (i >= quads) return;
    const size_t plane = static_cast<size_t>(M) * N;
    sk_f32x4 v = *reinterpret_cast<const sk_f32x4 *>(part + 4 * i);
    int s = 1;
    auto add = [&](auto count) __attribute__((always_inline)) {  // the next planes: their loads first
        constexpr int C = decltype(count)::value;
        sk_f32x4 p[C];
#pragma unroll
        for (int u = 0; u < C; ++u) p[u] = *reinterpret_cast<const sk_f32x4 *>(part + (s + u) * plane + 4 * i);
#pragma unroll
        for (int u = 0; u < C; ++u) v += p[u];
        s += C;
    };
    while (s + 6 <= splits) add(std::integral_constant<int, 6>{});
    if (s + 3 <= splits) add(std::integral_constant<int, 3>{});
    while (s < splits) add(std::integral_constant<int, 1>{});
    const int m = static_cast<int>(i / (N >> 2)), n = static_cast<int>(i % (N >> 2)) * 4;
    sk_store4<OUT>(y, nullptr, 0, M, ldy, m, n, v);
}

// Scratch address per device (a __device__ array has one copy, at its own address, on every device).
static float *sk_scratch_ptr() {
    static float *ptrs[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    float *p = __atomic_load_n(&ptrs[dev], __ATOMIC_ACQUIRE);
    if (!p) {
        if (hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(sk_scratch)) != hipSuccess) return nullptr;
        __atomic_store_n(&ptrs[dev], p, __ATOMIC_RELEASE);
    }
    return p;
}

float *q8_gemm_scratch(size_t *floats) {
    *floats = kSkScratchFloats;
    return sk_scratch_ptr();
}

// Adds `slices` f32 planes of (m, n) in order and writes the output form (as the GEMM epilogues: bf16, f32, f16, SwiGLU).
lhip_status q8_gemm_reduce_launch(const float *part, void *y, int m, int n, int slices, int out, hipStream_t s, int ldy = 0) {
    if (ldy <= 0) ldy = n;
    const size_t quads = static_cast<size_t>(m) * (n >> 2);
    const dim3 grid(static_cast<unsigned>((quads + 255) / 256));
    switch (out) {
        case kSkOutBf16: hipLaunchKernelGGL(q8_gemm_skinny_reduce_kernel<kSkOutBf16>, grid, dim3(256), 0, s, part, y, m, n, slices, ldy); break;
        case kSkOutF32: hipLaunchKernelGGL(q8_gemm_skinny_reduce_kernel<kSkOutF32>, grid, dim3(256), 0, s, part, y, m, n, slices, ldy); break;
        case kSkOutF16: hipLaunchKernelGGL(q8_gemm_skinny_reduce_kernel<kSkOutF16>, grid, dim3(256), 0, s, part, y, m, n, slices, ldy); break;
        default: hipLaunchKernelGGL(q8_gemm_skinny_reduce_kernel<kSkOutSwiglu>, grid, dim3(256), 0, s, part, y, m, n, slices, ldy); break;
    }
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

// K slices for a product: enough workgroups for the 256 CUs, slices of whole 512-k units, partial sums within the
// scratch array.
static int sk_splits_for(int strips, int m, int n, int k, size_t room) {
    const int units = sk_units(k), passes = (m + 127) / 128;
    int s = 256 / (strips * passes);
    if (s < 1) s = 1;
    if (s > units) s = units;
    while (s > 1 && static_cast<size_t>(s) * m * n > room) --s;
    const int per = (units + s - 1) / s;
    return (units + per - 1) / per;
}

// Compute waves per workgroup (strips of 16 rows each) for `splits` K slices (0: the slices are chosen with them).
struct SkPlan {
    int cw, splits;
    double of_base = 1.0;  // its time over that of strips of 128 (112) rows in the slices that fill the chip, by sk_us
};
constexpr int kSkWaves[] = {8, 7, 4, 3, 2};
constexpr bool sk_ragged_waves(int cw) { return cw % 2 == 0; }  // those built for a K that is no multiple of 512

// What the kernel takes for one pass of activation rows, us.  A workgroup walks 512 of K in the time of its table (the
// vector instructions of its waves: conversions, and four fmas per block and 16 rows) or in the time that the weights and
// activations of all of them take from memory and L2, whichever is longer (joined by a fourth power); a CU runs them one
// after the other; the sum of the slices is a launch and its planes.
struct SkTimes {
    double walk[4][5];                // by activation rows (16, 32, 64, 128) and kSkWaves (0: not built)
    double weights[4], activations;   // bytes per us
    double fixed[4], sum, planes;     // us, us, us per MB
    int x_bytes;
};
// bf16: fitted to 2800 measurements, the numbers of slices around those that fill the chip for 240 sizes (m of 16 to 128, N
// of 512 to 28672, K of 1024 to 14336).
static constexpr SkTimes kSkBf16 = {{{3.11, 2.60, 1.33, 1.10, 0.98}, {3.34, 2.96, 1.68, 1.42, 1.23},
                                     {5.24, 4.61, 2.69, 2.18, 1.99}, {5.96, 5.44, 3.62, 3.29, 3.10}},
                                    {6.2e6, 7.0e6, 5.8e6, 7.0e6}, 20e6, {3.2, 3.35, 3.65, 4.45}, 2.0, 0.52, 2};
// f32, and f16 too (so that both take the same plan, and an f16 result is the f32 form's rounded once; its own fit would
// gain 0.5 %): 1400 measurements for 120 sizes (m of 16 to 64).
static constexpr SkTimes kSkF32 = {{{3.15, 0.0, 1.64, 1.46, 1.34}, {4.12, 0.0, 2.67, 2.52, 2.37}, {6.58, 0.0, 4.57, 4.41, 4.15}, {}},
                                   {5.44e6, 5.59e6, 7.0e6, 7.0e6}, 20e6, {3.5, 3.6, 4.2, 0.0}, 1.7, 0.97, 4};

// One strip's part of that: what a workgroup's 512 of K take by its table and, per workgroup, from memory, and what does not depend
// on K.
struct SkStrip {
    double walk, stream, fixed;
    SkStrip(const SkTimes &t, int cw_index, int m) {
        const int rows = m <= 16 ? 0 : (m <= 32 ? 1 : (m <= 64 || t.x_bytes == 4 ? 2 : 3));
        walk = t.walk[rows][cw_index];
        stream = 16 * kSkWaves[cw_index] * (kSkUnit + kSkUnit / 16) / t.weights[rows] + (16 << rows) * t.x_bytes * kSkUnit / t.activations;
        fixed = t.fixed[rows];
    }
};
// `groups` workgroups of the strip walk `per` units of K; a plan that cannot come below `limit` is not worked out.
static double sk_us(const SkTimes &t, const SkStrip &strip, int slices, unsigned groups, int per, int m, int n, double limit) {
    const double walks = static_cast<double>((groups + 255) / 256 * static_cast<unsigned>(per));
    const double rest = strip.fixed + (slices > 1 ? t.sum + t.planes * static_cast<double>(slices) * m * n * 4e-6 : 0.0);
    if (strip.walk == 0.0 || rest + walks * strip.walk >= limit) return limit;
    const double stream = static_cast<double>(groups < 256 ? groups : 256) * strip.stream;
    const double w2 = strip.walk * strip.walk, s2 = stream * stream;
    return rest + walks * sqrt(sqrt(w2 * w2 + s2 * s2));
}

// `base`, or the strip and number of slices (fixed_s: that one) that sk_us puts below `margin` of it.  Where `base` has one
// slice it stays one: plain calls of such a product keep nothing in the library's array and may overlap.  (Three slices would be
// up to 25 % ahead, 13 % on average, at 1 % of sizes: 48 x 19588 x 14336 in f32, 64 x 18304 x 8192 in bf16.)
static SkPlan sk_faster_plan(const SkTimes &t, SkPlan base, double margin, int m, int n, int k, size_t room, int fixed_s, int passes = 1) {
    const int units = sk_units(k);
    auto strips_of = [n, passes](int cw) { return static_cast<unsigned>((n + 16 * cw - 1) / (16 * cw) * passes); };
    auto per_of = [units](int s) { return static_cast<int>(static_cast<unsigned>(units + s - 1) / static_cast<unsigned>(s)); };
    SkPlan best = base;
    const int base_index = base.cw == 8 ? 0 : 1;
    const double base_us = sk_us(t, SkStrip(t, base_index, m), base.splits, strips_of(base.cw) * base.splits, per_of(base.splits), m, n, 1e30);
    double best_us = margin * base_us;
    // The numbers of slices, none of which leaves one empty: each is the smallest for its length of slice.  K is sliced within one round
    // of 256 workgroups: another pays a start and an end of its own, which the tables do not hold (us, in one round / two: 3 x 5460 x 5632
    // bf16 15.2 / 18.0, 33 x 2728 x 11776 f32 29.0 / 31.7, 5 x 9320 x 7168 25.7 / 27.8).
    struct {
        int slices, per;
    } cuts[256];
    int n_cuts = 0;
    if (fixed_s) {
        if ((fixed_s - 1) * per_of(fixed_s) < units) cuts[n_cuts++] = {fixed_s, per_of(fixed_s)};
    } else {
        const unsigned most = base.splits == 1 ? 1 : 256 / strips_of(kSkWaves[0]);  // (the widest strips are the fewest)
        for (int s = 1, per = units;; s = per_of(per - 1), per = per_of(s)) {
            cuts[n_cuts++] = {s, per};
            if (per == 1 || static_cast<unsigned>(per_of(per - 1)) > most) break;
        }
    }
    for (int i = 0; i < static_cast<int>(sizeof(kSkWaves) / sizeof(kSkWaves[0])); ++i) {
        if (k % kSkUnit != 0 && !sk_ragged_waves(kSkWaves[i])) continue;
        const SkStrip strip(t, i, m);
        const unsigned strips = strips_of(kSkWaves[i]);
        for (int c = 0; c < n_cuts; ++c) {
            const int s = cuts[c].slices, per = cuts[c].per;
            if (s > 1 && !fixed_s && (strips * s > 256 || static_cast<size_t>(s) * m * n > room)) break;
            const double us = sk_us(t, strip, s, strips * s, per, m, n, best_us);
            if (us < best_us) best_us = us, best = SkPlan{kSkWaves[i], s, us / base_us};
        }
    }
    return best;
}

// A workgroup's time goes with the weights it streams (rows x its share of K) and the launch takes as many rounds of
// 256 workgroups as it has workgroups: eight waves, or seven if they make that product smaller, with the K slices that
// fill the chip.  That is right for many rows; one pass of up to 128 takes any other strip and number of slices that
// sk_us puts 6 % below (its own spread).  m x N x K, us: 16 x 14336 x 4096 7 waves, 2 slices 18.7 -> 4 waves, none 16.4;
// 16 x 4096 x 4096 8 waves, 8 slices 10.5 -> 4 waves, 4 slices 9.1; 64 x 4096 x 4096 18.1 -> 13.5; 128 x 4096 x 4096 21.4 -> 18.2;
// 16 x 4096 x 1024 8.4 -> 5.0; as it was: 32 x 10240 x 8192 29.3, 64 x 8192 x 14336 47.7.  Over the 240 sizes it is within
// 1.4 % of the best of all plans (the first rule alone: 17 %); mean of 1158 others 0.78 of the first rule's time.
static SkPlan sk_plan(int m, int n, int k, size_t room, int splits = 0) {
    const int units = sk_units(k), passes = (m + 127) / 128;
    SkPlan best{8, 1};
    long best_cost = -1;
    for (int cw = 8; cw >= (k % kSkUnit == 0 ? 7 : 8); --cw) {
        const int strips = (n + cw * 16 - 1) / (cw * 16);
        int s = splits > 0 ? (splits > units ? units : splits) : sk_splits_for(strips, m, n, k, room);
        const int per = (units + s - 1) / s;
        s = (units + per - 1) / per;  // no empty slice
        const long rounds = (static_cast<long>(strips) * s * passes + 255) / 256;
        const long cost = rounds * cw * per;
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = SkPlan{cw, s};
        }
    }
    return passes > 1 ? best : sk_faster_plan(kSkBf16, best, 0.94, m, n, k, room, splits > 0 ? best.splits : 0);
}

// The plan for `room` floats of partial planes: the one the library's own array allows wherever it fits (so that a
// caller's workspace of the recommended size gets the plain call's plan and bits), else the best within `room`.
static SkPlan sk_plan_within(int m, int n, int k, size_t room, int splits = 0) {
    const SkPlan plan = sk_plan(m, n, k, kSkScratchFloats, splits);
    if (plan.splits == 1 || static_cast<size_t>(plan.splits) * m * n <= room) return plan;
    return sk_plan(m, n, k, room, splits);
}

int q8_gemm_skinny_splits(int m, int n, int k, size_t room) { return sk_plan_within(m, n, k, room).splits; }

// What the plan takes, us (one pass: up to 128 rows).
double q8_gemm_skinny_us(int m, int n, int k, size_t room) {
    const SkPlan plan = sk_plan_within(m, n, k, room);
    int index = 0;
    while (kSkWaves[index] != plan.cw) ++index;
    const unsigned strips = static_cast<unsigned>((n + 16 * plan.cw - 1) / (16 * plan.cw));
    return sk_us(kSkBf16, SkStrip(kSkBf16, index, m), plan.splits, strips * plan.splits, (sk_units(k) + plan.splits - 1) / plan.splits, m, n, 1e30);
}

void q8_gemm_skinny_describe(int m, int n, int k, size_t room, int32_t plan[3]) {
    const SkPlan p = sk_plan_within(m, n, k, room);
    plan[0] = 1, plan[1] = 16 * p.cw, plan[2] = p.splits;
}

constexpr int kSkMaxRows = 128 * 64;  // passes are the grid's z extent

bool q8_gemm_skinny_supports(int m, int n, int k, int out, const void *y) {
    return m >= 1 && m <= kSkMaxRows && k % 64 == 0 && k >= 256 && n % 4 == 0 && aligned(y, out == kSkOutF32 ? 16 : (out == kSkOutBf16 ? 8 : 4));
}

// `splits` = 0: chosen here.  The caller has checked q8_gemm_skinny_supports.
// `own_workspace`: partial planes go to `ws` (ws_floats floats; none: no K slices) and the library's scratch array is
// not touched.
lhip_status q8_gemm_skinny_launch(const int8_t *qs, const __half *ds, const void *x_bf16, void *y, int m, int n, int k,
                                  int out, int splits, hipStream_t s, bool own_workspace, float *ws, size_t ws_floats) {
    const size_t room = own_workspace ? (ws ? std::min(ws_floats, kSkScratchFloats) : 0) : kSkScratchFloats;
    const SkPlan plan = sk_plan_within(m, n, k, room, splits);
    splits = plan.splits;
    float *part = nullptr;
    if (splits > 1) {
        if (static_cast<size_t>(splits) * m * n > room) return LHIP_ERR_UNSUPPORTED;
        part = own_workspace ? ws : sk_scratch_ptr();
        if (!part) return LHIP_ERR_HIP;
    }
    const __bf16 *x = static_cast<const __bf16 *>(x_bf16);
    auto launch = k % kSkUnit != 0 ? sk_launch_bf16_ragged : (plan.cw <= 4 ? sk_launch_bf16_narrow : sk_launch_bf16);
    const lhip_status st = launch(plan.cw, out, qs, ds, x, y, part, m, n, k, splits, s);
    if (st != LHIP_OK || splits == 1) return st;
    return q8_gemm_reduce_launch(part, y, m, n, splits, out, s);
}

// ---- the f32-accurate ("split") form behind the f32 / f16 operators

bool q8_gemm_split_supports(int n, int k, const void *x, const void *y, bool f16) {
    return k % kSkUnit == 0 && n % 4 == 0 && aligned(x, 16) && aligned(y, f16 ? 8 : 16);
}

// Passes of 64 rows of the kernel above, each streaming the weights once, as blockIdx.z of one launch; K is sliced only
// while strips x passes leave the chip unfilled.  At most kSkMaxPasses passes per launch (the grid's z extent).
constexpr int64_t kSkMaxPasses = 1024;

// K slices of one chunk of mc rows in strips of 128 weight rows: as many as fill the chip, within `room` floats of partial
// planes.
static int split_base_slices(int mc, int n, int k, size_t room) {
    const int units = k / kSkUnit, strips = (n + kSkRows - 1) / kSkRows, passes = (mc + 63) / 64;
    int splits = 256 / (strips * passes);
    if (splits < 1) splits = 1;
    if (splits > units) splits = units;
    while (splits > 1 && static_cast<size_t>(splits) * mc * n > room) --splits;
    const int per = (units + splits - 1) / splits;
    return (units + per - 1) / per;  // no empty slice
}
// The plan of a chunk: those, or up to 1024 rows any other strip and number of slices that sk_us puts 3 % below.  m x N x K, f32
// and f16, us: 16 x 4096 x 1024 9.2 -> 5.9 and 8.9 -> 5.8, 32 x 4096 x 4096 13.9 -> 12.7 and 12.8 -> 11.6, 64 x 2048 x 4096 17.4 -> 13.8
// and 16.2 -> 12.6, 16 x 14336 x 4096 21.2 -> 19.4 and 19.7 -> 17.6, 256 x 512 x 4096 17.3 -> 13.6 and 15.8 -> 12.4, 1000 x 256 x 1024
// 16.2 -> 11.4 and 14.7 -> 9.5; as it was: 16 x 8192 x 8192 23.2 and 21.4.  Mean of 2242 sizes of up to 64 rows 0.85, of 826
// above that 0.83, at none more than 3 % behind.
static SkPlan split_plan_for(int mc, int n, int k, size_t room) {
    const int passes = (mc + 63) / 64;
    const SkPlan base{8, split_base_slices(mc, n, k, room)};
    return passes > 16 ? base : sk_faster_plan(kSkF32, base, 0.97, mc, n, k, room, 0, passes);
}
// The library array's plan wherever it fits, as sk_plan_within.
static SkPlan split_plan(int mc, int n, int k, size_t room) {
    const SkPlan plan = split_plan_for(mc, n, k, kSkScratchFloats);
    if (plan.splits == 1 || static_cast<size_t>(plan.splits) * mc * n <= room) return plan;
    return split_plan_for(mc, n, k, room);
}

// ---- the choice of the kernel for the f32 / f16 operators

constexpr int kMaxRowsSlices = 40;

// What q8_gemm_rows.hip takes, us: a launch, a start and an end for every further round of 256 workgroups, a price per block of K that a
// workgroup walks (some of it for its 128 activation rows, some by its weight rows, some as the launch fills the chip), and for K
// slices the launch of their sum and its planes (N in steps of four: 16 bytes a load; else four).  Fitted to 10200 launches of 4300
// sizes; standard deviation 5 and 6 % (f32 and f16) up to 64 activation rows, of which most compute waves have none, 7 and 8 %
// above.
struct RowsTimes {
    double launch, round, sum, planes, planes_odd;  // us, us, us, us per MB
    double block, block_rows, block_fill;           // us per block; per block and 256 weight rows; per block at a full chip
};
static constexpr RowsTimes kRowsTimes[2][2] = {{{3.6, 2.75, 2.85, 0.51, 0.79, 0.12, 0.535, 0.105}, {5.7, 5.4, 2.0, 0.38, 0.725, 0.23, 0.71, 0.03}},
                                               {{3.5, 2.25, 2.75, 0.455, 0.75, 0.035, 0.455, 0.14}, {5.0, 4.1, 2.9, 0.36, 0.73, 0.08, 0.45, 0.075}}};
static double rows_us(const RowsTimes &t, int64_t workgroups, int width, int per) {  // (without the sum)
    const double rounds = static_cast<double>((workgroups + 255) >> 8), fill = workgroups < 256 ? static_cast<double>(workgroups) * (1.0 / 256.0) : 1.0;
    return t.launch + (rounds - 1.0) * t.round + rounds * per * (t.block + t.block_rows * (width * (1.0 / 256.0)) + t.block_fill * fill);
}
static double rows_sum_us(const RowsTimes &t, int slices, int64_t m, int64_t cols) {
    return slices > 1 ? t.sum + static_cast<double>(slices * m * cols) * 4e-6 * (cols % 4 == 0 ? t.planes : t.planes_odd) : 0.0;
}

// The plan that ends first, by what each kernel takes (us, measured): a workgroup of the streaming kernel 0.49 (f32) or
// 0.38 (f16) per block of K, 256 workgroups at a time, a 128x256 tile of q8_gemm_wide.hip 0.64 (f16), some microseconds per
// launch, 3 plus 8 TB/s for the sum of the slices, and q8_gemm_rows.hip what rows_us says.  The lines this draws (streaming ->
// chosen, us): 14336 x 4096 f32 at 64 rows (40), at 128 61 -> 53, at 256 117 -> 85, at 512 235 -> 147; f16 at 128 rows 50 -> 39, at 256 95 ->
// 57, at 512 186 -> 82; 4096 x 4096 f32 at 128 rows 25.4 -> 24.7, at 256 39 -> 36, at 300 57 -> 42, f16 at 256 32 -> 26.  Up to 64 rows, and
// for fewer than sixteen 128x256 tiles, the streaming kernel's narrower strips stay ahead.
// Tiles of 256 weight rows, or of 224, 192 or 128 in one round or without slices (us, 45 x 2880 x 2880 f32 12 slices of 256 14.6 -> 8 of 128
// 12.2, 300 x 6144 x 4096 55.6 -> 54.1 at 224, 485 x 9721 x 3488 118 -> 103 unsliced at 192, f16 387 x 1138 x 2432 26.1 -> 20.0; in two rounds of
// slices 138 x 9702 x 5056 72 <- 78).  Up to 40 slices, none of them empty (45 x 2880 x 2880 f32 6 -> 12 slices 18.1 -> 15.3 us, 45 x 1000 x
// 4480 7 -> 18 19.3 -> 12.0, 300 x 1000 x 8000 37 -> 29, f16 400 x 1000 x 8992 30.6 -> 25.0).  Without the price of a
// further round few rows of a wide matrix went to many: 3 x 12081 x 4736 f32 in 37 slices and seven rounds 49 us, in 5 and one 30; f16 3 x
// 22140 x 2400 in 19 and seven 43, in 2 of 192 26.
static RowsPlan rows_plan(int64_t m, int n, int k, bool f16, size_t room, bool stream) {
    RowsPlan best;
    const int64_t m_tiles = (m + 127) / 128, n_tiles = (n + 255) / 256;
    if (stream && (m <= 64 || m_tiles * n_tiles < 16)) return best;
    const RowsTimes &times = kRowsTimes[f16][m > 64];
    const double nblk = k / 32;
    auto rounds = [](int64_t workgroups) { return static_cast<double>((workgroups + 255) / 256); };
    auto sum_us = [&](int64_t slices, int64_t cols) { return 3.0 + static_cast<double>(slices * m * cols) * 4.0 / 8e6; };
    double best_us = 1e30, early_us = 1e30, bare_us = 1e30;
    RowsPlan early;  // the plan by which a plain call keeps planes or none (see the end)
    RowsPlan bare;   // the best that has no planes
    bool planes = false;
    if (stream) {  // (0.49 and 0.38 us are those of strips of 128 rows)
        const int mc = static_cast<int>(m < 64 * kSkMaxPasses ? m : 64 * kSkMaxPasses);
        const int splits = split_base_slices(mc, n, k, room);
        best_us = 6.0 + rounds(((n + kSkRows - 1) / kSkRows) * ((m + 63) / 64) * splits) * (nblk / splits) * (f16 ? 0.38 : 0.49) +
                  (splits > 1 ? sum_us(splits, n) : 0.0);
        planes = splits > 1;
        if (mc == m) best_us *= split_plan(mc, n, k, room).of_base;
    }
    if (f16 && q8_gemm_wide_supports(k)) {
        const double us = 8.0 + q8_gemm_wide_ends(m, n) * 0.32 * nblk;
        if (us < best_us) best_us = us, best.kind = RowsPlan::kWide;
    }
    early = bare = best, early_us = bare_us = best_us;
    // all columns, or those that whole rounds leave over, in K slices
    const int64_t per_round = m_tiles < 256 ? 256 / m_tiles : 1;
    const int64_t main_tiles = n_tiles / per_round * per_round;
    for (int part = 0; part < 2; ++part) {
        const int64_t lead = part == 0 ? 0 : main_tiles;
        if (part == 1 && (lead == 0 || lead == n_tiles || m_tiles > 256)) break;
        const int64_t cols = n - lead * 256, tiles = m_tiles * (n_tiles - lead);
        const double main_us = lead > 0 ? rows_us(times, m_tiles * lead, 256, k / 32) : 0.0;
        const double first_main_us = lead > 0 ? rounds(m_tiles * lead) * nblk * (f16 ? 0.66 : 1.2) + 8.0 : 0.0;
        constexpr int widths[] = {256, 224, 192, 128};
        int64_t tiles_of[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) tiles_of[i] = m_tiles * ((cols + widths[i] - 1) / widths[i]);
        bool gap = false;
        for (int slices = 1, per = q8_gemm_rows_slice_blocks(k, 1);;) {
            if (lead == 0 || slices > 1) {
                const size_t floats = slices > 1 ? static_cast<size_t>(slices) * m * cols : 0;
                if (floats > room || (slices > 1 && tiles * slices > 0x7ffffff0)) break;  // (the grid's x extent)
                const RowsPlan plan{RowsPlan::kRows, static_cast<int>(lead * 256), slices, 256, floats};
                const double others_us = main_us + rows_sum_us(times, slices, m, cols);
                for (int i = 0; i < 4; ++i) {
                    const int width = widths[i];
                    const int64_t all = tiles_of[i] * slices;
                    if (i > 0 && (lead > 0 || (slices > 1 && all > 256))) break;
                    double us = others_us + rows_us(times, all, width, per);
                    // (what the estimate is short of on average: the gap between two launches; narrow tiles that walk all of K in step)
                    if (lead > 0 || (width < 256 && slices == 1)) us *= 1.05;
                    if (us < best_us) best_us = us, best = plan, best.width = width;
                    if (floats == 0 && us < bare_us) bare_us = us, bare = plan, bare.width = width;
                }
                if (!gap && stream) {
                    const double first_us = first_main_us + 8.0 + rounds(tiles * slices) * per * (f16 ? 0.66 : 1.2) + (slices > 1 ? sum_us(slices, cols) : 0.0);
                    if (first_us < early_us) early_us = first_us, early = plan;
                }
            }
            if (per == 4) break;
            const int next = (k / 32 + per - 5) / (per - 4);  // the next number whose slices are shorter: those between leave one empty
            if (next > kMaxRowsSlices) break;
            gap = gap || next > slices + 1 || next > 16;
            slices = next;
            per = q8_gemm_rows_slice_blocks(k, slices);
        }
    }
    // A product of which the plain call kept nothing in the library's array, so that its calls may overlap, when these plans had tiles
    // of 256 in up to 16 slices, none of them behind a number that leaves one empty, at 1.2 (f32) or 0.66 us per block (`early`), keeps
    // nothing there now.
    if (stream && early.floats == 0 && !(early.kind == RowsPlan::kStream && planes)) best = bare, best_us = bare_us;
    // The kernel whose workgroups walk all of K, for f16 (three limbs an f32 value are staged for too few weight rows there): from one
    // round of its quads of blocks on, and where the streaming kernel takes the K, from three of that kernel's steps on or above 128
    // rows (up to 64, where its f16 results are those of f32 rounded, this rule is not reached).  A tenth ahead, the spread of the
    // estimates.  Measured, us, what the rules above choose -> that kernel: 45 x 2880 x 2880 11.8 -> 8.3, 128 x 2880 x 2880 17.8 -> 10.9,
    // 256 x 6000 x 1536 22.6 -> 14.1, 256 x 4096 x 4096 24.7 -> 20.7, 80 x 4096 x 4096 17.6 -> 12.6, 96 x 8148 x 2048
    // 18.8 -> 11.3; the other way 256 x 4096 x 14336 58 <- 75, 512 x 14336 x 4096
    // 84 <- 130, 186 x 9184 x 3072 30.5 <- 32.4.
    // Against K slices it is further what it loses from memory.
    // Measured, us, weights from memory, slices and that kernel: 6 x 8369 x 6144 24.4 and 29.1, 11 x 5048 x 11904 25.9 and 35.6, 32 x 5204 x 13888 35.2
    // and 42.2; the other way 251 x 848 x 5184 16.4 and 12.9.
    const double from_memory = best.kind == RowsPlan::kRows && best.slices > 1 ? q8_gemm_deep_from_memory_us(n, k) : 0.0;
    if (f16 && k >= 512 && (!stream || k >= 1536 || m > 128) && q8_gemm_deep_supports(k, nullptr)) {
        const DeepPlan deep = q8_gemm_deep_plan(m, n, k, (best_us - from_memory) / 1.1);
        if (deep.mt) {
            best = RowsPlan{RowsPlan::kDeep, 0, 1, 0, best.floats};  // (it needs no planes; callers' sizes stay what they were)
            best.deep = deep;
        }
    }
    return best;
}

size_t q8_gemm_split_workspace_floats(int64_t m, int n, int k, RowsPlan *plans) {
    const bool stream = k % kSkUnit == 0 && n % 4 == 0;
    size_t most = 0;
    bool streams = false;
    for (bool f16 : {false, true}) {
        const RowsPlan plan = rows_plan(m, n, k, f16, kSkScratchFloats, stream);
        if (plan.kind == RowsPlan::kStream)
            streams = true;
        else
            most = std::max(most, plan.floats);
        if (plans) plans[f16] = plan;
    }
    for (int64_t m0 = 0; streams && m0 < m; m0 += 64 * kSkMaxPasses) {
        const int mc = static_cast<int>(m - m0 < 64 * kSkMaxPasses ? m - m0 : 64 * kSkMaxPasses);
        // (at least what strips of 128 rows want, so that narrower ones without slices do not turn the answer into 0, "a matvec")
        const int splits = std::max(split_plan(mc, n, k, kSkScratchFloats).splits, split_base_slices(mc, n, k, kSkScratchFloats));
        if (splits > 1) most = std::max(most, static_cast<size_t>(splits) * mc * n);
    }
    return most;
}

void q8_gemm_split_describe(int64_t m, int n, int k, bool f16, size_t room, int32_t plan[3]) {
    room = std::min(room, kSkScratchFloats);
    const bool stream = k % kSkUnit == 0 && n % 4 == 0;
    RowsPlan p = rows_plan(m, n, k, f16, kSkScratchFloats, stream);
    if (p.floats > room) p = rows_plan(m, n, k, f16, room, stream);
    if (p.kind == RowsPlan::kStream) {
        const SkPlan strips = split_plan(static_cast<int>(m < 64 * kSkMaxPasses ? m : 64 * kSkMaxPasses), n, k, room);
        plan[0] = 1, plan[1] = 16 * strips.cw, plan[2] = strips.splits;
    } else if (p.kind == RowsPlan::kRows) {
        plan[0] = 2, plan[1] = p.width, plan[2] = p.n_main ? 0 : p.slices;
    } else if (p.kind == RowsPlan::kDeep) {
        plan[0] = 4, plan[1] = 32 * p.deep.nt, plan[2] = 1;
    } else {
        plan[0] = 3, plan[1] = q8_gemm_wide_special_height(m, n), plan[2] = 1;
    }
}

// y (m, N) = x (m, K) W^T for f32 or f16 activations and results, any m; x 16-byte aligned.
// `own_workspace`: partial planes go to `ws` (ws_floats floats; none: no K slices) and the library's scratch array
// is not touched, so calls may overlap in time.
lhip_status q8_gemm_split_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int64_t m, int n, int k,
                                 bool f16, hipStream_t s, bool own_workspace, float *ws, size_t ws_floats, const RowsPlan *known) {
    const size_t esz = f16 ? 2 : 4;
    const size_t room = own_workspace ? (ws ? std::min(ws_floats, kSkScratchFloats) : 0) : kSkScratchFloats;
    const bool stream = q8_gemm_split_supports(n, k, x, y, f16);
    RowsPlan plan = known ? *known : rows_plan(m, n, k, f16, kSkScratchFloats, stream);
    if (plan.floats > room) plan = rows_plan(m, n, k, f16, room, stream);
    float *scratch = own_workspace ? ws : (plan.kind == RowsPlan::kRows && plan.slices > 1 ? sk_scratch_ptr() : nullptr);
    if (plan.kind == RowsPlan::kWide) return q8_gemm_wide_launch(qs, ds, x, kWdF16, y, static_cast<int>(m), n, k, kWdOutF16, s);
    if (plan.kind == RowsPlan::kDeep)
        return q8_gemm_deep_launch(qs, ds, x, kWdF16, y, static_cast<int>(m), n, k, kWdOutF16, plan.deep, s);
    if (plan.kind == RowsPlan::kRows) {
        if (plan.slices > 1 && !scratch) return LHIP_ERR_HIP;
        const int mi = static_cast<int>(m), tail = n - plan.n_main;
        if (plan.n_main > 0)
            if (lhip_status st = q8_gemm_rows_launch(qs, ds, x, y, mi, plan.n_main, k, f16, 256, 1, nullptr, n, s)) return st;
        return q8_gemm_rows_launch(qs + static_cast<size_t>(plan.n_main) * k, ds + static_cast<size_t>(plan.n_main) * (k / 32), x,
                                   static_cast<unsigned char *>(y) + static_cast<size_t>(plan.n_main) * esz, mi, tail, k, f16,
                                   plan.width, plan.slices, scratch, n, s);
    }
    for (int64_t m0 = 0; m0 < m; m0 += 64 * kSkMaxPasses) {
        const int mc = static_cast<int>(m - m0 < 64 * kSkMaxPasses ? m - m0 : 64 * kSkMaxPasses);
        const int passes = (mc + 63) / 64;
        const SkPlan strips = split_plan(mc, n, k, room);
        const int splits = strips.splits;
        float *part = nullptr;
        if (splits > 1) {
            part = own_workspace ? ws : sk_scratch_ptr();
            if (!part) return LHIP_ERR_HIP;
        }
        const auto *xc = static_cast<const unsigned char *>(x) + static_cast<size_t>(m0) * k * esz;
        auto *yc = static_cast<unsigned char *>(y) + static_cast<size_t>(m0) * n * esz;
        const lhip_status st =
            f16 ? sk_launch_f16(strips.cw, qs, ds, reinterpret_cast<const __half *>(xc), yc, part, mc, n, k, splits, passes, s)
                : sk_launch_f32(strips.cw, qs, ds, reinterpret_cast<const float *>(xc), yc, part, mc, n, k, splits, passes, s);
        if (st != LHIP_OK) return st;
        if (splits > 1)
            if (lhip_status r = q8_gemm_reduce_launch(part, yc, mc, n, splits, f16 ? kSkOutF16 : kSkOutF32, s)) return r;
    }
    return LHIP_OK;
}

}  // namespace lhip
