// Q8_0 weights x some dozens to hundreds of activation rows (bf16 or f16) on the matrix cores: one launch whose workgroups walk all
// of K, no partial planes.
//
// The arithmetic is that of q8_gemm_wide.hip: int8 codes exact in bf16 / f16, the f32 sum of a block's products scaled by the
// block's d on the vector ALU.  That kernel's tiles of 128x256 are few for such products, so they were cut over K into f32 planes
// that a second launch adds, and where N has no whole quads they were not cut at all.
// Here the tile is small (16 MT x 32 NT) and K is dealt out inside the workgroup: four quad columns - every fourth quad of blocks,
// 128 of K - of two waves each, a wave all of the tile's rows and half of its weight rows, and the four sums meet in LDS at the end.
//   * A wave multiplies every code that it converts by up to 128 rows, without exchanging any with other waves: a lane loads 16
//     codes of each pair of blocks of its row (whole 128-byte lines of a quad), and an exchange between the wave's halves leaves it
//     with eight of each block, in an order of K that the activation reads follow.
//   * Activations come by direct loads, 64 of K a step and quad column, as whole lines of eight rows a request, permuted by the
//     requesting lane so that the operand reads meet no bank twice; the column's two waves read each piece from there.
// What bounds it: what a CU takes through its L1, 26 bytes a clock here - 10 KB per block of a 128 x 64 tile - beside the vector
// pipe (512 x 4096 x 14336: all of it 114 us; without the requests 76, without the arithmetic 86).  Activations held in registers two
// steps ahead of LDS instead (twice the bytes in flight) took the same, steps of a whole quad 0-5 % more; three stages of LDS in place of
// two up to 10 % less (up to 64 rows).  So it is the kernel for tiles that are few: up to some hundred rows, and a K whose planes would
// weigh more than its walk.  Measured, whole operator, before -> now, us: bf16 192 x 6000 x 1536 23.3 -> 11.7, 288 x 437 x 2496
// 28.9 -> 7.1, 256 x 4096 x 4096 27.0 -> 20.5, 384 x 4096 x 4096 31.7 -> 26.1, 256 x 1024 x 4096 20.3 -> 11.6, 18 x 4658 x 4288 81 -> 11.1,
// 200 x 2523 x 4672 88 -> 20.6; f16 192 x 6000 x 1536 20.5 -> 11.7, 128 x 2880 x 2880 17.8 -> 10.9, 256 x 4096 x 4096 24.7 -> 20.7.
// Geometric mean of 500 sizes of 8 to 2048 rows: bf16 1.36 times as fast, f16 1.13.
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "lds_request.h"
#include "q8_gemm_deep.h"
#include "q8_mma_device.h"

namespace lhip {

typedef uint32_t dp_u32x2 __attribute__((ext_vector_type(2)));

constexpr int kDpQuads = 4;  // quads of blocks (128 of K) that a workgroup walks side by side, two waves each

template <int MT, int NT>
struct DpShape {
    static constexpr int ST = MT <= 4 ? 3 : 2;                 // stages
    static constexpr int PAIR = MT * 16 * 128;                 // bytes of a pair's activations
    static constexpr int STAGE = kDpQuads * PAIR;              // a step: a pair of each quad column
    static constexpr int BN = 32 * NT;                         // weight rows of a workgroup
    static constexpr int EP = BN + 4;                          // floats per row of the epilogue's planes
    static constexpr int EPI = kDpQuads * MT * 16 * EP * 4;
    static constexpr int LDS = ST * STAGE > EPI ? ST * STAGE : EPI;
    static_assert(LDS <= 160 * 1024, "LDS");
};

// (qs and ds without __restrict__: the loads through them keep their place among the requests, which wait_loads counts.)
template <int MT, int NT, typename XT, int OUT>
__global__ __launch_bounds__(512) void q8_gemm_deep_kernel(const int8_t *qs, const unsigned short *ds, const XT *x, void *y, int M, int N, int K,
                                                           int m_tiles, int n_tiles) {
    using S = DpShape<MT, NT>;
    constexpr bool kF16 = std::is_same<XT, _Float16>::value;
    constexpr int ST = S::ST;
    extern __shared__ __attribute__((aligned(16))) unsigned char dp_lds[];
    int mt, nt;
    {
        const int u = xcd_item(blockIdx.x, m_tiles * n_tiles);
        if (u < 0) return;
        nt = u / m_tiles;
        mt = u - nt * m_tiles;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kq = wave >> 1, nh = wave & 1;
    const int r = lane & 15, g = lane >> 4;
    const int pairs = K >> 6, nblk = K >> 5, quads = (pairs + 1) >> 1;
    const int m0 = mt * (16 * MT), n0 = nt * S::BN + nh * (16 * NT);
    const int rounds = (quads + kDpQuads - 1) / kDpQuads;

    // ---- activations: this wave's half of its quad column's, eight rows of a pair a request, ST - 1 steps ahead of their use
    auto a_swizzle = [](int row) { return (row >> 1) & 7; };
    const unsigned char *xb = reinterpret_cast<const unsigned char *>(x) + static_cast<size_t>(m0) * K * 2;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)dp_lds));
    uint32_t a_off[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        const int row = (nh * MT + u) * 8 + (lane >> 3);
        a_off[u] = static_cast<uint32_t>(min(row, M - 1 - m0)) * static_cast<uint32_t>(K) * 2u + ((lane & 7) ^ a_swizzle(row)) * 16u;
    }
    // step t: a pair of this quad column's (past the end: the last pair again, never multiplied)
    auto request = [&](int t, int stage) __attribute__((always_inline)) {
        const int pair = min(((t >> 1) * kDpQuads + kq) * 2 + (t & 1), pairs - 1);
        const uint32_t st = lds0 + stage * S::STAGE + kq * S::PAIR + nh * (MT * 1024);
#pragma unroll
        for (int u = 0; u < MT; ++u) lds_request<16>(xb + static_cast<size_t>(pair) * 128, a_off[u], st + u * 1024);
    };

    // ---- codes and scales of a quad: lane (r, g) loads 16 codes of each pair of row r
    const int8_t *w_src[NT];
    const unsigned short *s_src[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int row = min(n0 + j * 16 + r, N - 1);
        w_src[j] = qs + static_cast<size_t>(row) * K + g * 16;
        s_src[j] = ds + static_cast<size_t>(row) * nblk;
    }
    mma_u32x4 wreg[NT][2];
    dp_u32x2 sreg[NT];
    auto load_scales = [&](int qi) __attribute__((always_inline)) {
        const int b = min((qi * kDpQuads + kq) * 4, nblk - 4);  // (an odd pair at the end: its scales are the upper two)
#pragma unroll
        for (int j = 0; j < NT; ++j) __builtin_memcpy(&sreg[j], __builtin_assume_aligned(s_src[j] + b, 4), 8);
    };
    auto load_codes = [&](int qi) __attribute__((always_inline)) {
        const int p = min((qi * kDpQuads + kq) * 2, pairs - 1);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                wreg[j][h] = *reinterpret_cast<const mma_u32x4 *>(w_src[j] + static_cast<size_t>(min(p + h, pairs - 1)) * 64);
    };

    mma_f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mma_f32x4{0.f, 0.f, 0.f, 0.f};
    const mma_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // K slots of a block: lane group g holds codes 0-7, 16-23, 8-15, 24-31 (what the exchange of load's halves leaves)
    const int piece = ((g & 1) << 1) | (g >> 1);
    const int a_lane = kq * S::PAIR + r * 128 + ((piece ^ a_swizzle(r)) * 16);  // fragment i: + 16 i rows; second block of a pair: ^ 64

    dp_u32x2 cur[NT][4], cur_s[NT];  // the quad's codes by block, its scales
    auto take = [&](int qi) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            asm volatile("" : "+v"(sreg[j]));
            const bool odd = (qi * kDpQuads + kq) * 4 > nblk - 4;
            cur_s[j] = dp_u32x2{odd ? sreg[j][1] : sreg[j][0], sreg[j][1]};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                mma_u32x4 &w = wreg[j][h];
                asm volatile("" : "+v"(w));
                const auto s02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
                const auto s13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
                cur[j][2 * h] = dp_u32x2{s02[0], s13[0]};
                cur[j][2 * h + 1] = dp_u32x2{s02[1], s13[1]};
            }
        }
    };
    mma_u32x4 bf[2][NT];
    auto convert = [&](int b, int p) __attribute__((always_inline)) {  // piece p of 4 NT of block b
        bf[b & 1][p >> 2][p & 3] = codes2<kF16>(cur[p >> 2][b][(p & 3) >> 1], p & 1);
    };
    auto scale_of = [&](int b, int j) __attribute__((always_inline)) {
        return __half2float(__ushort_as_half(static_cast<unsigned short>(cur_s[j][b >> 1] >> (16 * (b & 1)))));
    };

    // Blocks B0 and B0 + 1 of the quad, whose activations are the pair at `st`.
    auto blocks = [&](const unsigned char *st, auto b0c) __attribute__((always_inline)) {
        constexpr int B0 = decltype(b0c)::value, F = 2 * MT, AHEAD = 3, RING = 4;
        mma_u32x4 ar[RING];
        auto read_a = [&](auto fc) __attribute__((always_inline)) {
            constexpr int f = decltype(fc)::value;
            ar[f % RING] = *reinterpret_cast<const mma_u32x4 *>(st + ((a_lane ^ (f / MT * 64)) + f % MT * 16 * 128));
        };
        static_for<AHEAD>([&](auto fc) __attribute__((always_inline)) { read_a(fc); });
        float sc[2][NT];
        mma_f32x4 sum[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) sc[0][j] = scale_of(B0, j);
        static_for<F>([&](auto fc) __attribute__((always_inline)) {
            constexpr int f = decltype(fc)::value, b = f / MT, i = f % MT;
            constexpr int bp = (f - 1) / MT, ip = (f + MT - 1) % MT;
            if constexpr (f + AHEAD < F) read_a(std::integral_constant<int, f + AHEAD>{});
            mma_f32x4 s[NT];
            static_for<NT>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                __builtin_amdgcn_sched_barrier(0);
                s[j] = mma_16x16x32<kF16>(ar[f % RING], bf[(B0 + b) & 1][j], zero);
                asm volatile("" : "+v"(s[j]));
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (f > 0) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[ip][j][v] = fmaf(sc[bp][j], sum[j][v], acc[ip][j][v]);
                    asm volatile("" : "+v"(acc[ip][j]));
                }
            });
#pragma unroll
            for (int j = 0; j < NT; ++j) sum[j] = s[j];
            // the codes of the block after this one
            if constexpr (B0 + b < 3) {
                constexpr int PER = (4 * NT + MT - 1) / MT;
#pragma unroll
                for (int p = i * PER; p < i * PER + PER; ++p)
                    if (p < 4 * NT) convert(B0 + b + 1, p);
            }
            if constexpr (f == MT - 1) {
#pragma unroll
                for (int j = 0; j < NT; ++j) sc[1][j] = scale_of(B0 + 1, j);
            }
        });
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[MT - 1][j][v] = fmaf(sc[1][j], sum[j][v], acc[MT - 1][j][v]);
    };

    // The loads go out in this order: scales, requests, codes (the next quad's), then the odd step's requests.  They end in that
    // order, so a wait names the youngest that may still be under way.  (The compiler's own waits count its loads only, which the
    // requests among them can but lengthen; scales are older than the requests that the counts below stand on.)
    constexpr int CODES = 2 * NT;
    int stage = 0;
    auto next_stage = [&]() { return stage == ST - 1 ? 0 : stage + 1; };
    auto last_stage = [&]() { return stage == 0 ? ST - 1 : stage - 1; };  // the one that the step before this has read
    auto quad = [&](int qi) __attribute__((always_inline)) {
        const int left = pairs - (qi * kDpQuads + kq) * 2;  // pairs of the quad that are there
        wait_loads<(ST - 2) * MT>();
        bare_barrier();
        take(qi);
        __builtin_amdgcn_sched_barrier(0);
        load_scales(qi + 1);
        __builtin_amdgcn_sched_barrier(0);
        request(2 * qi + ST - 1, last_stage());
        __builtin_amdgcn_sched_barrier(0);
        load_codes(qi + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (left > 0) {
#pragma unroll
            for (int p = 0; p < 4 * NT; ++p) convert(0, p);
            blocks(dp_lds + stage * S::STAGE, std::integral_constant<int, 0>{});
        }
        stage = next_stage();
        __builtin_amdgcn_sched_barrier(0);
        wait_loads<(ST - 2) * MT + CODES>();
        bare_barrier();
        request(2 * qi + ST, last_stage());
        __builtin_amdgcn_sched_barrier(0);
        if (left > 1) blocks(dp_lds + stage * S::STAGE, std::integral_constant<int, 2>{});
        stage = next_stage();
        __builtin_amdgcn_sched_barrier(0);
    };
    // the same for the first quad
    load_scales(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ST == 3) request(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_codes(0);
    __builtin_amdgcn_sched_barrier(0);
    request(ST - 2, ST - 2);
    __builtin_amdgcn_sched_barrier(0);
    int qi = 0;
    do quad(qi); while (++qi < rounds);  // (at least once: behind a test the first loads would be moved past it)
    wait_loads<0>();  // no request outlives its buffer, which the epilogue now takes over
    bare_barrier();

    // ---- epilogue: the quad columns' sums through LDS, added in their order.  Element v of lane (r, g) is row 4 g + v,
    // column r of its 16 x 16 tile.
    float *ep = reinterpret_cast<float *>(dp_lds);
    constexpr int PLANE = MT * 16 * S::EP;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                ep[kq * PLANE + (i * 16 + 4 * g + v) * S::EP + nh * (16 * NT) + j * 16 + r] = acc[i][j][v];
    __syncthreads();
    using OT = std::conditional_t<OUT == kWdOutF32, float, std::conditional_t<OUT == kWdOutF16, _Float16, __bf16>>;
    constexpr int PER = OUT == kWdOutSwiglu ? 2 : 1, C = 4 / PER;  // weight rows per value of y; values a thread
    OT *yo = static_cast<OT *>(y);
    const size_t pitch = static_cast<size_t>(N / PER);
    const bool whole = (pitch * sizeof(OT)) % (C * sizeof(OT)) == 0 && (reinterpret_cast<uintptr_t>(y) & (C * sizeof(OT) - 1)) == 0;
    constexpr int QUADS = S::BN / 4, ITEMS = MT * 16 * QUADS;  // four weight rows each
#pragma unroll
    for (int t = 0; t < (ITEMS + 511) / 512; ++t) {
        const int item = t * 512 + tid;
        if (ITEMS % 512 != 0 && item >= ITEMS) break;
        const int er = item / QUADS, ec = (item % QUADS) * 4;
        const int row = m0 + er, col = nt * S::BN + ec;
        mma_f32x4 v = *reinterpret_cast<const mma_f32x4 *>(ep + er * S::EP + ec);
#pragma unroll
        for (int q = 1; q < kDpQuads; ++q) v += *reinterpret_cast<const mma_f32x4 *>(ep + q * PLANE + er * S::EP + ec);
        if (row >= M) continue;
        float o[C];
        if constexpr (PER == 2) {
            o[0] = swiglu_value(v[0], v[1]);
            o[1] = swiglu_value(v[2], v[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[e];
        }
        OT *p = yo + static_cast<size_t>(row) * pitch + col / PER;
        if (whole && col + 4 <= N) {
            typedef OT otxc __attribute__((ext_vector_type(C)));
            otxc w;
#pragma unroll
            for (int e = 0; e < C; ++e) w[e] = static_cast<OT>(o[e]);
            *reinterpret_cast<otxc *>(p) = w;
        } else {
#pragma unroll
            for (int e = 0; e < C; ++e)
                if (col + PER * e < N) p[e] = static_cast<OT>(o[e]);
        }
    }
}

template <int MT, int NT, typename XT, int OUT>
static lhip_status dp_launch_t(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, hipStream_t s) {
    using S = DpShape<MT, NT>;
    const int m_tiles = (m + 16 * MT - 1) / (16 * MT), n_tiles = (n + S::BN - 1) / S::BN;
    const int64_t total = static_cast<int64_t>(m_tiles) * n_tiles;
    if (total > 0x7ffffff0) return LHIP_ERR_INVALID_SHAPE;  // the grid's x extent
    auto kern = q8_gemm_deep_kernel<MT, NT, XT, OUT>;
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), S::LDS)) return st;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((total + 7) / 8 * 8)), dim3(512), S::LDS, s, qs,
                       reinterpret_cast<const unsigned short *>(ds), static_cast<const XT *>(x), y, m, n, k, m_tiles, n_tiles);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

template <typename XT, int OUT>
static lhip_status dp_launch(DeepPlan p, const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, hipStream_t s) {
#define LHIP_DP(MT, NT) \
    if (p.mt == MT && p.nt == NT) return dp_launch_t<MT, NT, XT, OUT>(qs, ds, x, y, m, n, k, s)
    LHIP_DP(2, 1);
    LHIP_DP(3, 1);
    LHIP_DP(4, 1);
    LHIP_DP(6, 1);
    LHIP_DP(8, 1);
    LHIP_DP(2, 2);
    LHIP_DP(3, 2);
    LHIP_DP(4, 2);
    LHIP_DP(6, 2);
    LHIP_DP(8, 2);
#undef LHIP_DP
    return LHIP_ERR_UNSUPPORTED;
}

bool q8_gemm_deep_supports(int64_t k, const void *x) { return k % 64 == 0 && k >= 128 && k <= kWdMaxK && aligned(x, 16); }

// What a launch takes, us: fixed, for every further round of 256 workgroups, and per 512 of K a price by the round and one by how
// full the chip is.  Fitted to 2800 launches of 300 sizes (m of 24 to 1200, N of 256 to 14336, K of 512 to 14336): standard
// deviation 6 to 13 %; the form that it chooses is 0.6 % behind the best one on average, 11 % at most.
struct DeepTimes {
    DeepPlan plan;
    double launch, round, walk, fill;
};
static constexpr DeepTimes kDpTimes[] = {
    {{2, 1}, 4.64, 0.15, 0.76, 0.10}, {{3, 1}, 4.71, 0.23, 0.86, 0.20}, {{4, 1}, 4.44, 1.06, 1.03, 0.40}, {{6, 1}, 4.11, 1.13, 1.44, 0.44},
    {{8, 1}, 3.85, 1.50, 1.86, 0.40}, {{2, 2}, 4.31, 0.49, 1.41, 0.03}, {{3, 2}, 4.41, 0.61, 1.58, 0.09}, {{4, 2}, 4.10, 1.94, 1.87, 0.25},
    {{6, 2}, 3.98, 2.24, 2.39, 0.31}, {{8, 2}, 4.06, 2.57, 3.01, 0.33}};

DeepPlan q8_gemm_deep_plan(int64_t m, int64_t n, int64_t k, double limit) {
    const double walks = static_cast<double>((k + 511) / 512);
    DeepPlan best;
    if (3.85 + 0.76 * walks >= limit || m > (1 << 30) || n > (1 << 30)) return best;  // (no form takes less)
    const uint32_t mu = static_cast<uint32_t>(m), nu = static_cast<uint32_t>(n);
#pragma unroll
    for (const DeepTimes &t : kDpTimes) {
        const uint32_t mr = 16 * t.plan.mt, nr = 32 * t.plan.nt;
        const int64_t groups = static_cast<int64_t>((mu + mr - 1) / mr) * ((nu + nr - 1) / nr);
        if (groups > 0x7ffffff0) continue;  // the grid's x extent
        const double rounds = static_cast<double>((groups + 255) >> 8), chips = static_cast<double>(groups) * (1.0 / 256.0);
        const double us = t.launch + (rounds - 1.0) * t.round + walks * (rounds * t.walk + chips * t.fill);
        if (us < limit) limit = us, best = t.plan;
    }
    return best;
}

lhip_status q8_gemm_deep_launch(const int8_t *qs, const __half *ds, const void *x, WdType type, void *y, int m, int n, int k,
                                int out, DeepPlan plan, hipStream_t s) {
    if (type == kWdBf16) {
        if (out == kWdOutF32) return dp_launch<__bf16, kWdOutF32>(plan, qs, ds, x, y, m, n, k, s);
        if (out == kWdOutBf16) return dp_launch<__bf16, kWdOutBf16>(plan, qs, ds, x, y, m, n, k, s);
        if (out == kWdOutSwiglu) return dp_launch<__bf16, kWdOutSwiglu>(plan, qs, ds, x, y, m, n, k, s);
    } else if (out == kWdOutF16) {
        return dp_launch<_Float16, kWdOutF16>(plan, qs, ds, x, y, m, n, k, s);
    }
    return LHIP_ERR_UNSUPPORTED;
}

}  // namespace lhip
