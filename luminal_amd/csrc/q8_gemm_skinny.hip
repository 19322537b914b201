// Q8_0 weights x activations for few activation rows (short prompts, small batches; up to 128 rows per pass); bf16
// activations for any K in steps of 64, f32 and f16 ones for K in steps of 512.
//
// With so few activation rows the product is bound by streaming the weights, not by the matrix cores, and the
// 128/256-row tiles of q8_gemm.hip leave most of the chip idle.  Here a workgroup owns a strip of up to 128 weight rows
// (and, when the strips alone would not fill the chip, a slice of K) and streams it from HBM straight into
// registers in matrix-core operand order:
//
//   * eight compute waves of 16 weight rows each, or seven, four, three or two (strips of 112, 64, 48 or 32 rows) where
//     those end first: sk_plan.  The int8 codes go to the matrix cores as they are (an int8 is
//     exact in bf16); an MFMA step (v_mfma_f32_16x16x32_bf16) is one Q8_0 block, a lane supplies eight of its
//     codes, and the block's scale multiplies the f32 block sum: acc += d * sum, the arithmetic of the matvec
//     kernels (crates/luminal_cuda/src/quantized.rs:93-96).  Eight groups of 64 k per row block are in flight per
//     wave, reloaded in place as they are consumed.
//   * four more waves ("loaders") stage the activations for all the compute waves: (16*MT) x (64*G) tiles of x go
//     through their registers into one of three LDS buffers, two tiles ahead, one barrier per tile.  The compute
//     waves never wait for an activation load, so their in-order load counter only ever sees the weight stream.
//     In LDS a tile is G panels of 64 k, a row of a panel 128 bytes at pitch 160 (free of bank conflicts for the
//     16-lane x 4-group operand reads).
//   * activations are bf16 (the prefill GEMM: one plane per tile), or f32 / f16 held as three / two bf16 limbs
//     whose sum is the value exactly (the f32 / f16 matmul operators for several rows: one plane and one chained
//     MFMA per limb).  Every product is exact; the only roundings are those of the f32 additions.
//
// K slices write f32 partial tiles to a scratch array owned by the library (one per device, shared by every
// call on it) and a second kernel adds them in slice order and applies the output form, so results do not depend
// on timing.
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include <algorithm>
#include <cmath>

#include "common.h"
#include "q8_gemm_rows.h"
#include "q8_gemm_wide.h"
#include "q8_mma_device.h"

namespace lhip {

typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));
typedef float sk_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t sk_u32x4 __attribute__((ext_vector_type(4)));

enum { kSkOutBf16 = 0, kSkOutF32 = 1, kSkOutSwiglu = 2, kSkOutPartial = 3, kSkOutF16 = 4 };  // first three as in q8_gemm.hip

constexpr int kSkRows = 128;    // weight rows per workgroup of eight compute waves (CW: 16 * CW)
constexpr int kSkPitch = 160;   // bytes per activation row of a panel in LDS
constexpr int kSkStages = 3;    // LDS buffers
constexpr int kSkUnit = 512;     // K slices are whole multiples of this (eight groups of 64 k); the last may end sooner
constexpr size_t kSkScratchFloats = size_t{8} << 20;  // 32 MiB of partial sums

static __device__ __align__(256) float sk_scratch[kSkScratchFloats];

// NL = bf16 planes of an activation tile (1: bf16 activations, 2: f16, 3: f32).  64 k per panel row.
template <int MT, int NL>
struct SkShape {
    static_assert(NL >= 1 && NL <= 3 && (MT <= 4 || NL == 1), "three or two planes per tile: at most 64 activation rows");
    static constexpr int G = MT >= 4 ? 1 : (MT == 2 ? 2 : 4);  // groups per activation tile; a slice is an even number of tiles
    static constexpr int PANEL = 16 * MT * kSkPitch;
    static constexpr int PLANE = G * PANEL;
    static constexpr int STAGE = NL * PLANE;
    static constexpr int CHUNKS = 16 * MT * G * 8;             // pieces of 8 k per tile
    static constexpr int CH = CHUNKS / 256;                    // per loader thread
    static_assert(CHUNKS % 256 == 0 && 8 % G == 0, "tile split");
    static constexpr size_t LDS = static_cast<size_t>(kSkStages) * STAGE;
};

// One output form for four consecutive weight rows n .. n+3 of activation row m.
template <int OUT>
__device__ __forceinline__ void sk_store4(void *y, float *part, int split, int M, int N, int m, int n, sk_f32x4 v) {
    if constexpr (OUT == kSkOutPartial) {
        *reinterpret_cast<sk_f32x4 *>(part + (static_cast<size_t>(split) * M + m) * N + n) = v;
    } else if constexpr (OUT == kSkOutF32) {
        *reinterpret_cast<sk_f32x4 *>(static_cast<float *>(y) + static_cast<size_t>(m) * N + n) = v;
    } else if constexpr (OUT == kSkOutBf16) {
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        const bf16x4 w = {static_cast<__bf16>(v[0]), static_cast<__bf16>(v[1]), static_cast<__bf16>(v[2]),
                          static_cast<__bf16>(v[3])};
        *reinterpret_cast<bf16x4 *>(static_cast<__bf16 *>(y) + static_cast<size_t>(m) * N + n) = w;
    } else if constexpr (OUT == kSkOutF16) {
        typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
        const f16x4 w = {static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1]), static_cast<_Float16>(v[2]),
                         static_cast<_Float16>(v[3])};
        *reinterpret_cast<f16x4 *>(static_cast<_Float16 *>(y) + static_cast<size_t>(m) * N + n) = w;
    } else {  // rows are (gate, up) pairs
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 w = {static_cast<__bf16>(swiglu_value(v[0], v[1])), static_cast<__bf16>(swiglu_value(v[2], v[3]))};
        *reinterpret_cast<bf16x2 *>(static_cast<__bf16 *>(y) + static_cast<size_t>(m) * (N >> 1) + (n >> 1)) = w;
    }
}

// grid (strips of 16 * CW weight rows, K slices, passes of 16 * MT activation rows); CW compute waves of 16 weight
// rows and four loader waves.  K % 512 == 0, N % 4 == 0.
// A slice is `slice_groups` groups of 64 k (a multiple of 8); the last may be shorter (also a multiple of 8).
// RING = groups in flight per wave; a slice is a multiple of RING groups.
// XT = __bf16, __half or float: the loaders write x as NL = 1, 2 or 3 bf16 planes per tile whose sum is the value
// exactly (an f16 has 11 significant bits, which two limbs hold; an f32's 24 take three).
// CW = compute waves: 8, or as few as sk_plan finds to end first (a strip is one workgroup per K slice and CU, so narrower
// strips fill the chip with fewer slices, whose planes cost 16-30 % of a product of few rows; a workgroup's time per k
// falls by less than its rows do, see the table there).
// RAG: any K in steps of 64 that is no multiple of 512, at least 256.  The last slice then ends inside a ring: groups are
// counted up to a whole one, x is zero behind K, codes behind it are the last group's again and the scales of the last
// ring are shifted into place with zeros behind them.  (16 x 2880 x 2880 9.9 us against 9.6 for a K of 3072.)
template <int MT, int OUT, int RING, typename XT, int CW = 8, bool RAG = false>
__global__ __launch_bounds__((CW + 4) * 64) void q8_gemm_skinny_kernel(const int8_t *__restrict__ qs, const __half *__restrict__ ds,
                                                             const XT *__restrict__ x, void *__restrict__ y,
                                                             float *__restrict__ part, int M, int N, int K,
                                                             int slice_groups) {
    constexpr int NL = sizeof(XT) == 4 ? 3 : (std::is_same<XT, __bf16>::value ? 1 : 2);  // bf16 limbs of an activation
    using S = SkShape<MT, NL>;
    constexpr int G = S::G;
    static_assert(CW >= 2 && CW <= 8, "compute waves");
    extern __shared__ __attribute__((aligned(16))) unsigned char sk_lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int strip = blockIdx.x, split = blockIdx.y;
    const int g_begin = split * slice_groups;
    const int n_groups = min(slice_groups, RAG ? (((K + 63) >> 6) + 7) / 8 * 8 - g_begin : (K >> 6) - g_begin);
    const int n_tiles = n_groups / G;
    // blockIdx.z takes 16 * MT activation rows of the M in all (one launch streams the weights once per pass)
    const int m_base = static_cast<int>(blockIdx.z) * (16 * MT);
    // With few activation rows every strip starts its walk over K at a different place (a whole number of rings):
    // the strips advance at the same pace and would otherwise all ask the same memory channels for the same k at
    // the same time (measured: 39 -> 36 us for 28672 x 4096 at 16 rows).  With many rows the strips reading the
    // same activation tile at the same time is worth more (57 against 64 us at 128 rows).
    const int rot = MT <= 2 && !RAG ? (strip % (n_groups / RING)) * RING : 0;

    if (wave >= CW) {
        // ---------------- loaders: x tiles -> LDS, two tiles ahead of the compute waves
        const int lt = tid - CW * 64;
        const XT *src[S::CH];
        int dst[S::CH], k_left[S::CH];  // (k_left: RAG only)
#pragma unroll
        for (int i = 0; i < S::CH; ++i) {
            const int c = lt + i * 256;
            const int m = c / (G * 8), j = c % (G * 8);
            const int panel = j >> 3, jj = j & 7;
            src[i] = x + static_cast<size_t>(min(m_base + m, M - 1)) * K + (static_cast<size_t>(g_begin) + panel) * 64 + jj * 8;
            k_left[i] = K - (g_begin + panel) * 64 - jj * 8;
            dst[i] = panel * S::PANEL + m * kSkPitch + jj * 16;  // pieces in natural order: an MFMA step is one Q8_0 block
        }
        constexpr int XL = sizeof(XT) == 4 ? 2 : 1;  // 16-byte loads per piece of 8 k
        sk_u32x4 xr[2][S::CH][XL];
        auto load_x = [&](int slot, int t) __attribute__((always_inline)) {
            int tt = min(t, n_tiles - 1) + rot / G;  // past the end: re-read, never used
            if (tt >= n_tiles) tt -= n_tiles;
            const size_t off = static_cast<size_t>(tt) * (G * 64);
#pragma unroll
            for (int i = 0; i < S::CH; ++i) {
                const XT *from = src[i] + off;
                if constexpr (RAG) {  // a piece behind K: read from the row's first k, stored as zero
                    if (static_cast<int>(off) >= k_left[i]) from = src[i] + (k_left[i] - K);
                }
#pragma unroll
                for (int l = 0; l < XL; ++l) xr[slot][i][l] = reinterpret_cast<const sk_u32x4 *>(from)[l];
            }
        };
        auto store_x = [&](int slot, int stage, int t) __attribute__((always_inline)) {
            unsigned char *base = sk_lds + stage * S::STAGE;
#pragma unroll
            for (int i = 0; i < S::CH; ++i) {
                if constexpr (RAG) {
                    if (t * (G * 64) >= k_left[i])
#pragma unroll
                        for (int l = 0; l < XL; ++l) xr[slot][i][l] = sk_u32x4{0, 0, 0, 0};
                }
                if constexpr (NL == 1) {
                    *reinterpret_cast<sk_u32x4 *>(base + dst[i]) = xr[slot][i][0];
                } else {
                    float v[8];
                    if constexpr (sizeof(XT) == 4) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(xr[slot][i][e >> 2][e & 3]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            v[e] = __half2float(__ushort_as_half(static_cast<unsigned short>(xr[slot][i][0][e >> 1] >> (16 * (e & 1)))));
                    }
                    constexpr int NLS = NL;
                    sk_u32x4 limbs[NLS];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t l3[NLS];
                        split_limbs2<NLS>(v[2 * e], v[2 * e + 1], l3);
#pragma unroll
                        for (int l = 0; l < NLS; ++l) limbs[l][e] = l3[l];
                    }
#pragma unroll
                    for (int l = 0; l < NLS; ++l) *reinterpret_cast<sk_u32x4 *>(base + l * S::PLANE + dst[i]) = limbs[l];
                }
            }
        };
        load_x(0, 0);
        load_x(1, 1);
        store_x(0, 0, 0);
        load_x(0, 2);
        store_x(1, 1, 1);
        load_x(1, 3);
        __syncthreads();
        int stage = 2;  // buffer of tile t + 2
        for (int t = 0; t < n_tiles; t += 2) {  // two tiles per trip: no branch between them, so the counted waits
                                                // are exact (the loads of a slot are two tiles old when it is stored)
            // The fences keep the arithmetic on one slot's values (the limb split) behind the barrier before it:
            // moved up, it waits for loads that are only one tile old instead of two.
            store_x(0, stage, t + 2);  // tile t + 2 (a buffer last read for tile t - 1)
            load_x(0, t + 4);
            stage = stage == 2 ? 0 : stage + 1;
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            store_x(1, stage, t + 3);  // tile t + 3
            load_x(1, t + 5);
            stage = stage == 2 ? 0 : stage + 1;
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }

    // ---------------- compute waves
    const int r = lane & 15, g = lane >> 4;
    const int n0 = strip * (CW * 16) + wave * 16;

    {
        // The codes go to the matrix cores as they are (an int8 is exact in bf16) and the block scale is applied to
        // the f32 sum of each block, as the matvec kernels do; only an f32 / f16 x is split, into NL bf16 limbs.
        // An MFMA step is one Q8_0 block and a lane supplies eight of its codes; the x pieces lie in natural
        // order in LDS and a lane reads the one that matches its codes.  Two ways to get the codes:
        //  - WIDE (few activation rows, where the weight stream is what bounds the kernel): lane (r, g) requests the
        //    16 codes 16g .. 16g+15 of a group of two blocks (one 16-byte load: a row's 64 bytes are contiguous over
        //    its four lanes) and a swap between the wave's halves (lanes l and l + 32, i.e. g and g + 2) leaves it
        //    with eight codes of each block: codes 0-7, 16-23, 8-15, 24-31 for g = 0 .. 3;
        //  - otherwise two 8-byte loads, codes 8g .. 8g+7 of each block (from 64 rows on: measured 3-8 % faster
        //    there for f32 activations than the wide loads, 3-5 % slower for f16; one choice for both types keeps
        //    the order of additions, and so the f16 result, equal to the f32 form's).
        // Per block and column block NL chained MFMAs (x2, x1, x0 for f32; exact products, 96 f32 additions; an
        // f16's x2 is zero and has no MFMA, which leaves every sum as it is) and four fmas acc += d * sum.
        constexpr bool WIDE = MT <= 2;
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const int n_rounds = n_groups >> 2;
        const int8_t *a_ptr = qs + static_cast<size_t>(min(n0 + r, N - 1)) * K + static_cast<size_t>(g_begin) * 64 + (WIDE ? 16 : 8) * g;
        const int x_lane = r * kSkPitch + (WIDE ? (g & 1) * 32 + (g >> 1) * 16 : g * 16);  // the x piece of this lane's codes
        const __half *d_ptr[4];  // scales of the four weight rows this lane accumulates: n0 + 4g + v
#pragma unroll
        for (int v = 0; v < 4; ++v)
            d_ptr[v] = ds + static_cast<size_t>(min(n0 + 4 * g + v, N - 1)) * (K >> 5) + static_cast<size_t>(g_begin) * 2;
        sk_u32x4 a_reg[RING];
        sk_u32x4 d_reg[RING / 4][4];
        auto load_a = [&](int u, int group) __attribute__((always_inline)) {
            int gg = min(group, (RAG ? min(n_groups, ((K + 63) >> 6) - g_begin) : n_groups) - 1) + rot;
            if (gg >= n_groups) gg -= n_groups;
            if constexpr (WIDE) {
                a_reg[u] = *reinterpret_cast<const sk_u32x4 *>(a_ptr + static_cast<size_t>(gg) * 64);
            } else {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const u32x2 v = *reinterpret_cast<const u32x2 *>(a_ptr + static_cast<size_t>(gg) * 64 + 32 * b);
                    a_reg[u][2 * b] = v[0];
                    a_reg[u][2 * b + 1] = v[1];
                }
            }
        };
        auto load_d = [&](int set, int round) __attribute__((always_inline)) {
            int rr = min(round, n_rounds - 1) + rot / 4;
            if (rr >= n_rounds) rr -= n_rounds;
            if constexpr (RAG) {  // at any multiple of two bytes; eight scales of the row, its last ones where it ends sooner
                typedef sk_u32x4 sk_u32x4_2 __attribute__((aligned(2)));
                const int first = min(rr * 8, (K >> 5) - 2 * g_begin - 8);
#pragma unroll
                for (int v = 0; v < 4; ++v) d_reg[set][v] = *reinterpret_cast<const sk_u32x4_2 *>(d_ptr[v] + first);
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) d_reg[set][v] = *reinterpret_cast<const sk_u32x4 *>(d_ptr[v] + static_cast<size_t>(rr) * 8);
            }
        };
        // The scales of round rr, which load_d may have read from `shift` scales before its first: zeros behind the row.
        auto settle_d = [&](int set, int rr) __attribute__((always_inline)) {
            const int shift = 8 * rr - min(8 * rr, (K >> 5) - 2 * g_begin - 8);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const unsigned __int128 all = __builtin_bit_cast(unsigned __int128, d_reg[set][v]);
                d_reg[set][v] = __builtin_bit_cast(sk_u32x4, shift < 8 ? all >> (16 * (shift & 7)) : static_cast<unsigned __int128>(0));
            }
        };
        // same order of requests in the prologue as in the loop: a0 .. a3, d0, a4 .. a7, d1
#pragma unroll
        for (int u = 0; u < RING; ++u) {
            load_a(u, u);
            if ((u & 3) == 3) load_d(u >> 2, u >> 2);
            __builtin_amdgcn_sched_barrier(0);  // or the requests are regrouped and the loop's counted waits follow
        }
        sk_f32x4 acc[MT];
#pragma unroll
        for (int cb = 0; cb < MT; ++cb) acc[cb] = sk_f32x4{0.f, 0.f, 0.f, 0.f};

        constexpr int UNITS = 2 * MT;  // (block, column block) pairs of a group
        constexpr int kPending = NL == 1 || (NL == 3 && MT <= 2 && CW <= 4) ? 2 : 0;
        auto b_read = [&](const unsigned char *xb, int i, int limb) __attribute__((always_inline)) {
            return *reinterpret_cast<const sk_bf16x8 *>(xb + limb * S::PLANE + (i % MT) * 16 * kSkPitch + (i / MT) * 64);
        };
        const unsigned char *xb_cur = sk_lds + x_lane;
        __syncthreads();  // tiles 0 and 1 are staged
        // The x operands of a unit are requested two units ahead (into the next group's tile too, which is staged
        // by then) in four rotating register sets, three of them live at a time; the fence keeps the request where
        // it is, or the reads sink to their use and every unit waits a full LDS round trip.
        sk_bf16x8 bq[4][NL];
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            bq[0][l] = b_read(xb_cur, 0, l);
            bq[1][l] = UNITS > 1 ? b_read(xb_cur, 1 % UNITS, l) : b_read(xb_cur, 0, l);
        }
        // A unit's block sums are added kPending units after their MFMA, when they are there: with bf16 activations (one MFMA
        // per unit) a wave alone on its SIMD otherwise waits out every MFMA (64 x 512 x 1024 8.1 -> 7.0 us, 128 x 4096 x 1024
        // 12.4 -> 10.3, 16 x 14336 x 4096 16.4 -> 16.2; two units, one gives half of it).  So does the chain of three of an f32
        // for up to 32 rows in narrow strips (2-7 % of the product); elsewhere the limbs fill the pipe by themselves and
        // it costs 1-4 % (64 x 14336 x 4096 f32 37.9 -> 38.6 us).
        sk_f32x4 sum[4];
        float dv[2][2][4];  // scales of this group and of the one before it
        static_for<kPending>([&](auto ic) __attribute__((always_inline)) {
            sum[(4 - kPending + decltype(ic)::value) % 4] = sk_f32x4{0.f, 0.f, 0.f, 0.f};
        });
#pragma unroll
        for (int v = 0; v < 4; ++v) dv[1][0][v] = dv[1][1][v] = 0.f;
        auto add_unit = [&](auto uc, auto ic) __attribute__((always_inline)) {  // unit i of group u, i < 0: of the group before
            constexpr int i = decltype(ic)::value, u = decltype(uc)::value + (i < 0 ? 7 : 8), j = i < 0 ? i + UNITS : i;
            constexpr int slot = (u * UNITS + j) % 4;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[j % MT][v] = fmaf(dv[u & 1][j / MT][v], sum[slot][v], acc[j % MT][v]);
        };
        int stage = 0;
        int R = 0;
        do {  // a slice is never empty: no guard, so the requests above stay where the fences put them
            if constexpr (RAG) {  // (one body for every ring: a second for the last spills)
                if (R + RING / 4 >= n_rounds)
#pragma unroll
                    for (int set = 0; set < RING / 4; ++set) settle_d(set, R + set);
            }
            static_for<RING>([&](auto uc) __attribute__((always_inline)) {
                constexpr int u = decltype(uc)::value;
                constexpr bool tile_ends = (u + 1) % G == 0;
                const int gl = R * 4 + u;
                const int stage_next = tile_ends ? (stage == 2 ? 0 : stage + 1) : stage;
                const unsigned char *xb_next = sk_lds + stage_next * S::STAGE + ((u + 1) % G) * S::PANEL + x_lane;
                // the eight codes of each block as bf16
                asm volatile("" : "+v"(a_reg[u]));
                u32x2 a_blk[2];  // after the swap: dwords 0, 1 are codes of the group's first block, 2, 3 of its second
                if constexpr (WIDE) {
                    const auto s02 = __builtin_amdgcn_permlane32_swap(a_reg[u][0], a_reg[u][2], false, false);
                    const auto s13 = __builtin_amdgcn_permlane32_swap(a_reg[u][1], a_reg[u][3], false, false);
                    a_blk[0] = u32x2{s02[0], s13[0]};
                    a_blk[1] = u32x2{s02[1], s13[1]};
                } else {
                    a_blk[0] = u32x2{a_reg[u][0], a_reg[u][1]};
                    a_blk[1] = u32x2{a_reg[u][2], a_reg[u][3]};
                }
                sk_u32x4 a_bf[2];
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t w = a_blk[b][e >> 1];
                        const float lo = static_cast<float>(static_cast<signed char>(w >> (16 * (e & 1))));
                        const float hi = static_cast<float>(static_cast<signed char>(w >> (16 * (e & 1) + 8)));
                        a_bf[b][e] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xffff0000u);
                    }
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        dv[u & 1][b][v] = __half2float(__ushort_as_half(static_cast<unsigned short>(d_reg[u >> 2][v][u & 3] >> (16 * b))));
                load_a(u, gl + RING);
                static_for<UNITS>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    constexpr int U = u * UNITS + i;  // RING * UNITS is a multiple of four: the sets rotate statically
                    constexpr int ahead = i + 2;
#pragma unroll
                    for (int l = 0; l < NL; ++l)
                        bq[(U + 2) % 4][l] = ahead < UNITS ? b_read(xb_cur, ahead, l) : b_read(xb_next, ahead - UNITS, l);
                    __builtin_amdgcn_sched_barrier(0);
                    const sk_bf16x8 a = __builtin_bit_cast(sk_bf16x8, a_bf[i / MT]);
                    sk_f32x4 t = sk_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int l = NL - 1; l >= 0; --l)
                        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bq[U % 4][l], t, 0, 0, 0);
                    sum[U % 4] = t;
                    add_unit(uc, std::integral_constant<int, i - kPending>{});
                });
                // a set of scales is requested again once its last group has read it (requested earlier, the load
                // gets other registers and a copy at the end of the trip that waits for every load in flight)
                if constexpr ((u & 3) == 3) load_d(u >> 2, R + RING / 4 + (u >> 2));
                xb_cur = xb_next;
                if constexpr (tile_ends) {
                    stage = stage_next;
                    __syncthreads();
                }
            });
        } while ((R += RING / 4) < n_rounds);
        static_for<kPending>([&](auto ic) __attribute__((always_inline)) {
            add_unit(std::integral_constant<int, RING - 1>{}, std::integral_constant<int, UNITS - kPending + decltype(ic)::value>{});
        });
        const int n = n0 + 4 * g;
        if (n < N) {
#pragma unroll
            for (int cb = 0; cb < MT; ++cb) {
                const int m = m_base + cb * 16 + r;
                if (m < M) sk_store4<OUT>(y, part, split, M, N, m, n, acc[cb]);
            }
        }
        return;
    }

}

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
static int sk_units(int k) { return k / kSkUnit + (k % kSkUnit != 0); }
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

// `groups` workgroups of kSkWaves[cw_index] compute waves walk `per` units of K; a plan that cannot come below `limit` is not
// worked out.
static double sk_us(const SkTimes &t, int cw_index, int slices, unsigned groups, int per, int m, int n, double limit) {
    const int rows = m <= 16 ? 0 : (m <= 32 ? 1 : (m <= 64 || t.x_bytes == 4 ? 2 : 3)), strip = 16 * kSkWaves[cw_index];
    const double walk = t.walk[rows][cw_index], walks = static_cast<double>((groups + 255) / 256 * static_cast<unsigned>(per));
    const double rest = t.fixed[rows] + (slices > 1 ? t.sum + t.planes * static_cast<double>(slices) * m * n * 4e-6 : 0.0);
    if (walk == 0.0 || rest + walks * walk >= limit) return limit;
    const double stream = static_cast<double>(groups < 256 ? groups : 256) *
                          (strip * (kSkUnit + kSkUnit / 16) / t.weights[rows] + (16 << rows) * t.x_bytes * kSkUnit / t.activations);
    const double w2 = walk * walk, s2 = stream * stream;
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
    const double base_us = sk_us(t, base_index, base.splits, strips_of(base.cw) * base.splits, per_of(base.splits), m, n, 1e30);
    double best_us = margin * base_us;
    for (int i = 0; i < static_cast<int>(sizeof(kSkWaves) / sizeof(kSkWaves[0])); ++i) {
        if (k % kSkUnit != 0 && !sk_ragged_waves(kSkWaves[i])) continue;
        const unsigned strips = strips_of(kSkWaves[i]);
        for (int s = fixed_s ? fixed_s : 1; s <= (fixed_s ? fixed_s : base.splits > 1 ? units : 1); ++s) {
            // (two rounds of workgroups are enough for any strip)
            if (s > 1 && !fixed_s && (strips * s > 512 || static_cast<size_t>(s) * m * n > room)) break;
            const int per = per_of(s);
            if ((s - 1) * per >= units) continue;  // an empty slice
            const double us = sk_us(t, i, s, strips * s, per, m, n, best_us);
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
// 1.4 % of the best of all plans (the first rule alone: 17 %), and at none more than 1 % behind the first rule.
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
    return sk_us(kSkBf16, index, plan.splits, strips * plan.splits, (sk_units(k) + plan.splits - 1) / plan.splits, m, n, 1e30);
}

constexpr int kSkMaxRows = 128 * 64;  // passes are the grid's z extent

bool q8_gemm_skinny_supports(int m, int n, int k, int out, const void *y) {
    return m >= 1 && m <= kSkMaxRows && k % 64 == 0 && k >= 256 && n % 4 == 0 && aligned(y, out == kSkOutF32 ? 16 : (out == kSkOutBf16 ? 8 : 4));
}

template <typename XT>
constexpr int sk_limbs() { return sizeof(XT) == 4 ? 3 : (std::is_same<XT, __bf16>::value ? 1 : 2); }

template <int MT, int OUT, typename XT, int CW = 8, bool RAG = false>
static lhip_status sk_launch_t(const int8_t *qs, const __half *ds, const XT *x, void *y, float *part, int m, int n,
                               int k, int splits, int passes, hipStream_t s) {
    if constexpr (!RAG && sk_ragged_waves(CW) && std::is_same<XT, __bf16>::value)
        if (k % kSkUnit != 0) return sk_launch_t<MT, OUT, XT, CW, true>(qs, ds, x, y, part, m, n, k, splits, passes, s);
    auto kern = q8_gemm_skinny_kernel<MT, OUT, 8, XT, CW, RAG>;
    constexpr size_t lds_bytes = SkShape<MT, sk_limbs<XT>()>::LDS;
    static LdsOptIn opt;  // opting in to more than 64 KiB of dynamic LDS is a per-function attribute
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), lds_bytes)) return st;
    const int units = sk_units(k), per = (units + splits - 1) / splits;
    hipLaunchKernelGGL(kern,
                       dim3(static_cast<unsigned>((n + CW * 16 - 1) / (CW * 16)), static_cast<unsigned>(splits),
                            static_cast<unsigned>(passes)),
                       dim3((CW + 4) * 64), lds_bytes, s, qs, ds, x, y, part, m, n, k, per * 8);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

// bf16 activations: passes of 16 * MT rows (one plane per tile leaves room for 128-row tiles)
template <int MT, int CW>
static lhip_status sk_launch_mt(int out, const int8_t *qs, const __half *ds, const __bf16 *x, void *y, float *part, int m,
                                int n, int k, int splits, hipStream_t s) {
    const int passes = (m + 16 * MT - 1) / (16 * MT);
    if (splits > 1) return sk_launch_t<MT, kSkOutPartial, __bf16, CW>(qs, ds, x, y, part, m, n, k, splits, passes, s);
    switch (out) {
        case kSkOutBf16: return sk_launch_t<MT, kSkOutBf16, __bf16, CW>(qs, ds, x, y, part, m, n, k, 1, passes, s);
        case kSkOutF32: return sk_launch_t<MT, kSkOutF32, __bf16, CW>(qs, ds, x, y, part, m, n, k, 1, passes, s);
        default: return sk_launch_t<MT, kSkOutSwiglu, __bf16, CW>(qs, ds, x, y, part, m, n, k, 1, passes, s);
    }
}
template <int CW>
static lhip_status sk_launch_rows(int out, const int8_t *qs, const __half *ds, const __bf16 *x, void *y, float *part, int m,
                                  int n, int k, int splits, hipStream_t s) {
    if (m <= 16) return sk_launch_mt<1, CW>(out, qs, ds, x, y, part, m, n, k, splits, s);
    if (m <= 32) return sk_launch_mt<2, CW>(out, qs, ds, x, y, part, m, n, k, splits, s);
    if (m <= 64) return sk_launch_mt<4, CW>(out, qs, ds, x, y, part, m, n, k, splits, s);
    return sk_launch_mt<8, CW>(out, qs, ds, x, y, part, m, n, k, splits, s);
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
    lhip_status st;
    switch (plan.cw) {
        case 2: st = sk_launch_rows<2>(out, qs, ds, x, y, part, m, n, k, splits, s); break;
        case 3: st = sk_launch_rows<3>(out, qs, ds, x, y, part, m, n, k, splits, s); break;
        case 4: st = sk_launch_rows<4>(out, qs, ds, x, y, part, m, n, k, splits, s); break;
        case 7: st = sk_launch_rows<7>(out, qs, ds, x, y, part, m, n, k, splits, s); break;
        default: st = sk_launch_rows<8>(out, qs, ds, x, y, part, m, n, k, splits, s); break;
    }
    if (st != LHIP_OK || splits == 1) return st;
    return q8_gemm_reduce_launch(part, y, m, n, splits, out, s);
}

// ---- the f32-accurate ("split") form behind the f32 / f16 operators

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
// 16.2 -> 11.4 and 14.7 -> 9.5; as it was: 16 x 8192 x 8192 23.2 and 21.4.  Mean of 500 sizes of up to 64 rows 0.87, of 900 above
// that 0.85 (0.82 - 0.88 by type and rows), at none more than 2 % behind.
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

// How a product is run: by passes of 64 rows of the kernel above (kStream), by q8_gemm_rows.hip (kRows: `n_main` leading
// weight rows in whole rounds of workgroups, the others over `slices` K slices; n_main = 0: all of them), or by the
// tiles of q8_gemm_wide.hip (kWide).
struct RowsPlan {
    enum Kind { kStream, kRows, kWide } kind = kStream;
    int n_main = 0, slices = 1, width = 256;  // width = weight rows of a tile (of the n_main: 256)
    size_t floats = 0;  // of partial planes
};

// What q8_gemm_rows.hip takes for up to 64 rows, us: per block of K that the slowest compute unit walks, for the sum of the slices
// and its planes.  Fitted to 420 sizes (6 % of standard deviation).
static double few_rows_us(int64_t m, int64_t n, bool f16, double blocks, int slices) {
    const double sum = slices > 1 ? (f16 ? 4.1 : 3.8) + static_cast<double>(slices * m * n) * 4e-6 * 0.56 : 0.0;
    return blocks * (f16 ? 0.63 : 0.78) + sum;
}

// The plan that ends first, by what each kernel takes (us, measured): a workgroup of the streaming kernel 0.49 (f32) or
// 0.38 (f16) per block of K, one of q8_gemm_rows.hip 1.2 or 0.66, a 128x256 tile of q8_gemm_wide.hip 0.64 (f16); 256
// workgroups at a time, some microseconds per launch, and 3 plus 8 TB/s for the sum of the slices; up to 64 rows what
// few_rows_us says.  The lines this draws (streaming -> chosen, us): 14336 x 4096 f32 at 64 rows 38 -> (54), at 128 61 -> 54,
// at 256 120 -> 97, at 512 239 -> 162; f16 at 64 rows 34 -> (36), at 128 50 -> 36, at 512 188 -> 90; 4096 x 4096 f32 at 256
// rows 39 -> (41), at 300 63 -> 44.  Up to 64 rows, and for fewer than sixteen 128x256 tiles, the streaming kernel's narrower
// strips stay ahead.  Tiles of 224, 192 or 128 weight rows are taken where the plan puts them 6 % ahead: in one round, or without
// slices (45 x 2880 x 2880 f32 12 slices of 256 14.6 -> 8 of 128 12.2, 300 x 6144 x 4096 54.8 -> 52.6 at 224, 485 x 9721 x 3488 117 -> 100
// unsliced at 192, f16 387 x 1138 x 2432 25.8 -> 20.1; in two rounds of slices 138 x 9702 x 5056 72 <- 78).  A number of slices that leaves one empty is passed over; with 16 slices at most, and none behind the
// first number that leaves one empty, few weight rows or a K of 90 blocks left most compute units idle: 45 x 2880 x 2880 f32
// 6 -> 12 slices 18.1 -> 15.3 us, 45 x 1000 x 4480 18.9 -> 13.6, 300 x 1000 x 8000 37.4 -> 27.2, f16 400 x 1000 x 8992 30.4 ->
// 25.7.
static RowsPlan rows_plan(int64_t m, int n, int k, bool f16, size_t room, bool stream) {
    RowsPlan best;
    const int64_t m_tiles = (m + 127) / 128, n_tiles = (n + 255) / 256;
    if (stream && (m <= 64 || m_tiles * n_tiles < 16)) return best;
    const double nblk = k / 32, block = f16 ? 0.66 : 1.2;
    auto rounds = [](int64_t workgroups) { return static_cast<double>((workgroups + 255) / 256); };
    auto sum_us = [&](int64_t slices, int64_t cols) { return 3.0 + static_cast<double>(slices * m * cols) * 4.0 / 8e6; };
    double best_us = 1e30, early_us = 1e30, bare_us = 1e30;
    RowsPlan early;  // the best of tiles of 256 in up to 16 slices that come before a number leaving one empty
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
        const double us = 8.0 + static_cast<double>(q8_gemm_wide_ends(m, n)) * 0.32 * nblk;
        if (us < best_us) best_us = us, best.kind = RowsPlan::kWide;
    }
    early = bare = best, early_us = bare_us = best_us;
    // all columns, or those that whole rounds leave over, in K slices
    const int64_t per_round = m_tiles < 256 ? 256 / m_tiles : 1;
    const int64_t main_tiles = n_tiles / per_round * per_round;
    for (int64_t lead : {int64_t{0}, main_tiles}) {
        if (lead == n_tiles || (lead > 0 && m_tiles > 256)) continue;
        const int64_t cols = n - lead * 256, tiles = m_tiles * (n_tiles - lead);
        const double main_us = lead > 0 ? rounds(m_tiles * lead) * nblk * (m <= 64 ? (f16 ? 0.63 : 0.78) : block) + 8.0 : 0.0;
        constexpr int widths[] = {256, 224, 192, 128};
        int64_t tiles_of[4];
        for (int i = 0; i < 4; ++i) tiles_of[i] = m_tiles * ((cols + widths[i] - 1) / widths[i]);
        bool gap = false;
        for (int slices = 1; slices <= kMaxRowsSlices; ++slices) {
            if (lead > 0 && slices == 1) continue;
            const int per = q8_gemm_rows_slice_blocks(k, slices);
            gap = gap || slices > 16;
            if (static_cast<int64_t>(slices - 1) * per >= k / 32) {  // an empty slice (the next number may have none)
                if (per == 4) break;  // (the smallest: every further number leaves one empty)
                gap = true;
                continue;
            }
            const size_t floats = slices > 1 ? static_cast<size_t>(slices) * m * cols : 0;
            if (floats > room || (slices > 1 && tiles * slices > 0x7ffffff0)) break;  // (the grid's x extent)
            for (int i = 0; i < 4; ++i) {
                const int width = widths[i];
                const int64_t all = tiles_of[i] * slices;
                if (i > 0 && (lead > 0 || (slices > 1 && all > 256))) break;  // (a second round of slices pays a start and an end of its own)
                const double walk = (width + 20.0) / 276.0, blocks = rounds(all) * per;
                double us = main_us + (m <= 64 ? few_rows_us(m, cols, f16, blocks * walk, slices)
                                               : 8.0 + blocks * walk * block + (slices > 1 ? sum_us(slices, cols) : 0.0));
                RowsPlan plan;
                plan.kind = RowsPlan::kRows;
                plan.n_main = static_cast<int>(lead * 256);
                plan.slices = slices;
                plan.width = width;
                plan.floats = floats;
                if (i == 0 && !gap && us < early_us) early_us = us, early = plan;
                if (i > 0) us *= 1.06;  // only where clearly ahead
                if (us < best_us) best_us = us, best = plan;
                if (floats == 0 && us < bare_us) bare_us = us, bare = plan;
            }
        }
    }
    // A product of which the plain call keeps nothing in the library's array, so that its calls may overlap, keeps nothing there by
    // the further numbers of slices and widths either.
    return stream && early.floats == 0 && !(early.kind == RowsPlan::kStream && planes) ? bare : best;
}

// Floats of partial planes the plan for (m, n, k) uses when it has the library's own scratch array to itself: what a
// caller's workspace must hold for the same plan (and the same bits) with either activation type.
size_t q8_gemm_split_workspace_floats(int64_t m, int n, int k) {
    const bool stream = k % kSkUnit == 0 && n % 4 == 0;
    size_t most = 0;
    for (bool f16 : {false, true}) {
        const RowsPlan plan = rows_plan(m, n, k, f16, kSkScratchFloats, stream);
        if (plan.kind != RowsPlan::kStream) {
            most = std::max(most, plan.floats);
            continue;
        }
        for (int64_t m0 = 0; m0 < m; m0 += 64 * kSkMaxPasses) {
            const int mc = static_cast<int>(m - m0 < 64 * kSkMaxPasses ? m - m0 : 64 * kSkMaxPasses);
            // (at least what strips of 128 rows want, so that narrower ones without slices do not turn the answer into 0, "a matvec")
            const int splits = std::max(split_plan(mc, n, k, kSkScratchFloats).splits, split_base_slices(mc, n, k, kSkScratchFloats));
            if (splits > 1) most = std::max(most, static_cast<size_t>(splits) * mc * n);
        }
    }
    return most;
}

// y (m, N) = x (m, K) W^T for f32 or f16 activations and results, any m; x 16-byte aligned.
// `own_workspace`: partial planes go to `ws` (ws_floats floats; none: no K slices) and the library's scratch array
// is not touched, so calls may overlap in time.
lhip_status q8_gemm_split_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int64_t m, int n, int k,
                                 bool f16, hipStream_t s, bool own_workspace, float *ws, size_t ws_floats) {
    const size_t esz = f16 ? 2 : 4;
    const size_t room = own_workspace ? (ws ? std::min(ws_floats, kSkScratchFloats) : 0) : kSkScratchFloats;
    const bool stream = q8_gemm_split_supports(n, k, x, y, f16);
    RowsPlan plan = rows_plan(m, n, k, f16, kSkScratchFloats, stream);
    if (plan.floats > room) plan = rows_plan(m, n, k, f16, room, stream);
    float *scratch = own_workspace ? ws : (plan.kind == RowsPlan::kRows && plan.slices > 1 ? sk_scratch_ptr() : nullptr);
    if (plan.kind == RowsPlan::kWide) return q8_gemm_wide_launch(qs, ds, x, kWdF16, y, static_cast<int>(m), n, k, kWdOutF16, s);
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
        lhip_status st = f16 ? sk_launch_split_rows<__half, kSkOutF16>(strips.cw, qs, ds, reinterpret_cast<const __half *>(xc), yc, part,
                                                                       mc, n, k, splits, passes, s)
                             : sk_launch_split_rows<float, kSkOutF32>(strips.cw, qs, ds, reinterpret_cast<const float *>(xc), yc, part,
                                                                      mc, n, k, splits, passes, s);
        if (st != LHIP_OK) return st;
        if (splits > 1)
            if (lhip_status r = q8_gemm_reduce_launch(part, yc, mc, n, splits, f16 ? kSkOutF16 : kSkOutF32, s)) return r;
    }
    return LHIP_OK;
}

}  // namespace lhip
