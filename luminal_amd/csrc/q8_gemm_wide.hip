// Q8_0 weights x many activation rows on the matrix cores:  Y[M][N] = X[M][K] . W[N][K]^T.
//
// The tile kernel behind the prompt products (bf16 activations: lhip_q8_0_matmul_bf16 and its forms; f16 activations of
// many rows: lhip_q8_0_matmul_f16).  Weights stay exact: the int8 codes go to the
// matrix cores as they are (exact in bf16 and in f16), the sum of a Q8_0 block's products is formed there in f32, and
// the block's scale multiplies that sum on the vector ALU, acc += d * sum - the arithmetic of the reference's matvec
// kernel (crates/luminal_cuda/src/quantized.rs:93-96).  Activations are bf16 or f16 as given, so every product is exact.
//
// What bounds it: the scale costs one vector fma per output element and block, 64 cycles per 32 x 32 outputs and
// block against 64 cycles of matrix steps, and a matrix step holds the vector pipe for nine cycles of its own: the
// kernel is bound by the vector pipe (a register-only loop of that mix, rate_bf16_scaled_kernel in calibrate.hip: 1287
// TFLOP/s of useful work on random data; by the counters at 2048 x 14336 x 4096 the pipe is held for 82 % of the tiles' time).
// Hence:
//   * v_mfma_f32_16x16x32: a block is ONE step (nothing is read back as an accumulator), and on random data the part
//     holds 2.2 GHz with it where the 32x32x16 form drops to 1.6-1.9;
//   * a wave owns 32 weight rows of the tile and all of its BM activation rows, so a code is converted to bf16 / f16
//     once per workgroup, in the registers of the wave that multiplies it, and the price per output falls with BM;
//   * every operand arrives in LDS by direct loads (no registers, no LDS stores): activations in rows of 64 K values,
//     codes and scales as they lie in memory.  16-byte pieces of a row are permuted by the requesting lane so that the
//     activation reads meet no bank twice (counters: 128 conflict cycles a K tile and workgroup are left, 10 % of LDS time);
//   * one barrier per K tile, in the middle of it: the operand reads run on across the tile's edge, and a tile is
//     requested kStages - 1 tiles ahead.  The requests are dealt out over the second half of the tile (all at once
//     they hold up the operand reads behind them: 256x256 tile 2.15 -> 1.98 us per 64 of K).
// Measured, us per 64 of K and tile, all CUs busy: 256x256 2.0 (1070 TFLOP/s), 128x256 1.2 (890); the kernel this one
// replaced (256x128, 32x32x16 steps, codes stored to LDS as bf16) 1.33 per 128x256 outputs.  Whole products, weights
// rotating, old -> new: 2048 x 14336 x 4096 328 -> 279 us (862 TFLOP/s), 2048 x 8192 x 4096 182 -> 146, 2000 x 28672 x
// 4096 609 -> 510, 2048 x 4096 x 4096 (one round of 128x256) 92 -> 85, 777 x 2880 x 2880 62 -> 38.
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "lds_request.h"
#include "q8_gemm_wide.h"
#include "q8_mma_device.h"

namespace lhip {

typedef uint32_t wd_u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWdBN = 256;  // weight rows per workgroup: eight waves of 32

// BM activation rows; a tile is 64 of K, two Q8_0 blocks.
template <int BM>
struct WdShape {
    static constexpr int A_ROW = 128, B_ROW = 64;            // bytes of an activation row and of a row of codes
    static constexpr int A_BYTES = (BM + 63) / 64 * 64 * A_ROW;  // in whole requests of eight waves
    static constexpr int B_WAVE = 32 * B_ROW;                // the codes of a wave's weight rows
    static constexpr int B_BYTES = 8 * B_WAVE;
    static constexpr int S_BYTES = 8 * 256;                  // one dword (two blocks' scales) per lane
    static constexpr int STAGE = A_BYTES + B_BYTES + S_BYTES;
    static constexpr int STAGES = 4 * STAGE <= 160 * 1024 ? 4 : 3;
    static constexpr int LDS = STAGES * STAGE;
    static constexpr int A_REQ = A_BYTES / (8 * 1024);       // requests per wave: activations (1 KiB each),
    static constexpr int B_REQ = B_WAVE / 1024;              // codes,
    static constexpr int REQ = A_REQ + B_REQ + 1;            // scales
    static_assert(LDS <= 160 * 1024 && A_REQ * 8 * 1024 == A_BYTES && B_REQ * 1024 == B_WAVE, "staging split");
};

// Order of the tiles.  An XCD runs its workgroups in order, 32 at a time.  The (M tile, N tile, K slice) triples are numbered with the M tiles of a group of m_group (2048 rows)
// innermost, then the slices of an N tile, then the N tiles, then the groups, and each XCD takes an equal share of
// consecutive numbers: the workgroups in flight on it share each weight tile, and the activation tiles of the group,
// out of its L2.  (Whole N tiles per XCD, the form before, leave XCDs with a tile more than others: 777 x 2880 x 2880,
// 12 N tiles over three slices, 51 against 33 us.)  False: a slot of the padded grid.
__device__ __forceinline__ bool wd_tile(int id, int m_tiles, int n_tiles, int slices, int m_group, int &mt, int &nt, int &slice) {
    const int u = xcd_item(id, m_tiles * n_tiles * slices);
    if (u < 0) return false;
    const int per_group = m_group * n_tiles * slices;
    const int group = u / per_group, rem = u - group * per_group;
    const int cur = min(m_group, m_tiles - group * m_group);
    const int ns = rem / cur;
    mt = group * m_group + (rem - ns * cur);
    nt = ns / slices;
    slice = ns - nt * slices;
    return true;
}

// One tile: rows m0 .. of x, weight rows n0 .. below n_end, K tiles kt0 .. kt0 + KT - 1.
// `y` already points at this K slice's plane; ldy = row pitch of y in weight rows.
template <int BM, typename XT, int OUT>
__device__ __forceinline__ void wd_tile_body(unsigned char *lds, const int8_t *__restrict__ qs, const __half *__restrict__ ds,
                                             const XT *__restrict__ x, void *__restrict__ y, int M, int K, int m0, int n0,
                                             int n_end, int kt0, int KT, int ldy) {
    using S = WdShape<BM>;
    constexpr bool kF16 = std::is_same<XT, _Float16>::value;
    const mma_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr int NI = BM / 16;    // 16-row fragments
    constexpr int NF = 2 * NI;     // (block, fragment) pairs of a tile
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int nblk = K >> 5;
    const int last_n = n_end - 1;

    // ---- requests.  A wave brings in 1/8 of the activation rows, and the codes and scales of its own 32 weight rows.
    // Rows past the end repeat the last one.
    auto a_swizzle = [](int row) { return (row >> 1) & 7; };
    auto b_swizzle = [](int row) { return (4 - (row >> 2)) & 3; };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)lds));
    uint32_t a_off[S::A_REQ], b_off[S::B_REQ], s_off;
#pragma unroll
    for (int q = 0; q < S::A_REQ; ++q) {  // eight rows per request
        const int row = (wave * S::A_REQ + q) * 8 + (lane >> 3);
        const int piece = (lane & 7) ^ a_swizzle(row);
        a_off[q] = static_cast<uint32_t>(min(m0 + row, M - 1) - m0) * static_cast<uint32_t>(K) * 2u + piece * 16u;
    }
    const int wn0 = n0 + wave * 32, wbase = min(wn0, last_n);
#pragma unroll
    for (int q = 0; q < S::B_REQ; ++q) {  // sixteen rows per request
        const int row = q * 16 + (lane >> 2);
        const int piece = (lane & 3) ^ b_swizzle(row);
        b_off[q] = static_cast<uint32_t>(min(wn0 + row, last_n) - wbase) * static_cast<uint32_t>(K) + piece * 16u;
    }
    s_off = static_cast<uint32_t>(min(wn0 + (lane & 31), last_n) - wbase) * static_cast<uint32_t>(nblk) * 2u;
    const unsigned char *xb = reinterpret_cast<const unsigned char *>(x) + (static_cast<size_t>(m0) * K + static_cast<size_t>(kt0) * 64) * 2;
    const int8_t *qb = qs + static_cast<size_t>(wbase) * K + static_cast<size_t>(kt0) * 64;
    const __half *db = ds + static_cast<size_t>(wbase) * nblk + static_cast<size_t>(kt0) * 2;
    auto request_piece = [&](int t, int stage, auto pc) __attribute__((always_inline)) {
        constexpr int p = decltype(pc)::value;
        static_assert(p >= 0 && p < S::REQ, "no such request");
        const int tt = min(t, KT - 1);  // past the end: the last tile again, never used
        const uint32_t st = lds0 + stage * S::STAGE;
        if constexpr (p < S::A_REQ) {
            lds_request<16>(xb + static_cast<size_t>(tt) * 128, a_off[p], st + (wave * S::A_REQ + p) * 1024);
        } else if constexpr (p < S::A_REQ + S::B_REQ) {
            constexpr int q = p - S::A_REQ;
            lds_request<16>(qb + static_cast<size_t>(tt) * 64, b_off[q], st + S::A_BYTES + wave * S::B_WAVE + q * 1024);
        } else {  // a row's two scales are one aligned dword (K / 32 is even)
            lds_request<4>(db + static_cast<size_t>(tt) * 2, s_off, st + S::A_BYTES + S::B_BYTES + wave * 256);
        }
    };
    auto request = [&](int t, int stage) __attribute__((always_inline)) {
        static_for<S::REQ>([&](auto pc) __attribute__((always_inline)) { request_piece(t, stage, pc); });
    };

    // ---- operands
    const int a_lane = r * S::A_ROW + (g ^ a_swizzle(r)) * 16;  // fragment i: + i * 16 rows; block 1: ^ 64
    const int b_lane = S::A_BYTES + wave * S::B_WAVE + r * S::B_ROW + ((g >> 1) ^ b_swizzle(r)) * 16 + (g & 1) * 8;  // n tile 1: + 16 rows; block 1: ^ 32
    const int s_lane = S::A_BYTES + S::B_BYTES + wave * 256 + r * 4;  // n tile 1: + 64
    mma_f32x4 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mma_f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int AHEAD = 3, RING = AHEAD + 1;  // activation fragments requested from LDS ahead of their use
    static_assert(NF % RING == 0, "the ring has the same phase in every tile");
    mma_u32x4 ar[RING];
    mma_u32x4 bf[2][2];   // weight operands of two successive blocks, [block parity][n tile]
    wd_u32x2 raw[2];     // codes of the block after this one
    float sc[2][2];      // scales [block parity][n tile]
    uint32_t sraw[2];    // the next tile's
    mma_f32x4 sum[2];     // block sums whose scaling is still to be issued
    auto read_raw = [&](const unsigned char *p) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) raw[j] = *reinterpret_cast<const wd_u32x2 *>(p + j * 16 * S::B_ROW);
    };
    auto read_scales = [&](const unsigned char *st) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) sraw[j] = *reinterpret_cast<const uint32_t *>(st + s_lane + j * 64);
    };
    auto half_of = [](uint32_t w, int h) { return __half2float(__ushort_as_half(static_cast<unsigned short>(w >> (16 * h)))); };
    auto set_scales = [&]() __attribute__((always_inline)) {  // from sraw
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            sc[0][j] = half_of(sraw[j], 0);
            sc[1][j] = half_of(sraw[j], 1);
        }
    };
    auto convert = [&](int b, int p) __attribute__((always_inline)) {  // piece p of 8
        bf[b][p >> 2][p & 3] = codes2<kF16>(raw[p >> 2][(p & 3) >> 1], p & 1);
    };

#pragma unroll
    for (int i = 0; i < S::STAGES - 1; ++i) request(i, i);
    wait_loads<(S::STAGES - 2) * S::REQ>();
    bare_barrier();
#pragma unroll
    for (int f = 0; f < AHEAD; ++f) ar[f] = *reinterpret_cast<const mma_u32x4 *>(lds + a_lane + f * 16 * S::A_ROW);
    read_raw(lds + b_lane);
    read_scales(lds);
    set_scales();
#pragma unroll
    for (int p = 0; p < 8; ++p) convert(0, p);

    constexpr int STEP = NI / S::REQ >= 2 ? 2 : 1;  // fragments between two requests
    static_assert(1 + (S::REQ - 1) * STEP < NI, "the requests fit the second half");
    int stage = 0;
    for (int t = 0; t < KT; ++t) {
        const int next = stage == S::STAGES - 1 ? 0 : stage + 1, last = stage == 0 ? S::STAGES - 1 : stage - 1;
        const unsigned char *st = lds + stage * S::STAGE, *st_next = lds + next * S::STAGE;
        const unsigned char *a0 = st + a_lane, *a1 = st + (a_lane ^ 64), *a2 = st_next + a_lane;
        static_for<NF>([&](auto fc) __attribute__((always_inline)) {
            constexpr int f = decltype(fc)::value, b = f / NI, i = f % NI;
            constexpr int bp = (f - 1) / NI, ip = (f + NI - 1) % NI;  // the fragment before this one (f > 0)
            if constexpr (f == 0) read_raw(st + (b_lane ^ 32));  // block 1
            if constexpr (f == NI) {
                // This wave's requests for the next tile have landed, and behind the barrier everybody's; the buffer of
                // the tile before this one is free.
                wait_loads<(S::STAGES - 3) * S::REQ>();
                bare_barrier();
                read_raw(st_next + b_lane);
                read_scales(st_next);
            }
            if constexpr (f > NI && (f - NI - 1) % STEP == 0 && (f - NI - 1) / STEP < S::REQ)
                request_piece(t + S::STAGES - 1, last, std::integral_constant<int, (f - NI - 1) / STEP>{});
            constexpr int fa = f + AHEAD;
            ar[fa % RING] = *reinterpret_cast<const mma_u32x4 *>((fa < NI ? a0 : (fa < NF ? a1 : a2)) + (fa % NI) * 16 * S::A_ROW);
            mma_f32x4 s[2];
            static_for<2>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                // The fences hold the order: left alone, the scheduler issues the matrix steps first and keeps their sums
                // alive.  The sums of the fragment before are scaled under this one's matrix steps.
                __builtin_amdgcn_sched_barrier(0);
                s[j] = mma_16x16x32<kF16>(ar[f % RING], bf[b][j], zero);
                asm volatile("" : "+v"(s[j]));
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (f > 0) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[ip][j][v] = fmaf(sc[bp][j], sum[j][v], acc[ip][j][v]);
                    asm volatile("" : "+v"(acc[ip][j]));
                }
            });
            sum[0] = s[0];
            sum[1] = s[1];
            // the codes of the block after this one
            constexpr int C0 = NI >= 16 ? 4 : 3, PER = NI >= 16 ? 1 : 2;
            if constexpr (i >= C0 && (i - C0) * PER < 8) {
#pragma unroll
                for (int p = (i - C0) * PER; p < (i - C0) * PER + PER; ++p) convert(b ^ 1, p);
            }
        });
        // the last fragment's sums, with this tile's scales
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[NI - 1][j][v] = fmaf(sc[1][j], sum[j][v], acc[NI - 1][j][v]);
        set_scales();
        stage = next;
    }
    wait_loads<0>();  // no request outlives its buffer, which the epilogue now takes over
    bare_barrier();

    // ---- epilogue.  Accumulator element v of lane (r, g) is row 4 g + v, column r of its 16 x 16 tile: two-byte stores
    // of 32-byte runs.  The wave turns 64 rows at a time round in its own part of LDS, so that the lanes of a store are
    // neighbours in y: 16 bytes each where the rows of y start on 16 bytes, else a word or one value each.  (Several stores a
    // lane, each with gaps between the lanes, measured: f32 planes 0.36 us a MB and not 0.27, 300 x 2879 x 256 21 us and not 11.)
    constexpr int EP = 36;  // floats per row of 32
    float *ep = reinterpret_cast<float *>(lds) + wave * (64 * EP);
    static_assert(8 * 64 * EP * 4 <= S::LDS, "epilogue buffer");
    using OT = std::conditional_t<OUT == kWdOutF32, float, std::conditional_t<OUT == kWdOutF16, _Float16, __bf16>>;
    constexpr int PER = OUT == kWdOutSwiglu ? 2 : 1;  // weight rows per value of y
    OT *yo = static_cast<OT *>(y);
    const size_t pitch = static_cast<size_t>(ldy / PER);
    auto starts_on = [&](size_t bytes) { return (pitch * sizeof(OT)) % bytes == 0 && (reinterpret_cast<uintptr_t>(y) & (bytes - 1)) == 0; };
    auto store_rows = [&](int i0, auto wc) __attribute__((always_inline)) {
        constexpr int W = decltype(wc)::value, LANES = 32 / W, ROWS = 64 / LANES, C = W / PER;  // weight rows and values a lane
        const int ecol = (lane % LANES) * W, col = wn0 + ecol;
#pragma unroll
        for (int q = 0; q < LANES; ++q) {
            const int er = q * ROWS + lane / LANES, row = m0 + i0 * 16 + er;
            typedef float f32xw __attribute__((ext_vector_type(W)));
            float v[W];
            if constexpr (W == 8) {
                const mma_f32x4 lo = *reinterpret_cast<const mma_f32x4 *>(ep + er * EP + ecol);
                const mma_f32x4 hi = *reinterpret_cast<const mma_f32x4 *>(ep + er * EP + ecol + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = lo[e], v[4 + e] = hi[e];
            } else if constexpr (W == 1) {
                v[0] = ep[er * EP + ecol];
            } else {
                const f32xw w = *reinterpret_cast<const f32xw *>(ep + er * EP + ecol);
#pragma unroll
                for (int e = 0; e < W; ++e) v[e] = w[e];
            }
            if constexpr (PER == 2) {
#pragma unroll
                for (int e = 0; e < C; ++e) v[e] = swiglu_value(v[2 * e], v[2 * e + 1]);
            }
            if (row >= M || (NI % 4 != 0 && i0 * 16 + er >= BM)) continue;
            OT *p = yo + static_cast<size_t>(row) * pitch + col / PER;
            if (C > 1 && col + W <= n_end) {
                typedef OT otxc __attribute__((ext_vector_type(C)));
                otxc w;
#pragma unroll
                for (int e = 0; e < C; ++e) w[e] = static_cast<OT>(v[e]);
                *reinterpret_cast<otxc *>(p) = w;
            } else {
#pragma unroll
                for (int e = 0; e < C; ++e)
                    if (col + PER * e < n_end) p[e] = static_cast<OT>(v[e]);
            }
        }
    };
    constexpr int WIDE = OUT == kWdOutF32 ? 4 : 8, LESS = PER == 2 ? 4 : (OUT == kWdOutF32 ? 1 : 2);
    const bool wide = starts_on(WIDE / PER * sizeof(OT)), less = starts_on(LESS / PER * sizeof(OT));
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 4) {
#pragma unroll
        for (int i = 0; i < (NI - i0 < 4 ? NI - i0 : 4); ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) ep[(i * 16 + 4 * g + v) * EP + j * 16 + r] = acc[i0 + i][j][v];
        if (wide) store_rows(i0, std::integral_constant<int, WIDE>{});
        else if (LESS > 1 && less) store_rows(i0, std::integral_constant<int, LESS>{});
        else store_rows(i0, std::integral_constant<int, PER>{});
    }
}

// Weight rows below n_big in tiles of 256x256 (the first big_blocks workgroups), the others in tiles of 128, 192 or 224 rows (`small`) x 256
// (wd_cut chooses both).  With `slices` > 1 every slice of kt_slice K tiles goes into an f32 plane of (M, N) of its
// own (tiles of 128x256).
template <typename XT, int OUT>
__global__ __launch_bounds__(512) void q8_gemm_wide_kernel(const int8_t *__restrict__ qs, const __half *__restrict__ ds,
                                                           const XT *__restrict__ x, void *__restrict__ y, int M, int N, int K,
                                                           int n_big, int big_blocks, int small, int slices, int kt_slice, int ldy) {
    extern __shared__ __attribute__((aligned(16))) unsigned char wd_lds[];
    const int kt_all = K / 64;
    int mt, nt, slice;
    if (static_cast<int>(blockIdx.x) < big_blocks) {
        const int m_tiles = (M + 255) / 256;
        if (!wd_tile(blockIdx.x, m_tiles, n_big / kWdBN, 1, min(m_tiles, 8), mt, nt, slice)) return;
        wd_tile_body<256, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 256, nt * kWdBN, n_big, 0, kt_all, ldy);
        return;
    }
    const int m_tiles = (M + small - 1) / small;
    if (!wd_tile(static_cast<int>(blockIdx.x) - big_blocks, m_tiles, (N - n_big + kWdBN - 1) / kWdBN, slices, min(m_tiles, 2048 / small), mt, nt, slice))
        return;
    const int n0 = n_big + nt * kWdBN;
    if (small == 192) {
        wd_tile_body<192, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 192, n0, N, 0, kt_all, ldy);
    } else if (small == 224) {
        wd_tile_body<224, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 224, n0, N, 0, kt_all, ldy);
    } else {
        const int kt0 = slice * kt_slice;
        if (slices > 1) y = static_cast<float *>(y) + static_cast<size_t>(slice) * M * N;
        wd_tile_body<128, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 128, n0, N, kt0, min(kt_slice, kt_all - kt0), ldy);
    }
}

// How many weight rows go to 256x256 tiles, and the height of the tiles for the others.  A tile takes the same time whatever its
// neighbours do, one of 256 / 224 / 192 rows 1.5 / 1.37 / 1.18 times one of 128 (one round of each at K = 4096: 125, 116, 100 and 86
// us), and the launch ends with its slowest CU, so what is taken is the list of big tiles followed by smaller ones that ends first when
// dealt to 256 CUs in order: big tiles up to the last or last but one whole round of them, all of them, or none.  Tiles of 192 and 224
// rows are for a last (or only) round that 128-row tiles overfill and 256-row tiles leave CUs out of; they have to be 5 % ahead (at 3 % a
// second round of 224 rows at 2048 x 14336 x 4096 gave nothing).
// Measured, us, 256 and 128 rows -> with them: 1500 x 6144 x 4096 (144 tiles of 256 or 288 of 128) 126 -> 102 by 192 of 192 rows, 2000 x 6144
// x 4096 127 -> 120 by 216 of 224 rows, 700 x 14336 x 4096 126 -> 107, 800 x 10000 x 2880 90 -> 74, 1700 x 14336 x 4096 262 -> 224.
struct WdCut {
    int n_big = 0, small = 128;
    double end = 0.0;  // in half units of a 128x256 tile's time
};
static WdCut wd_cut(int64_t m, int64_t n) {
    const int64_t mt256 = (m + 255) / 256, n_tiles = n / kWdBN, n_all = (n + kWdBN - 1) / kWdBN;  // whole tiles, all of them
    const int64_t rounds = mt256 * n_tiles / 256;
    const int64_t cuts[4] = {0, n_tiles, rounds * 256 / mt256, (rounds - 1) * 256 / mt256};
    constexpr double kBig = 3.0;
    constexpr struct {
        int rows;
        double time, margin;
    } heights[3] = {{128, 2.0, 1.0}, {192, 2.35, 1.05}, {224, 2.74, 1.05}};
    WdCut best;
    best.end = 1e300;
#pragma unroll
    for (const auto &h : heights) {
        const int64_t mt = (m + h.rows - 1) / h.rows;
        for (int i = 0; i < 4; ++i) {
            const int64_t c = cuts[i];
            if ((i > 0 && c <= 0) || (h.rows != 128 && c == n_all)) continue;
            const int64_t big = mt256 * c, small = mt * (n_all - c);
            const int64_t busy = big % 256, free = 256 - busy;  // CUs free from t0 on, and from t0 + kBig on
            const double t0 = static_cast<double>(big / 256) * kBig;
            double end = busy ? kBig : 0.0;
            if (small > 0) {
                // by whole tiles on the CUs that are free first, or on the others; from about their share of rounds on
                auto done = [&](double t) {
                    const int64_t f = static_cast<int64_t>(t / h.time + 1e-6), g = t > kBig ? static_cast<int64_t>((t - kBig) / h.time + 1e-6) : 0;
                    return free * f + busy * g;
                };
                int64_t f = small / 256 > 0 ? small / 256 : 1;
                while (done(static_cast<double>(f) * h.time) < small) ++f;
                double t = static_cast<double>(f) * h.time;
                if (busy)
                    for (int64_t g = f; g >= 1; --g) {
                        const double u = kBig + static_cast<double>(g) * h.time;
                        if (u < t && done(u) >= small) t = u;
                        if (u < t - 2.0 * h.time - kBig) break;
                    }
                if (t > end) end = t;
            }
            end += t0;
            if (end * h.margin < best.end) best.n_big = static_cast<int>(c) * kWdBN, best.small = h.rows, best.end = end;
        }
    }
    return best;
}

double q8_gemm_wide_ends(int64_t m, int64_t n) { return wd_cut(m, n).end; }

int q8_gemm_wide_special_height(int64_t m, int64_t n) {
    const WdCut cut = wd_cut(m, n);
    return cut.small != 128 ? cut.small : 0;
}

template <typename XT, int OUT>
static lhip_status wd_launch_t(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, int slices,
                               int ldy, hipStream_t s) {
    const WdCut cut = slices == 1 ? wd_cut(m, n) : WdCut{};
    auto blocks = [](int64_t m_tiles, int64_t n_tiles) { return (m_tiles * n_tiles + 7) / 8 * 8; };  // whole eights, see wd_tile
    const int64_t big = blocks((m + 255) / 256, cut.n_big / kWdBN);
    const int64_t small = blocks((m + cut.small - 1) / cut.small, static_cast<int64_t>((n - cut.n_big + kWdBN - 1) / kWdBN) * slices);
    if (big + small > 0x7fffffff) return LHIP_ERR_INVALID_SHAPE;  // the grid's x extent
    auto kern = q8_gemm_wide_kernel<XT, OUT>;
    constexpr int lds_small = WdShape<128>::LDS, lds_most = WdShape<256>::LDS;
    static_assert(lds_most >= lds_small && lds_most >= WdShape<192>::LDS && lds_most >= WdShape<224>::LDS, "the opt-in covers all heights");
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), lds_most)) return st;
    const int kt = k / 64, kt_slice = (kt + slices - 1) / slices;
    if (slices < 1 || (slices - 1) * kt_slice >= kt) return LHIP_ERR_UNSUPPORTED;  // an empty slice
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(big + small)), dim3(512),
                       static_cast<unsigned>(cut.n_big > 0 || cut.small != 128 ? lds_most : lds_small), s, qs, ds, static_cast<const XT *>(x), y, m, n, k,
                       cut.n_big, static_cast<int>(big), cut.small, slices, kt_slice, ldy > 0 ? ldy : n);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

bool q8_gemm_wide_supports(int64_t k) { return k % 64 == 0 && k <= kWdMaxK; }

lhip_status q8_gemm_wide_launch(const int8_t *qs, const __half *ds, const void *x, WdType type, void *y, int m, int n, int k,
                                int out, hipStream_t s, int slices, int ldy) {
#define LHIP_WD(XT, OUT) return wd_launch_t<XT, OUT>(qs, ds, x, y, m, n, k, slices, ldy, s)
    if (type == kWdBf16) {
        if (out == kWdOutF32) LHIP_WD(__bf16, kWdOutF32);
        if (out == kWdOutBf16) LHIP_WD(__bf16, kWdOutBf16);
        if (out == kWdOutSwiglu) LHIP_WD(__bf16, kWdOutSwiglu);
    } else if (out == kWdOutF16) {
        LHIP_WD(_Float16, kWdOutF16);
    }
#undef LHIP_WD
    return LHIP_ERR_UNSUPPORTED;
}

}  // namespace lhip
