// Q8_0 weights x many activation rows on the matrix cores:  Y[M][N] = X[M][K] . W[N][K]^T.
//
// The tile kernel behind the prompt products (bf16 activations: lhip_q8_0_matmul_bf16 and its forms; f16 activations of
// many rows: lhip_q8_0_matmul_f16).  Weights stay exact: the int8 codes go to the
// matrix cores as they are (exact in bf16 and in f16), the sum of a Q8_0 block's products is formed there in f32, and
// the block's scale multiplies that sum on the vector ALU, acc += d * sum - the arithmetic of the reference's matvec
// kernel (crates/luminal_cuda/src/quantized.rs:93-96).  Activations are bf16 or f16 as given, so every product is exact.
//
// What bounds it: the scale costs one vector fma per output element and block, 64 cycles per 32 x 32 outputs and
// block against 64 cycles of matrix steps, and a matrix step holds the vector pipe for about ten cycles of its own: the
// kernel is bound by the vector pipe (a register-only loop of that mix: 1330 TFLOP/s of useful work on random data).
// Hence:
//   * v_mfma_f32_16x16x32: a block is ONE step (nothing is read back as an accumulator), and on random data the part
//     holds 2.2 GHz with it where the 32x32x16 form drops to 1.6-1.9;
//   * a wave owns 32 weight rows of the tile and all of its BM activation rows, so a code is converted to bf16 / f16
//     once per workgroup, in the registers of the wave that multiplies it, and the price per output falls with BM;
//   * every operand arrives in LDS by direct loads (no registers, no LDS stores): activations in rows of 64 K values,
//     codes and scales as they lie in memory.  16-byte pieces of a row are permuted by the requesting lane so that the
//     operand reads meet no bank twice;
//   * one barrier per K tile, in the middle of it: the operand reads run on across the tile's edge, and a tile is
//     requested kStages - 1 tiles ahead.  The requests are dealt out over the second half of the tile (all at once
//     they hold up the operand reads behind them: 256x256 tile 2.15 -> 1.98 us per 64 of K).
// Measured, us per 64 of K and tile, all CUs busy: 256x256 2.0 (1070 TFLOP/s), 128x256 1.2 (890); the kernel this one
// replaced (256x128, 32x32x16 steps, codes stored to LDS as bf16) 1.33 per 128x256 outputs.  Whole products, weights
// rotating, old -> new: 2048 x 14336 x 4096 337 -> 273 us (880 TFLOP/s), 2048 x 8192 x 4096 182 -> 146, 2000 x 28672 x
// 4096 609 -> 510, 2048 x 4096 x 4096 (one round of 128x256) 92 -> 85, 777 x 2880 x 2880 62 -> 38.
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "q8_gemm_wide.h"

namespace lhip {

typedef __bf16 wd_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 wd_f16x8 __attribute__((ext_vector_type(8)));
typedef float wd_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t wd_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t wd_u32x2 __attribute__((ext_vector_type(2)));

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>), expanded at compile time (register arrays indexed
// at run time land in scratch memory).
template <class F, int... Is>
__device__ __forceinline__ void wd_static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void wd_static_for(F &&f) {
    wd_static_for_impl(static_cast<F &&>(f), std::make_integer_sequence<int, N>{});
}

constexpr int kWdBN = 256;  // weight rows per workgroup: eight waves of 32

// BM activation rows; a tile is 64 of K, two Q8_0 blocks.
template <int BM>
struct WdShape {
    static constexpr int A_ROW = 128, B_ROW = 64;            // bytes of an activation row and of a row of codes
    static constexpr int A_BYTES = BM * A_ROW;
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

// The tile's requests: 64 lanes x 16 (4) bytes from base + the lane's offset to consecutive LDS from `lds` on.
// Inline assembly, because the compiler would otherwise wait for the newest of them ahead of every LDS read.
template <int BYTES>
__device__ __forceinline__ void wd_request(const void *base, uint32_t voff, uint32_t lds) {
    if constexpr (BYTES == 16)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wd_wait_requests() {  // until at most N of this wave's requests are under way
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ void wd_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Codes 2h and 2h + 1 of a dword in the activations' type, exactly.
template <typename XT>
__device__ __forceinline__ uint32_t wd_codes2(uint32_t w, int h) {
    const float lo = static_cast<float>(static_cast<signed char>(w >> (16 * h)));
    const float hi = static_cast<float>(static_cast<signed char>(w >> (16 * h + 8)));
    if constexpr (std::is_same<XT, __bf16>::value)
        return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    else
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
}

template <typename XT>
__device__ __forceinline__ wd_f32x4 wd_mfma(const wd_u32x4 &a, const wd_u32x4 &b) {
    const wd_f32x4 c = {0.f, 0.f, 0.f, 0.f};
    if constexpr (std::is_same<XT, __bf16>::value)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wd_bf16x8, a), __builtin_bit_cast(wd_bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(wd_f16x8, a), __builtin_bit_cast(wd_f16x8, b), c, 0, 0, 0);
}

// Order of the tiles.  Workgroups are dealt to the eight XCDs in turn (id modulo 8) and an XCD runs its own in order, 32
// at a time.  The (M tile, N tile, K slice) triples are numbered with the M tiles of a group of m_group (2048 rows)
// innermost, then the slices of an N tile, then the N tiles, then the groups, and each XCD takes an equal share of
// consecutive numbers: the workgroups in flight on it share each weight tile, and the activation tiles of the group,
// out of its L2.  (Whole N tiles per XCD, the form before, leave XCDs with a tile more than others: 777 x 2880 x 2880,
// 12 N tiles over three slices, 51 against 33 us.)  False: a slot of the padded grid.
__device__ __forceinline__ bool wd_tile(int id, int m_tiles, int n_tiles, int slices, int m_group, int &mt, int &nt, int &slice) {
    const int total = m_tiles * n_tiles * slices, share = total >> 3, more = total & 7;
    const int xcd = id & 7, slot = id >> 3;
    if (slot >= share + (xcd < more ? 1 : 0)) return false;
    const int u = xcd * share + min(xcd, more) + slot;
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
            wd_request<16>(xb + static_cast<size_t>(tt) * 128, a_off[p], st + (wave * S::A_REQ + p) * 1024);
        } else if constexpr (p < S::A_REQ + S::B_REQ) {
            constexpr int q = p - S::A_REQ;
            wd_request<16>(qb + static_cast<size_t>(tt) * 64, b_off[q], st + S::A_BYTES + wave * S::B_WAVE + q * 1024);
        } else {  // a row's two scales are one aligned dword (K / 32 is even)
            wd_request<4>(db + static_cast<size_t>(tt) * 2, s_off, st + S::A_BYTES + S::B_BYTES + wave * 256);
        }
    };
    auto request = [&](int t, int stage) __attribute__((always_inline)) {
        wd_static_for<S::REQ>([&](auto pc) __attribute__((always_inline)) { request_piece(t, stage, pc); });
    };

    // ---- operands
    const int a_lane = r * S::A_ROW + (g ^ a_swizzle(r)) * 16;  // fragment i: + i * 16 rows; block 1: ^ 64
    const int b_lane = S::A_BYTES + wave * S::B_WAVE + r * S::B_ROW + ((g >> 1) ^ b_swizzle(r)) * 16 + (g & 1) * 8;  // n tile 1: + 16 rows; block 1: ^ 32
    const int s_lane = S::A_BYTES + S::B_BYTES + wave * 256 + r * 4;  // n tile 1: + 64
    wd_f32x4 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = wd_f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int AHEAD = 3, RING = AHEAD + 1;  // activation fragments requested from LDS ahead of their use
    static_assert(NF % RING == 0, "the ring has the same phase in every tile");
    wd_u32x4 ar[RING];
    wd_u32x4 bf[2][2];   // weight operands of two successive blocks, [block parity][n tile]
    wd_u32x2 raw[2];     // codes of the block after this one
    float sc[2][2];      // scales [block parity][n tile]
    uint32_t sraw[2];    // the next tile's
    wd_f32x4 sum[2];     // block sums whose scaling is still to be issued
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
        bf[b][p >> 2][p & 3] = wd_codes2<XT>(raw[p >> 2][(p & 3) >> 1], p & 1);
    };

#pragma unroll
    for (int i = 0; i < S::STAGES - 1; ++i) request(i, i);
    wd_wait_requests<(S::STAGES - 2) * S::REQ>();
    wd_barrier();
#pragma unroll
    for (int f = 0; f < AHEAD; ++f) ar[f] = *reinterpret_cast<const wd_u32x4 *>(lds + a_lane + f * 16 * S::A_ROW);
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
        wd_static_for<NF>([&](auto fc) __attribute__((always_inline)) {
            constexpr int f = decltype(fc)::value, b = f / NI, i = f % NI;
            constexpr int bp = (f - 1) / NI, ip = (f + NI - 1) % NI;  // the fragment before this one (f > 0)
            if constexpr (f == 0) read_raw(st + (b_lane ^ 32));  // block 1
            if constexpr (f == NI) {
                // This wave's requests for the next tile have landed, and behind the barrier everybody's; the buffer of
                // the tile before this one is free.
                wd_wait_requests<(S::STAGES - 3) * S::REQ>();
                wd_barrier();
                read_raw(st_next + b_lane);
                read_scales(st_next);
            }
            if constexpr (f > NI && (f - NI - 1) % STEP == 0 && (f - NI - 1) / STEP < S::REQ)
                request_piece(t + S::STAGES - 1, last, std::integral_constant<int, (f - NI - 1) / STEP>{});
            constexpr int fa = f + AHEAD;
            ar[fa % RING] = *reinterpret_cast<const wd_u32x4 *>((fa < NI ? a0 : (fa < NF ? a1 : a2)) + (fa % NI) * 16 * S::A_ROW);
            wd_f32x4 s[2];
            wd_static_for<2>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                // The fences hold the order: left alone, the scheduler issues the matrix steps first and keeps their sums
                // alive.  The sums of the fragment before are scaled under this one's matrix steps.
                __builtin_amdgcn_sched_barrier(0);
                s[j] = wd_mfma<XT>(ar[f % RING], bf[b][j]);
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
    wd_wait_requests<0>();  // no request outlives its buffer, which the epilogue now takes over
    wd_barrier();

    // ---- epilogue.  Accumulator element v of lane (r, g) is row 4 g + v, column r of its 16 x 16 tile: two-byte stores
    // of 32-byte runs.  The wave turns 64 rows at a time round in its own part of LDS and stores 16 bytes per lane.
    constexpr int EP = 36;  // floats per row of 32
    float *ep = reinterpret_cast<float *>(lds) + wave * (64 * EP);
    static_assert(8 * 64 * EP * 4 <= S::LDS, "epilogue buffer");
    constexpr int ESZ = OUT == kWdOutF32 ? 4 : 2, CW = OUT == kWdOutSwiglu ? 4 : 8;  // bytes and columns a lane writes of 8 weight rows
    const size_t pitch = OUT == kWdOutSwiglu ? static_cast<size_t>(ldy >> 1) : static_cast<size_t>(ldy);
    const bool whole = (pitch * ESZ) % (CW * ESZ < 16 ? CW * ESZ : 16) == 0 &&
                       (reinterpret_cast<uintptr_t>(y) & (CW * ESZ < 16 ? CW * ESZ - 1 : 15)) == 0;
    const bool words = (pitch * ESZ) % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 3) == 0;
    const int ecol = (lane & 3) * 8, col = wn0 + ecol;  // eight weight rows per lane, four lanes per row of y
    auto put = [&](size_t at, float v) __attribute__((always_inline)) {
        if constexpr (OUT == kWdOutF32) static_cast<float *>(y)[at] = v;
        else if constexpr (OUT == kWdOutF16) static_cast<_Float16 *>(y)[at] = static_cast<_Float16>(v);
        else static_cast<__bf16 *>(y)[at] = static_cast<__bf16>(v);
    };
#pragma unroll
    for (int i0 = 0; i0 < NI; i0 += 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) ep[(i * 16 + 4 * g + v) * EP + j * 16 + r] = acc[i0 + i][j][v];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int er = q * 16 + (lane >> 2), row = m0 + i0 * 16 + er;
            const wd_f32x4 lo = *reinterpret_cast<const wd_f32x4 *>(ep + er * EP + ecol);
            const wd_f32x4 hi = *reinterpret_cast<const wd_f32x4 *>(ep + er * EP + ecol + 4);
            float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if constexpr (OUT == kWdOutSwiglu) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = swiglu_value(v[2 * e], v[2 * e + 1]);
            }
            if (row >= M) continue;
            const size_t at = static_cast<size_t>(row) * pitch + (OUT == kWdOutSwiglu ? col >> 1 : col);
            if (whole && col + 8 <= n_end) {
                if constexpr (OUT == kWdOutF32) {
                    wd_f32x4 *p = reinterpret_cast<wd_f32x4 *>(static_cast<float *>(y) + at);
                    p[0] = lo;
                    p[1] = hi;
                } else if constexpr (OUT == kWdOutF16) {
                    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
                    f16x8 w;
#pragma unroll
                    for (int e = 0; e < 8; ++e) w[e] = static_cast<_Float16>(v[e]);
                    *reinterpret_cast<f16x8 *>(static_cast<_Float16 *>(y) + at) = w;
                } else {
                    typedef __bf16 bf16xn __attribute__((ext_vector_type(CW)));
                    bf16xn w;
#pragma unroll
                    for (int e = 0; e < CW; ++e) w[e] = static_cast<__bf16>(v[e]);
                    *reinterpret_cast<bf16xn *>(static_cast<__bf16 *>(y) + at) = w;
                }
            } else if (ESZ == 2 && words && col + 8 <= n_end) {  // rows that start on a word only (N even)
#pragma unroll
                for (int e = 0; e < CW; e += 2) {
                    uint32_t w;
                    if constexpr (OUT == kWdOutF16) {
                        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
                        w = __builtin_bit_cast(uint32_t, f16x2{static_cast<_Float16>(v[e]), static_cast<_Float16>(v[e + 1])});
                    } else {
                        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                        w = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(v[e]), static_cast<__bf16>(v[e + 1])});
                    }
                    *reinterpret_cast<uint32_t *>(static_cast<unsigned char *>(y) + (at + e) * 2) = w;
                }
            } else {
#pragma unroll
                for (int e = 0; e < CW; ++e)
                    if (col + (8 / CW) * e < n_end) put(at + e, v[e]);
            }
        }
    }
}

// Weight rows below n_big in tiles of 256x256 (the first big_blocks workgroups), the others in tiles of 128x256
// (wd_big_rows chooses the cut).  With `slices` > 1 every slice of kt_slice K tiles goes into an f32 plane of (M, N) of its
// own.
template <typename XT, int OUT>
__global__ __launch_bounds__(512) void q8_gemm_wide_kernel(const int8_t *__restrict__ qs, const __half *__restrict__ ds,
                                                           const XT *__restrict__ x, void *__restrict__ y, int M, int N, int K,
                                                           int n_big, int big_blocks, int slices, int kt_slice, int ldy) {
    extern __shared__ __attribute__((aligned(16))) unsigned char wd_lds[];
    const int kt_all = K / 64;
    int mt, nt, slice;
    if (static_cast<int>(blockIdx.x) < big_blocks) {
        const int m_tiles = (M + 255) / 256;
        if (!wd_tile(blockIdx.x, m_tiles, n_big / kWdBN, 1, min(m_tiles, 8), mt, nt, slice)) return;
        wd_tile_body<256, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 256, nt * kWdBN, n_big, 0, kt_all, ldy);
        return;
    }
    const int m_tiles = (M + 127) / 128;
    if (!wd_tile(static_cast<int>(blockIdx.x) - big_blocks, m_tiles, (N - n_big + kWdBN - 1) / kWdBN, slices, min(m_tiles, 16), mt, nt, slice))
        return;
    const int kt0 = slice * kt_slice;
    if (slices > 1) y = static_cast<float *>(y) + static_cast<size_t>(slice) * M * N;
    wd_tile_body<128, XT, OUT>(wd_lds, qs, ds, x, y, M, K, mt * 128, n_big + nt * kWdBN, N, kt0, min(kt_slice, kt_all - kt0), ldy);
}

// How many weight rows go to 256x256 tiles.  A tile of either height takes the same time whatever its neighbours do, a
// 256-row one about 1.5 times a 128-row one (2.0 against 1.2-1.3 us per 64 of K), and the launch ends with its slowest CU, so
// the cut is taken where the list of big tiles followed by small ones, dealt to 256 CUs in order, ends first: after the
// last or last but one whole round of big tiles, or with tiles of one height only.
static int wd_big_rows(int64_t m, int64_t n, int64_t *end = nullptr) {
    const int64_t mt256 = (m + 255) / 256, mt128 = (m + 127) / 128;
    const int64_t n_tiles = n / kWdBN, n_all = (n + kWdBN - 1) / kWdBN;  // whole tiles, all of them
    auto ends = [&](int64_t c) {  // in half units of a small tile's time: a big tile is 3, a small one 2
        const int64_t big = mt256 * c, small = mt128 * (n_all - c);
        const int64_t t0 = big / 256 * 3, busy = big % 256;  // 256 - busy CUs are free from t0 on, busy of them from t0 + 3
        int64_t q = busy ? 3 : 0;
        if ((2 * small + 3 * busy) / 256 - 2 > q) q = (2 * small + 3 * busy) / 256 - 2;
        while ((256 - busy) * (q / 2) + (q > 3 ? busy * ((q - 3) / 2) : 0) < small) ++q;
        return t0 + q;
    };
    const int64_t rounds = mt256 * n_tiles / 256;
    const int64_t cuts[3] = {n_tiles, rounds * 256 / mt256, (rounds - 1) * 256 / mt256};
    int64_t best = 0, best_t = ends(0);
    for (int64_t c : cuts)
        if (c > 0 && ends(c) < best_t) best = c, best_t = ends(c);
    if (end) *end = best_t;
    return static_cast<int>(best) * kWdBN;
}

int64_t q8_gemm_wide_ends(int64_t m, int64_t n) {
    int64_t end = 0;
    wd_big_rows(m, n, &end);
    return end;
}

template <typename XT, int OUT>
static lhip_status wd_launch_t(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, int slices,
                               int ldy, hipStream_t s) {
    const int n_big = slices == 1 ? wd_big_rows(m, n) : 0;
    auto blocks = [](int64_t m_tiles, int64_t n_tiles) { return (m_tiles * n_tiles + 7) / 8 * 8; };  // whole eights, see wd_tile
    const int64_t big = blocks((m + 255) / 256, n_big / kWdBN);
    const int64_t small = blocks((m + 127) / 128, static_cast<int64_t>((n - n_big + kWdBN - 1) / kWdBN) * slices);
    if (big + small > 0x7fffffff) return LHIP_ERR_INVALID_SHAPE;  // the grid's x extent
    auto kern = q8_gemm_wide_kernel<XT, OUT>;
    constexpr int lds_small = WdShape<128>::LDS, lds_most = WdShape<256>::LDS;
    static_assert(lds_most >= lds_small, "the opt-in covers both heights");
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), lds_most)) return st;
    const int kt = k / 64, kt_slice = (kt + slices - 1) / slices;
    if (slices < 1 || (slices - 1) * kt_slice >= kt) return LHIP_ERR_UNSUPPORTED;  // an empty slice
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(big + small)), dim3(512),
                       static_cast<unsigned>(n_big > 0 ? lds_most : lds_small), s, qs, ds, static_cast<const XT *>(x), y, m, n, k,
                       n_big, static_cast<int>(big), slices, kt_slice, ldy > 0 ? ldy : n);
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
