// Grouped GEMM of the exact expert layer for experts of many rows (see mxfp4_moe_exact.hip for the arithmetic, which is the same:
// e2m1 codes times their block's scale expanded to bf16 exactly, f32 accumulation on the bf16 matrix instruction).
//
// A workgroup of four waves owns up to 96 routed rows of one expert and 256 weight rows, a wave 64 of these (two tiles of 32;
// gated: a tile is 16 rows of gate and the same 16 of up).  K goes by in stages of 64.
//
// What bounds it: the matrix pipe is busy for 60 % of the launch at T = 1024 (56 % in the down product), vector instructions are issued for
// 32 % (27 %), LDS works for 26 % (25 %); the rest are the waits of a workgroup's four waves for each other, for LDS and for memory at
// every stage, so as many workgroups as possible share a CU and a stage costs each as little as possible (variants' times are of the
// layer of 32 experts of 2880 x 2880, top 4, while this form took 240 to 246 us at T = 1024 and 147 to 155 at T = 512):
//   * v_mfma_f32_32x32x16: half the issue slots of 16x16x32, and an activation operand read from LDS feeds two of them (one, with
//     32 weight rows a wave: LDS holds up the matrix pipe, T = 1024 292 us);
//   * everything arrives in LDS by direct loads, and a wave keeps nothing of the next stage in registers: 150 registers, three
//     workgroups a CU.  Two with a third stage of activations: T = 1024 273 us.  Weights held a stage ahead in registers: the
//     compiler's waits for them count the direct loads too, and stop at those;
//   * activation fragments that the tile does not have are not requested (all 96 rows always: 5 % slower at T = 1024);
//   * tiles of 128 rows, and of 64, are level or slower (T = 1024 289 and 259, T = 512 173 and 172), of 160 rows at two workgroups a CU
//     241 at T = 1024 and 174 at T = 512.
// A stage takes longer when the workgroup is alone on its CU (4 experts of 2048 x 2048 at 32 rows, 64 workgroups: 58 us, by 64-row tiles
// 47), so this is taken only where there are enough (exact_tile_fragments).  Measured, us per layer, 64-row tiles of mx_moe_gemm_exact_kernel -> this: T = 192 117 ->
// 110, T = 512 184 -> 147, T = 1024 266 -> 231 (880 TFLOP/s of useful work), T = 2048 449 -> 409.
#include <algorithm>

#include "lds_request.h"
#include "mxfp4_moe_exact_device.h"

namespace lhip {

typedef float v16f __attribute__((ext_vector_type(16)));

struct TallShape {
    static constexpr int MF = kTallRows / 32;         // 32-row activation fragments
    static constexpr int NJ = 2, NW = 4;              // weight tiles of 32 a wave, waves
    static constexpr int A_STAGES = 2, W_STAGES = 3;  // the weights come from further away, and are each wave's own
    static constexpr int A_STAGE = kTallRows * 128;   // a row's 64 values
    static constexpr int W_WAVE = NJ * 1024 + 256;    // a wave's codes; its scales (128 bytes, twice)
    static constexpr int W_BASE = A_STAGES * A_STAGE;
    static constexpr int LDS = W_BASE + NW * W_STAGES * W_WAVE;
    static constexpr int W_REQ = NJ + 1;              // requests of a stage's weights
    static_assert(3 * LDS <= 160 * 1024, "three workgroups a CU");
};

// Until at most N of this wave's requests are under way and its LDS accesses are done.
template <int N>
__device__ __forceinline__ void tall_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(N) : "memory");
}

template <bool GATED>
__global__ __launch_bounds__(64 * TallShape::NW, 3) void mx_moe_gemm_tall_kernel(MoeExactArgs g) {
    using S = TallShape;
    constexpr int MF = S::MF, NJ = S::NJ, NW = S::NW, AS = S::A_STAGES, WS = S::W_STAGES;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    int tile, cb, expert, row0, rows;
    exact_tile(g, tile, cb, expert, row0, rows);
    if (rows == 0) return;
    expert = __builtin_amdgcn_readfirstlane(expert);
    row0 = __builtin_amdgcn_readfirstlane(row0);
    rows = __builtin_amdgcn_readfirstlane(rows);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int K = g.K, stages = (K + 63) / 64;
    const int frags = (rows + 31) >> 5;

    // ---- requests of weights.  A 16-row panel's KiB of a 128-wide chunk is (block, row) pieces of 16 bytes, so a stage is one
    // half of it; lane (r, h) asks for block h of the stage, of row r of the tile, which is what it multiplies.  The stage's
    // scales are 32 bytes a panel: lanes 0 to 31 hold the four panels', the others repeat them.
    const int n_first = (cb * NW + wave) * NJ * (GATED ? 16 : 32);  // the wave's first column
    const bool idle = n_first >= g.N;                               // a wave without columns only stages activations
    const uint32_t panel_bytes = static_cast<uint32_t>(g.Kp / kChunk) * 1024u;
    auto panel_of = [&](int j, int half) {  // (a tile past the last column repeats the last panel, unused)
        return static_cast<uint32_t>(GATED ? (min(n_first + 16 * j, g.N - 16) + half * g.N) >> 4 : min(n_first + 32 * j + 16 * half, g.N - 16) >> 4);
    };
    const size_t expert_panel = static_cast<size_t>(expert) * g.rows_per_expert >> 4;
    const uint8_t *w_base = g.w_nib + expert_panel * panel_bytes;
    const uint8_t *s_base = g.w_sc + expert_panel * (panel_bytes >> 4);
    uint32_t w_off[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) w_off[j] = panel_of(j, (lane >> 4) & 1) * panel_bytes + h * 256 + (lane & 15) * 16;
    const uint32_t s_off = panel_of((lane >> 4) & (NJ - 1), (lane >> 3) & 1) * (panel_bytes >> 4) + (lane & 7) * 4;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char *)lds));
    const int w_lds = S::W_BASE + wave * WS * S::W_WAVE;
    auto request_w = [&](int t, int buf) __attribute__((always_inline)) {
        const int tt = min(t, stages - 1);  // past the end: the last stage again, never used
        const uint32_t dst = lds0 + w_lds + buf * S::W_WAVE;
#pragma unroll
        for (int j = 0; j < NJ; ++j) lds_request<16>(w_base + static_cast<size_t>(tt) * 512, w_off[j], dst + j * 1024);
        lds_request<4>(s_base + static_cast<size_t>(tt) * 32, s_off, dst + NJ * 1024);
    };

    // ---- requests of activations: number q of a wave brings eight rows of fragment q; piece p of a row lies at slot
    // p ^ (row / 2 % 8), which gives the fragment reads 16 lanes on 16 different slots of two rows.
    static_assert(NW * 8 == 32, "a fragment is one request of each wave");
    const int a_piece = (lane & 7) ^ ((lane >> 4) & 3) ^ ((wave & 1) * 4);
    uint32_t a_off[MF];
#pragma unroll
    for (int q = 0; q < MF; ++q) {
        const int slot = row0 + min(q * 32 + wave * 8 + (lane >> 3), rows - 1);  // rows past the tile repeat its last
        const int arow = g.a_index ? g.a_index[slot] / g.a_div : slot - row0;
        a_off[q] = static_cast<uint32_t>(arow) * static_cast<uint32_t>(K) * 2u + a_piece * 16u;
    }
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(g.a) + (g.a_index ? 0 : static_cast<size_t>(row0) * K * 2);
    auto request_a = [&](int t, int buf) __attribute__((always_inline)) {
        const int tt = min(t, stages - 1);
        const uint8_t *base = a_base + static_cast<size_t>(tt) * 128;
        const bool whole = tt * 64 + 64 <= K;
        const bool in = tt * 64 + a_piece * 8 < K;  // pieces past K are zeros: the padding weights are, but zero times what lies there need not be
#pragma unroll
        for (int q = 0; q < MF; ++q) {
            if (q >= frags) continue;
            const int at = buf * S::A_STAGE + (q * NW + wave) * 1024;
            if (whole) lds_request<16>(base, a_off[q], lds0 + at);
            else if (in) lds_request<16>(base, a_off[q], lds0 + at);
            else *reinterpret_cast<mu32x4 *>(lds + at + lane * 16) = mu32x4{0, 0, 0, 0};
        }
    };

    v16f acc[MF][NJ];
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    // Step d of a stage takes dword d of a lane's codes: k = 32 h + 8 d .. + 7.
    const int a_lane = r * 128 + (((4 * h) ^ ((r >> 1) & 7)) & 7) * 16;  // step d: ^ 16 d; fragment i: + 4096 i
    const int s_lane = w_lds + NJ * 1024 + (r >> 4) * 32 + h * 16 + (r & 15);
    constexpr int AHEAD = 2, RING = AHEAD + 1, UNITS = 4 * MF;  // activation operands requested from LDS ahead of their use
    v8bf ar[RING], wb[2][NJ];
    mu32x4 raw[NJ];  // a stage's codes and scales
    float scale[NJ];
    auto expand = [&](auto dc, auto pc) __attribute__((always_inline)) {  // conversion p of 4 NJ of step d
        constexpr int d = decltype(dc)::value, j = decltype(pc)::value >> 2, b = decltype(pc)::value & 3;
        const v2bf v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw[j][d], scale[j], b);
        wb[d & 1][j][2 * b] = v[0];
        wb[d & 1][j][2 * b + 1] = v[1];
    };
    auto stage = [&](int t, auto turn) __attribute__((always_inline)) {
        constexpr int as = decltype(turn)::value % AS, ws = decltype(turn)::value % WS;
        // Of this wave's requests only the weights of the stage after this one may be under way (a stage requests the next
        // one's activations, then the weights of the one after it).  Behind the barrier everybody's activations of this
        // stage are there, and the buffer of the stage before is free.
        tall_wait<S::W_REQ>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        request_a(t + AS - 1, (as + AS - 1) % AS);
        request_w(t + WS - 1, (ws + WS - 1) % WS);
        if (idle) return;
        const unsigned char *a_buf = lds + as * S::A_STAGE;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            raw[j] = *reinterpret_cast<const mu32x4 *>(lds + w_lds + ws * S::W_WAVE + j * 1024 + lane * 16);
            scale[j] = __uint_as_float(static_cast<uint32_t>(*(lds + s_lane + ws * S::W_WAVE + j * 64)) << 23);
        }
        auto read_a = [&](auto uc) __attribute__((always_inline)) {
            constexpr int u = decltype(uc)::value, d = u / MF, i = u % MF;
            ar[u % RING] = *reinterpret_cast<const v8bf *>(a_buf + (a_lane ^ (16 * d)) + i * 4096);
        };
        static_for_n<AHEAD>([&](auto uc) __attribute__((always_inline)) { read_a(uc); });
        __builtin_amdgcn_sched_barrier(0);
        static_for_n<4 * NJ>([&](auto pc) __attribute__((always_inline)) { expand(std::integral_constant<int, 0>{}, pc); });
        static_for_n<UNITS>([&](auto uc) __attribute__((always_inline)) {
            constexpr int u = decltype(uc)::value, d = u / MF, i = u % MF;
            if constexpr (u + AHEAD < UNITS) read_a(std::integral_constant<int, u + AHEAD>{});
            __builtin_amdgcn_sched_barrier(0);
            int live = frags;
            asm volatile("" : "+s"(live));  // (compared anew: kept as a mask the comparison costs vector instructions)
            if (i < live) {
                static_for_n<NJ>([&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ar[u % RING], wb[d & 1][j], acc[i][j], 0, 0, 0);
                    asm volatile("" : "+v"(acc[i][j]));
                });
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (d < 3) {
                constexpr int P0 = i * 4 * NJ / MF, P1 = (i + 1) * 4 * NJ / MF;
                static_for_n<P1 - P0>([&](auto pc) __attribute__((always_inline)) {
                    expand(std::integral_constant<int, d + 1>{}, std::integral_constant<int, P0 + decltype(pc)::value>{});
                });
            }
        });
    };
    static_assert(AS == 2 && WS == 3, "the order of requests and their wait");
    request_w(0, 0);
    request_a(0, 0);
    request_w(1, 1);
    constexpr int TURN = AS * WS;
    for (int t = 0; t < stages; t += TURN) {
        bool more = true;
        static_for_n<TURN>([&](auto jc) __attribute__((always_inline)) {
            if (more) stage(t + decltype(jc)::value, jc);
            if (t + decltype(jc)::value + 1 >= stages) more = false;
        });
    }
    tall_wait<0>();  // no request outlives its buffer, which the epilogue now takes over
    if (idle) return;

    // ---- epilogue: acc[i][j][v] is row 32 i + 8 (v / 4) + 4 h + v % 4, weight row r of tile j.  A fragment's rows are turned round
    // in the wave's own part of the weights' buffers, so that a lane stores 16 bytes.  (N is a multiple of 32.)
    unsigned char *ep = lds + w_lds;
#pragma unroll
    for (int i = 0; i < MF; ++i) {
        if (i >= frags) break;
        if constexpr (GATED) {
            constexpr int COLS = 16 * NJ, PITCH = COLS * 2 + 16, LANES = COLS / 8;  // LANES a row
            static_assert(32 * PITCH <= WS * S::W_WAVE, "epilogue buffer");
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int v = 0; v < 16; v += 2) {
                    // Lanes of rows 0 and 2 hold gate values, of rows 1 and 3 up values of the same columns: two elements trade
                    // halves, and every lane has a pair.
                    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][j][v]), __float_as_uint(acc[i][j][v + 1]), false, false);
                    const float y = exact_swiglu(__uint_as_float(p[0]), __uint_as_float(p[1]));
                    const int m = 8 * (v >> 2) + 4 * h + (v & 3) + ((lane >> 4) & 1);
                    *reinterpret_cast<__bf16 *>(ep + m * PITCH + (16 * j + (lane & 15)) * 2) = static_cast<__bf16>(y);
                }
#pragma unroll
            for (int q = 0; q < LANES / 2; ++q) {
                const int m = q * (64 / LANES) + lane / LANES, c = lane % LANES;
                const mu32x4 y = *reinterpret_cast<const mu32x4 *>(ep + m * PITCH + c * 16);
                if (i * 32 + m < rows)
                    *reinterpret_cast<mu32x4 *>(static_cast<__bf16 *>(g.out) + static_cast<size_t>(row0 + i * 32 + m) * g.N + n_first + c * 8) = y;
            }
        } else {
            constexpr int PITCH = 36 * 4;
            static_assert(32 * PITCH <= WS * S::W_WAVE, "epilogue buffer");
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if (n_first + 32 * j >= g.N) break;
#pragma unroll
                for (int v = 0; v < 16; ++v) *reinterpret_cast<float *>(ep + (8 * (v >> 2) + 4 * h + (v & 3)) * PITCH + r * 4) = acc[i][j][v];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int m = q * 8 + (lane >> 3), c = lane & 7;
                    const mu32x4 y = *reinterpret_cast<const mu32x4 *>(ep + m * PITCH + c * 16);
                    if (i * 32 + m < rows)
                        *reinterpret_cast<mu32x4 *>(static_cast<float *>(g.out) + static_cast<size_t>(row0 + i * 32 + m) * g.N + n_first + 32 * j + c * 4) = y;
                }
            }
        }
    }
}

bool moe_tall_supports(int64_t t, int64_t h, int64_t i) {
    const int64_t rows = t > kTallRows ? t : kTallRows;  // rows of x, and of a tile
    return std::max({rows * h * 2, kTallRows * i * 2, i * pad128(h), h * pad128(i) / 2}) < (int64_t{1} << 32);
}

template <bool GATED>
static lhip_status launch_tall(const MoeExactArgs &a, int max_tiles, hipStream_t s) {
    auto kern = mx_moe_gemm_tall_kernel<GATED>;
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), TallShape::LDS)) return st;
    constexpr int cols = TallShape::NW * TallShape::NJ * (GATED ? 16 : 32);
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((a.N + cols - 1) / cols), static_cast<unsigned>(max_tiles)),
                       dim3(64 * TallShape::NW), TallShape::LDS, s, a);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

lhip_status moe_tall_gemm(const MoeExactArgs &a, bool gated, int max_tiles, hipStream_t s) {
    return gated ? launch_tall<true>(a, max_tiles, s) : launch_tall<false>(a, max_tiles, s);
}

}  // namespace lhip
