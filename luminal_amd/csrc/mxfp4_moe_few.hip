// The exact expert layer (mxfp4_moe_exact.hip: its arithmetic and operands) for a few routed rows, up to kFewRows: tokens decoding.
//
// Every expert's weights are read for a handful of rows, so a launch is bound by the weight stream and by what stands before and
// behind it.  Hence:
//   * no plan launch: a wave holds the routing in its lanes, lane i the expert of routed row i, and finds its tile - up to 16
//     rows of one expert - by ballots;
//   * a column block is 16 (gated: 2 x 16) columns and the four waves of a workgroup split K: a KiB of weights costs the wave that
//     expands it some 140 vector cycles, and 64 columns of all K a wave, the form before, was a chain of 5 us in a launch of 10;
//   * activations come straight from memory in operand order, 64 bytes a lane and chunk (rows the tile does not have repeat its
//     last one), and stay in registers while a workgroup walks several column blocks, whose weights it requests one block ahead
//     (a workgroup a block, requests resting from its last weight until the next workgroup's first: T = 8 79 us);
//   * with up to four routed rows, one token's, the down product has four waves for each of them and adds the experts up.
// Measured, 32 experts of 2880 x 2880, top 4, weights that no cache holds, us a layer with its router, plan form (T = 1: a direct form of 64 columns a wave) -> this:
// T = 1 23.1 -> 21.3, 2 42.6 -> 29.1, 3 52.2 -> 37.1, 4 56.0 -> 41.6, 6 65.4 -> 51.8, 8 73.1 -> 57.8 (4.8 TB/s of weights with the launches),
// 12 77.5 -> 66.3, 16 79.9 -> 73.6.
#include <type_traits>

#include "mxfp4_moe_exact_device.h"

namespace lhip {

constexpr int kFewD = 8;      // most chunks of weights and activations a wave holds: K up to 4096 a segment

// One wave's loads: chunk c of a panel is a KiB of codes, lane (r, g) holding block g of row r, and 64 bytes of scales.
struct FewPanels {
    const uint8_t *codes, *scales;  // of this lane: its piece, the dword that holds its scale byte
    __device__ __forceinline__ void load(size_t at, mu32x4 &q, uint32_t &s) const {
        q = __builtin_nontemporal_load(reinterpret_cast<const mu32x4 *>(codes + at));
        s = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(scales + (at >> 4)));
    }
};
// Lane (r, g)'s activations of chunk c: 32 of row r, block g.  (Past K: the row's first; few_mask_a.)
__device__ __forceinline__ void few_load_a(const __bf16 *row, int K, int c, int grp, mu32x4 (&a)[4]) {
    const int k0 = c * kChunk + grp * 32;
    const mu32x4 *p = reinterpret_cast<const mu32x4 *>(row + (k0 < K ? k0 : 0));
#pragma unroll
    for (int d = 0; d < 4; ++d) a[d] = p[d];
}
__device__ __forceinline__ void few_mask_a(int K, int c, int grp, mu32x4 (&a)[4]) {  // zero times what lies past K need not be zero
    if ((c + 1) * kChunk > K && c * kChunk + grp * 32 >= K) {
#pragma unroll
        for (int d = 0; d < 4; ++d) a[d] = mu32x4{0, 0, 0, 0};
    }
}
__device__ __forceinline__ void few_multiply(const mu32x4 &q, uint32_t scale, const mu32x4 (&a)[4], v4f &acc) {
    v8bf wb[4];
    mx_expand_block(q, scale & 0xffu, wb);
#pragma unroll
    for (int d = 0; d < 4; ++d) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[d]), wb[d], acc, 0, 0, 0);
}

// The tile of a workgroup: tile blockIdx.y of the experts in the order of their first routed row, each in tiles of 16 rows.
struct FewTile {
    int expert, count;  // count: its rows (0: there is no such tile)
    int list;           // lane i < count: the routed row that is its row i
    __device__ __forceinline__ int routed_row(int i) const { return __builtin_amdgcn_ds_bpermute(min(i, count - 1) * 4, list); }
};
__device__ __forceinline__ FewTile few_tile(const int *sel, int n_experts, int R, int *slot_of) {
    const int lane = threadIdx.x & 63;
    const int mine = lane < R ? sel[lane] : -1;
    const bool known = mine >= 0 && mine < n_experts;
    if (slot_of && lane < R) slot_of[lane] = known ? lane : -1;
    uint64_t left = __ballot(known), rows = 0;
    int expert = 0, tile = blockIdx.y;
    while (left != 0) {
        expert = __builtin_amdgcn_readlane(mine, __builtin_ctzll(left));
        rows = __ballot(known && mine == expert);
        const int tiles = (__popcll(rows) + 15) >> 4;
        if (tile < tiles) break;
        tile -= tiles;
        left &= ~rows;
    }
    FewTile t;
    t.expert = expert;
    t.count = left == 0 ? 0 : min(__popcll(rows) - 16 * tile, 16);
    const int rank = __popcll(rows & ((uint64_t{1} << lane) - 1)) - 16 * tile;
    const bool listed = ((rows >> lane) & 1) && rank >= 0 && rank < 16;
    t.list = __builtin_amdgcn_ds_permute((listed ? rank : 63) * 4, lane);
    return t;
}

// Gate|up (GATED: bf16 up * swish(gate) of the activations' rows) or down (f32) of every routed row; results at the routed row's
// number.  grid = (column blocks / `blocks`, tiles at most); a workgroup behind the last tile ends.  A workgroup walks `blocks` column
// blocks of two weight panels (GATED: 16 columns of gate and of up, else 32 columns) of its tile.  Wave w takes chunks w, w + 4, ... of K,
// D of them a segment; while it multiplies a segment it requests the next one's weights, chunk by chunk, and with more than one
// segment (SEG) the activations too, which otherwise stay in registers.
template <bool GATED, int D, bool SEG>
__global__ __launch_bounds__(256, 2) void mx_moe_few_kernel(const int *sel, const uint8_t *w_nib, const uint8_t *w_sc, const __bf16 *a,
                                                            int rows_per_expert, int K, int Kp, int N, int n_experts, int R,
                                                            int a_div, int blocks, int *slot_of, void *out) {
    constexpr int NT = 2, COLS = GATED ? 16 : 32;
    __shared__ float part[2][4][NT][4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, grp = lane >> 4;
    const FewTile t = few_tile(sel, n_experts, R, GATED && blockIdx.x == 0 && blockIdx.y == 0 && wave == 0 ? slot_of : nullptr);
    if (t.count == 0) return;
    const int entry = t.routed_row(r), m = 4 * grp + wave, to = t.routed_row(m);

    const int chunks = Kp / kChunk, segs = SEG ? (chunks + 4 * D - 1) / (4 * D) : 1;
    const int b0 = blockIdx.x * blocks, b1 = min(b0 + blocks, N / COLS);
    // panel f of column block b: f panels of the expert's half (gate, up) or of the block (32 columns) further on
    const size_t panel_bytes = static_cast<size_t>(chunks) * 1024;
    const size_t panel0 = (static_cast<size_t>(t.expert) * rows_per_expert) >> 4;
    const size_t step = GATED ? 1 : 2, second = GATED ? static_cast<size_t>(N >> 4) : 1;
    const FewPanels w{w_nib + panel0 * panel_bytes + lane * 16, w_sc + panel0 * (panel_bytes >> 4) + (lane & ~3)};
    const int s_shift = 8 * (lane & 3);
    const __bf16 *a_row = a + static_cast<size_t>(GATED ? entry / a_div : entry) * K;
    mu32x4 q[D][NT], av[D][4];
    uint32_t sc[D][NT];
    auto chunk_of = [&](int seg, int j) { return (seg * D + j) * 4 + wave; };
    auto load_w = [&](int j, int b, int seg) __attribute__((always_inline)) {
        const int c = min(chunk_of(seg, j), chunks - 1);
#pragma unroll
        for (int f = 0; f < NT; ++f) w.load((b * step + f * second) * panel_bytes + static_cast<size_t>(c) * 1024, q[j][f], sc[j][f]);
    };
    auto load_a = [&](int j, int seg) __attribute__((always_inline)) { few_load_a(a_row, K, min(chunk_of(seg, j), chunks - 1), grp, av[j]); };
#pragma unroll
    for (int j = 0; j < D; ++j) {
        load_w(j, b0, 0);
        load_a(j, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!SEG) {
#pragma unroll
        for (int j = 0; j < D; ++j) few_mask_a(K, chunk_of(0, j), grp, av[j]);
    }
    v4f acc[NT];
#pragma unroll
    for (int f = 0; f < NT; ++f) acc[f] = v4f{0.f, 0.f, 0.f, 0.f};
    auto segment = [&](int seg, int next_b, int next_seg, auto more) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
#pragma unroll
            for (int f = 0; f < NT; ++f) asm volatile("" : "+v"(q[j][f]), "+v"(sc[j][f]));
            const int c = chunk_of(seg, j);
            if (c < chunks) {  // wave-uniform
                if constexpr (SEG) few_mask_a(K, c, grp, av[j]);
#pragma unroll
                for (int f = 0; f < NT; ++f) few_multiply(q[j][f], sc[j][f] >> s_shift, av[j], acc[f]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (decltype(more)::value) {
                load_w(j, next_b, next_seg);
                if constexpr (SEG) load_a(j, next_seg);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The waves' shares, added in wave order: thread (wave, lane) takes element `wave`, row 4 grp + wave of column r.
    auto finish = [&](int b) __attribute__((always_inline)) {
        float(&mine)[4][NT][4][64] = part[(b - b0) & 1];  // (free again: everybody has passed the barrier of the block between)
#pragma unroll
        for (int f = 0; f < NT; ++f) {
#pragma unroll
            for (int v = 0; v < 4; ++v) mine[wave][f][v][lane] = acc[f][v];
            acc[f] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        __syncthreads();
        float sum[NT];
#pragma unroll
        for (int f = 0; f < NT; ++f)
            sum[f] = ((mine[0][f][wave][lane] + mine[1][f][wave][lane]) + mine[2][f][wave][lane]) + mine[3][f][wave][lane];
        if (m < t.count) {
            const size_t at = static_cast<size_t>(to) * N + b * COLS + r;
            if constexpr (GATED) {
                static_cast<__bf16 *>(out)[at] = static_cast<__bf16>(exact_swiglu(sum[0], sum[1]));
            } else {
                static_cast<float *>(out)[at] = sum[0];
                static_cast<float *>(out)[at + 16] = sum[1];
            }
        }
    };
    int b = b0, seg = 0;
    while (true) {
        const bool whole = seg + 1 == segs;
        const int next_b = whole ? b + 1 : b, next_seg = whole ? 0 : seg + 1;
        if (next_b == b1) break;
        segment(seg, next_b, next_seg, std::true_type{});
        if (whole) finish(b);
        b = next_b;
        seg = next_seg;
    }
    segment(seg, 0, 0, std::false_type{});
    finish(b);
}

// Down projection of up to four routed rows with the weighted sum over a token's experts folded in: a workgroup owns 16 output columns
// of all of them, four waves each, which split K: D chunks of weights in flight (all of them, K up to 512 D), AD of activations.
template <int D>
__global__ __launch_bounds__(64 * 4 * kDirectRows) void mx_moe_few_down_kernel(const int *sel, const uint8_t *w_nib, const uint8_t *w_sc,
                                                                               const __bf16 *act, int rows_per_expert, int K, int Kp,
                                                                               int N, int n_experts, int R, int topk, const float *wts,
                                                                               float *out, __bf16 *y) {
    constexpr int AD = D < 3 ? D : 3;
    static_assert(D % AD == 0, "the ring has the same phase in every segment");
    __shared__ float part[kDirectRows][4][16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, grp = lane >> 4, t = wave >> 2;
    const int n0 = blockIdx.x * 16, chunks = Kp / kChunk;
    const int mine = lane < R ? sel[lane] : -1;
    const float weight = lane < R ? wts[lane] : 0.f;
    const __bf16 *a_row = act + static_cast<size_t>(min(t, R - 1)) * K;  // all sixteen rows of the fragment
    mu32x4 q[D], av[AD][4];
    uint32_t sc[D];
    auto chunk_of = [&](int step) { return 4 * step + (wave & 3); };
    auto load_a = [&](int set, int step) __attribute__((always_inline)) { few_load_a(a_row, K, min(chunk_of(step), chunks - 1), grp, av[set]); };
#pragma unroll
    for (int j = 0; j < AD; ++j) load_a(j, j);  // ahead of the weights, whose address is still to come
    __builtin_amdgcn_sched_barrier(0);
    const uint64_t known = __ballot(mine >= 0 && mine < n_experts);
    if ((known >> t) & 1) {  // wave-uniform
        const int expert = __builtin_amdgcn_readlane(mine, t), s_shift = 8 * (lane & 3);
        const size_t at0 = ((static_cast<size_t>(expert) * rows_per_expert + n0) >> 4) * chunks * 1024;
        const FewPanels w{w_nib + lane * 16 + at0, w_sc + (lane & ~3) + (at0 >> 4)};
        auto load_w = [&](int set, int step) __attribute__((always_inline)) {
            w.load(static_cast<size_t>(min(chunk_of(step), chunks - 1)) * 1024, q[set], sc[set]);
        };
#pragma unroll
        for (int j = 0; j < D; ++j) load_w(j, j);
        __builtin_amdgcn_sched_barrier(0);
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        auto segment = [&](int s0, auto more) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < D; ++j) {
                asm volatile("" : "+v"(q[j]), "+v"(sc[j]));
                const int c = chunk_of(s0 + j);
                if (c < chunks) {  // wave-uniform
                    few_mask_a(K, c, grp, av[j % AD]);
                    few_multiply(q[j], sc[j] >> s_shift, av[j % AD], acc);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (decltype(more)::value) load_w(j, s0 + j + D);
                if (decltype(more)::value || j + AD < D) load_a(j % AD, s0 + j + AD);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int s0 = 0;
        for (; 4 * (s0 + D) < chunks; s0 += D) segment(s0, std::true_type{});
        segment(s0, std::false_type{});
        if (grp == 0) part[t][wave & 3][r] = acc[0];
    }
    __syncthreads();
    if (wave != 0) return;
    float wt[kDirectRows], down[kDirectRows];
#pragma unroll
    for (int i = 0; i < kDirectRows; ++i) wt[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), i));
    if (grp != 0) return;
    const int col = n0 + r;
#pragma unroll
    for (int i = 0; i < kDirectRows; ++i) {
        down[i] = (known >> i) & 1 ? ((part[i][0][r] + part[i][1][r]) + part[i][2][r]) + part[i][3][r] : 0.f;
        if (i < R) out[static_cast<size_t>(i) * N + col] = down[i];
    }
    for (int token = 0; token * topk < R; ++token) {
        float sum = 0.f;
        for (int k = 0; k < topk; ++k) {
            const int i = token * topk + k;
            const float d = i == 0 ? down[0] : i == 1 ? down[1] : i == 2 ? down[2] : down[3];
            const float wi = i == 0 ? wt[0] : i == 1 ? wt[1] : i == 2 ? wt[2] : wt[3];
            if ((known >> i) & 1) sum = fmaf(wi, d, sum);
        }
        y[static_cast<size_t>(token) * N + col] = static_cast<__bf16>(sum);
    }
}

// Experts that T tokens' choices are expected to touch (T small).
static double few_tiles(int T, int E, int topk) {
    double none = 1.0;  // an expert's chance of no row
    for (int i = 0; i < T; ++i) none *= 1.0 - static_cast<double>(topk) / E;
    return E * (1.0 - none);
}

// Column blocks a workgroup walks.  Two workgroups are resident a CU; with as many as one round of them takes, requests never stop, and
// five (32 columns: six) are the most, beyond which workgroups of few tiles leave the CUs at different times.  Where the blocks of all
// expected tiles are up to six a CU, the number of at most three with which the fullest CU walks the fewest, half a block counted for each
// of its workgroups: of 1080 launches (760 layers of 4 to 64 experts, up to 6144 wide, T = 1 to 8) 1.0 % behind the best number on average.
// Measured, us a layer by (gate|up, down) blocks, 32 experts of 2880 x 2880, top 4: T = 2 (3, 3) 29.2, (5, 3) 32.4, (2, 1) 33.6; T = 4 (5, 3) 41.6,
// (3, 3) 43.9, (12, 6) 42.5; T = 8 (5, 5) 59.2, (3, 1) 69.5; T = 16 (5, 6) 73.1, (3, 3) 79.9, (8, 4) 83.8.  By the fullest CU, gate|up in 1 / 2 / 3 /
// 4 blocks: four tiles of 4096 x 4096 - / 27.7 / 30.0 / 27.8, of 3840 x 2240 (three) 18.5 / 17.7 / 19.2 / 20.3, of 2880 - / 22.9 / 21.9 / 22.6, of 3392 x 896
// 12.8 / 14.1 / 15.0 / 16.4.
static int few_blocks(const MoeFewLayer &l, int all, int most) {
    const double tiles = few_tiles(l.T, l.E, l.topk), units = tiles * all;
    if (units <= 1500.0) {
        int blocks = 1;
        double least = 1e30;
        const int whole = static_cast<int>(tiles);
        const double more = tiles - whole;
        for (int b = 1; b <= 3; ++b) {
            const int columns = (all + b - 1) / b;
            auto turns = [&](int n) { return (b + 0.5) * ((n * columns + 255) / 256); };  // of n tiles
            const double expected = (1.0 - more) * turns(whole) + more * turns(whole + 1);
            if (expected < least) least = expected, blocks = b;
        }
        return blocks;
    }
    const int blocks = static_cast<int>(units / 480.0) + 1;
    return blocks > most ? most : blocks;
}

template <bool GATED>
static lhip_status launch_few(const uint8_t *nib, const uint8_t *sc, const __bf16 *a, const MoeFewLayer &l, int rows_per_expert, int K, int N,
                              void *out, hipStream_t s) {
    const int R = l.T * l.topk, Kp = static_cast<int>(pad128(K)), steps = (Kp / kChunk + 3) / 4;
    const unsigned tiles = static_cast<unsigned>(R < l.E + R / 16 ? R : l.E + R / 16);  // at most
    const int all = N / (GATED ? 16 : 32), blocks = few_blocks(l, all, GATED ? 5 : 6);
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((all + blocks - 1) / blocks), tiles), dim3(256), 0, s, l.sel, nib, sc, a,
                           rows_per_expert, K, Kp, N, l.E, R, l.topk, blocks, l.slot_of, out);
    };
    // a segment of as many chunks a wave as K has, or of equal parts of it
    const int segs = (steps + kFewD - 1) / kFewD, per = (steps + segs - 1) / segs;
    if (segs > 1) {
        if (per <= 6) launch(mx_moe_few_kernel<GATED, 6, true>);
        else if (per == 7) launch(mx_moe_few_kernel<GATED, 7, true>);
        else launch(mx_moe_few_kernel<GATED, 8, true>);
    } else if (per <= 2) launch(mx_moe_few_kernel<GATED, 2, false>);
    else if (per == 3) launch(mx_moe_few_kernel<GATED, 3, false>);
    else if (per == 4) launch(mx_moe_few_kernel<GATED, 4, false>);
    else if (per <= 6) launch(mx_moe_few_kernel<GATED, 6, false>);
    else launch(mx_moe_few_kernel<GATED, kFewD, false>);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

// A K of several segments pays while the tiles are few: 8 experts of 4096 x 14336, top 2, T = 1 118 -> 43 us, T = 16 147 -> 125 (T = 20 of them
// 150 and 131); 32 of 5120 x 5120, top 2, T = 6 103 -> 97, T = 8 110 <- 116.  A hidden size of several segments re-reads the activations
// besides: from seven experts and 420 MB of weights on the plan's tiles are ahead (16 of 5120 x 8192, top 1, T = 8 104 <- 116, T = 24 160 <- 182;
// 8 of 6144 x 6144, top 2, T = 12 98 <- 109; the other way T = 6 96 -> 85, 4 of 8192 x 8192, T = 8 112 -> 93).
bool moe_few_takes(int T, int H, int I, int E, int topk) {
    const int64_t R = static_cast<int64_t>(T) * topk;
    if (R > kFewRows || (H <= 512 * kFewD && I <= 512 * kFewD)) return R <= kFewRows;
    const double experts = few_tiles(T, E, topk);
    if (H > 512 * kFewD && experts > 6.0 && experts * 1.6 * H * I > 420e6) return false;
    return R <= (E <= 16 ? 32 : 12);
}

lhip_status moe_few_forward(const MoeFewLayer &l, hipStream_t s) {
    const int R = l.T * l.topk;
    if (lhip_status st = launch_few<true>(l.gu, l.gu_sc, l.x, l, 2 * l.I, l.H, l.I, l.act, s)) return st;
    if (R <= kDirectRows) {
        const int Kp = static_cast<int>(pad128(l.I)), steps = (Kp / kChunk + 3) / 4;
        auto kern = steps <= 2 ? mx_moe_few_down_kernel<2> : steps == 3 ? mx_moe_few_down_kernel<3> : mx_moe_few_down_kernel<6>;
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(l.H / 16)), dim3(64 * 4 * kDirectRows), 0, s, l.sel, l.dn, l.dn_sc, l.act, l.H,
                           l.I, Kp, l.H, l.E, R, l.topk, l.wts, l.out, l.y);
        LHIP_CHECK_LAUNCH();
        return LHIP_OK;
    }
    if (lhip_status st = launch_few<false>(l.dn, l.dn_sc, l.act, l, l.H, l.I, l.H, l.out, s)) return st;
    return moe_launch_combine(l.out, l.slot_of, l.wts, l.y, l.T, l.H, l.topk, s);
}

}  // namespace lhip
