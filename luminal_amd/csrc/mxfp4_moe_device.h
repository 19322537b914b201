// Shared pieces of the MXFP4 mixture-of-experts kernels (mxfp4_moe.hip: the block-scaled fast form;
// mxfp4_moe_exact.hip: the bf16 form): tile plan, workspace layout, small device helpers.
#pragma once

#include "common.h"

#include <type_traits>
#include <utility>

namespace lhip {


typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t mu32x4 __attribute__((ext_vector_type(4)));

constexpr int kChunk = 128;      // K elements per MFMA
constexpr int kLoShift = 5;      // the lo plane of an activation is held times 2^5 and multiplied with block scale - 5
constexpr float kLoGain = 32.f;
constexpr int kARow = 160;       // LDS bytes per activation row of a chunk: 128 fp8 + 32 padding (with 16 the fragment reads,
                                 // lane (r, g) at r * pitch + 16 g, take twice as long: measured 8.0 against 4.3 cycles per read)

static inline int64_t pad128(int64_t k) { return (k + 127) / 128 * 128; }

// ---------------------------------------------------------------------------
// Plan: group the R = T*topk routed entries by expert and cut each expert's rows
// into tiles of BM.  One workgroup; E <= 1024.
// ---------------------------------------------------------------------------
struct MoePlan {
    int *offsets;      // [E+1] first slot of each expert
    int *slot_src;     // [R]   slot -> routed entry r = t*topk + s
    int *slot_of;      // [R]   routed entry -> slot (-1 if its expert id is invalid)
    int *tile_expert;  // [max_tiles]
    int *tile_row0;    // [max_tiles] first slot of the tile
    int *tile_rows;    // [max_tiles] valid rows in the tile (0 = unused entry)
    // [max_tiles] the run of a tile: the consecutive list entries that hold tiles of the same expert (on the same XCD)
    // start at entry tile_run0 and number tile_runlen (0 = unused entry).  The exact
    // GEMMs walk a run column block by column block, so that the workgroups that read the same weights run together.
    int *tile_run0, *tile_runlen;
    int *n_tiles;      // [1]
    int max_tiles;     // entries of the tile arrays
    int by_rows;       // whether experts are listed by their rows (else in their own order)
    int fragment;      // rows of a matrix step: a tile is some number of these, but for the end of an expert
    // The list is cut into eight ranges of this many entries, one per XCD (range x is read by the workgroups whose
    // dispatch number is x modulo 8), and the
    // tiles, an expert's behind each other, are dealt to the ranges in eight contiguous, equal shares: the tiles of an
    // expert, and all column blocks of a tile, then run on one XCD and find each other's weights and
    // activation rows in its L2.
    int tiles_per_xcd;
};

__device__ __forceinline__ void moe_plan_block(const int *__restrict__ sel, int R, int E, int BM, const MoePlan &p) {
    // The counts and places of all experts are read by every expert's thread, four at a time.
    __shared__ __attribute__((aligned(16))) int cnt[1024], pos[1024], tiles[1024];
    __shared__ int off[1025], cur[1024];
    constexpr int KEEP = 4;  // routed entries a thread keeps in registers between the two passes over them
    int kept[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int r = threadIdx.x + i * 1024;
        kept[i] = r < R ? sel[r] : -1;
    }
    for (int e = threadIdx.x; e < 1024; e += 1024) {  // (all of them: those from E on are read in fours)
        cnt[e] = 0;
        cur[e] = 0;
        pos[e] = 1024;
        tiles[e] = 0;
    }
    for (int t = threadIdx.x; t < p.max_tiles; t += 1024) {  // entries no tile is written to stay marked unused
        p.tile_expert[t] = 0;
        p.tile_row0[t] = 0;
        p.tile_rows[t] = 0;
        p.tile_run0[t] = t;
        p.tile_runlen[t] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
        if (kept[i] >= 0 && kept[i] < E) atomicAdd(&cnt[kept[i]], 1);
    for (int r = threadIdx.x + KEEP * 1024; r < R; r += 1024) {
        const int e = sel[r];
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    const int4 *cnt4 = reinterpret_cast<const int4 *>(cnt), *pos4 = reinterpret_cast<const int4 *>(pos), *tiles4 = reinterpret_cast<const int4 *>(tiles);
    const int E4 = (E + 3) >> 2;
    // The list's order of experts: their own, or (by_rows) by rows, the most first, dealt to eight shares back and forth, share
    // behind share.  Cut into eight ranges of as many tiles, the ranges then have about as many rows each, and tall tiles start
    // first.  A wave ranks an expert by counting those before it, 64 at a time.
    for (int e = threadIdx.x; e < E; e += 1024) {
        tiles[e] = (cnt[e] + BM - 1) / BM;
        if (!p.by_rows) pos[e] = e;
    }
    if (p.by_rows) {
        const int lane = threadIdx.x & 63;
        for (int e = threadIdx.x >> 6; e < E; e += 16) {
            const int mine = cnt[e];
            int rank = 0;
            for (int q = lane; q < (E + 63) / 64 * 64; q += 64)  // (counts behind the last expert are zero, and not before any: q > e)
                rank += __popcll(__ballot(cnt[q] > mine || (cnt[q] == mine && q < e)));
            const int turn = rank >> 3, whole = E >> 3, more = E & 7;
            const bool back = turn & 1, last_back = whole & 1;
            const int share = back ? 7 - (rank & 7) : rank & 7;
            const int extra = last_back ? max(share - (8 - more), 0) : min(share, more);  // experts of the last turn in the shares before
            if (lane == 0) pos[e] = share * whole + extra + turn;
        }
    }
    __syncthreads();
    // Thread e lays out expert e: its first slot and first tile are prefix sums over the experts before it, then it writes its
    // own tiles.
    // ceil(cnt / BM) tiles that differ by at most a fragment: 140 rows with BM = 128 become 80 + 60 rather
    // than 128 + 12, and the GEMM skips the row fragments a tile does not have.
    for (int e = threadIdx.x; e < E; e += 1024) {
        int o = 0, nt = 0, total = 0;
        const int at_e = pos[e];
        for (int q = 0; q < E4; ++q) {
            const int4 c = cnt4[q], at = pos4[q], t = tiles4[q];
            auto add = [&](int n, int place, int tq, int i) {
                if (4 * q + i < e) o += n;
                if (place < at_e) nt += tq;
                total += tq;
            };
            add(c.x, at.x, t.x, 0), add(c.y, at.y, t.y, 1), add(c.z, at.z, t.z, 2), add(c.w, at.w, t.w, 3);
        }
        off[e] = o;
        p.offsets[e] = o;
        const int tiles_e = tiles[e];
        const int frags_e = (cnt[e] + p.fragment - 1) / p.fragment;
        const int nt_first = nt, nt_end = nt + tiles_e;
        for (int m0 = 0, i = 0; m0 < cnt[e]; ++i) {
            const int per = (frags_e / tiles_e + (i < frags_e % tiles_e ? 1 : 0)) * p.fragment;
            // tile nt of `total` goes to range x = floor(8 nt / total), behind that range's earlier tiles
            const int x = nt * 8 / total;
            const int x_first = (x * total + 7) / 8, x_end = ((x + 1) * total + 7) / 8;  // the tiles of range x
            const int at = x * p.tiles_per_xcd + nt - x_first;
            const int run_first = max(nt_first, x_first), run_end = min(nt_end, x_end);
            p.tile_expert[at] = e;
            p.tile_row0[at] = o + m0;
            p.tile_rows[at] = min(per, cnt[e] - m0);
            p.tile_run0[at] = at - (nt - run_first);
            p.tile_runlen[at] = run_end - run_first;
            m0 += per;
            ++nt;
        }
        if (e == E - 1) {
            off[E] = o + cnt[e];
            p.offsets[E] = o + cnt[e];
            *p.n_tiles = total;
        }
    }
    __syncthreads();
    // Order inside an expert's range is arbitrary (atomic): every row is computed
    // independently, and slot_of lets the combine step find it again.
    auto place = [&](int r, int e) {
        if (e >= 0 && e < E) {
            const int slot = off[e] + atomicAdd(&cur[e], 1);
            p.slot_src[slot] = r;
            p.slot_of[r] = slot;
        } else {
            p.slot_of[r] = -1;
        }
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
        if (static_cast<int>(threadIdx.x) + i * 1024 < R) place(threadIdx.x + i * 1024, kept[i]);
    for (int r = threadIdx.x + KEEP * 1024; r < R; r += 1024) place(r, sel[r]);
}


// Maximum over the 16 lanes of a DPP row, in every lane of the row (quad swaps, then the two mirrors): register
// moves only, where a shuffle would go through the LDS pipeline.
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true)));
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true)));
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true)));
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true)));
    return v;
}

// f(integral_constant<int, 1>) ... f(integral_constant<int, N-1>), expanded at compile time.
template <class F, int... Is>
__device__ __forceinline__ void static_for_from1_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is + 1>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for_from1(F &&f) {
    static_for_from1_impl(static_cast<F &&>(f), std::make_integer_sequence<int, (N > 1 ? N - 1 : 0)>{});
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>), expanded at compile time.
template <class F, int... Is>
__device__ __forceinline__ void static_for_n_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for_n(F &&f) {
    static_for_n_impl(static_cast<F &&>(f), std::make_integer_sequence<int, N>{});
}

template <int MT, int NT>
struct BSet {
    mu32x4 q[NT];
    uint32_t s[NT];
    bool valid;  // wave-uniform: false for a dead chunk past the padded K
};

// ---------------------------------------------------------------------------
// Workspace carving (256-byte aligned pieces, in this order).
// ---------------------------------------------------------------------------
struct MoeWorkspace {
    MoePlan plan;
    uint8_t *x_hi, *x_lo, *x_sc;  // quantised x, T rows of Kp(H)
    __bf16 *act;                  // [R][I]
    uint8_t *a_hi, *a_lo, *a_sc;  // quantised act, R rows of Kp(I)
    float *out;                   // [R][H]
    size_t total;
};

static inline MoeWorkspace carve(void *base, int64_t T, int64_t H, int64_t I, int64_t E, int64_t topk) {
    MoeWorkspace w{};
    w.plan.fragment = 16;
    const int64_t R = T * topk;
    const int64_t max_tiles = R / 16 + E + 8;  // tiles of at least 16 rows, one partial tile per expert, rounded up to eight
    size_t off = 0;
    auto take = [&](size_t bytes) {
        uint8_t *p = base ? static_cast<uint8_t *>(base) + off : nullptr;
        off += (bytes + 255) & ~size_t{255};
        return p;
    };
    w.plan.offsets = reinterpret_cast<int *>(take((E + 1) * 4));
    w.plan.slot_src = reinterpret_cast<int *>(take(R * 4));
    w.plan.slot_of = reinterpret_cast<int *>(take(R * 4));
    w.plan.tile_expert = reinterpret_cast<int *>(take(max_tiles * 4));
    w.plan.tile_row0 = reinterpret_cast<int *>(take(max_tiles * 4));
    w.plan.tile_rows = reinterpret_cast<int *>(take(max_tiles * 4));
    w.plan.tile_run0 = reinterpret_cast<int *>(take(max_tiles * 4));
    w.plan.tile_runlen = reinterpret_cast<int *>(take(max_tiles * 4));
    w.plan.n_tiles = reinterpret_cast<int *>(take(4));
    const int64_t Hp = pad128(H), Ip = pad128(I);
    w.x_hi = take(T * Hp);
    w.x_lo = take(T * Hp);
    w.x_sc = take(T * (Hp / 32));
    w.act = reinterpret_cast<__bf16 *>(take(R * I * 2));
    w.a_hi = take(R * Ip);
    w.a_lo = take(R * Ip);
    w.a_sc = take(R * (Ip / 32));
    w.out = reinterpret_cast<float *>(take(R * H * 4));
    w.total = off;
    return w;
}

// Routed rows whose down product adds the experts up itself: one token's top-4.
constexpr int kDirectRows = 4;

// mxfp4_moe.hip: y[t][h] = bf16( sum_s wts[t][s] * out[slot_of[t*topk+s]][h] )
lhip_status moe_launch_combine(const float *out, const int *slot_of, const float *wts, __bf16 *y, int T, int H, int topk,
                               hipStream_t s);
// mxfp4_moe_few.hip: whether a layer of so few routed rows goes to its kernels, which expand the weights exactly, in either mode: the
// block-scaled form, whose price is its quantised activations' launch and tiles, was slower there (us, block-scaled / exact, 32
// experts of 2880 x 2880, top 4: T = 1 24.5 / 21.3, T = 4 52 / 41, T = 8 73 / 58, T = 16 82 / 74).
bool moe_few_takes(int T, int H, int I, int E, int topk);
// mxfp4_moe_exact.hip: the layer on the bf16 matrix instruction (weights expanded exactly), and its intermediates.
lhip_status moe_exact_forward(const uint8_t *gu, const uint8_t *dn, const __bf16 *x, const int32_t *sel_dev,
                              const float *wts_dev, __bf16 *y, int T, int H, int I, int E, int topk, MoeWorkspace &w,
                              hipStream_t s);
lhip_status moe_exact_read_intermediates(const MoeWorkspace &w, float *act_dev, float *down_dev, int R, int I, int H,
                                         hipStream_t s);

}  // namespace lhip
