// What the two grouped GEMMs of the exact expert layer share (mxfp4_moe_exact.hip: row tiles of 16 to 64, mxfp4_moe_tall.hip: of
// 96): arguments, the tile a workgroup takes, SwiGLU.
#pragma once

#include "mxfp4_moe_device.h"

namespace lhip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// up * swish(gate) with the hardware exp2 and reciprocal (1 ulp each), as the block-scaled form computes it.
__device__ __forceinline__ float exact_swiglu(float gate, float up) {
    return up * (gate * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504f * gate)));
}

// The 32 codes of one block (four dwords, even k in the low nibble) times 2^(code - 127), as the four weight
// operands of the block's matrix steps.
__device__ __forceinline__ void mx_expand_block(const mu32x4 &q, uint32_t scale_code, v8bf (&w)[4]) {
    const float s = __uint_as_float(scale_code << 23);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const v2bf p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q[d], s, 0);
        const v2bf p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q[d], s, 1);
        const v2bf p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q[d], s, 2);
        const v2bf p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q[d], s, 3);
        w[d] = v8bf{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
}

struct MoeExactArgs {
    const __bf16 *a;      // activation rows, K elements each
    const int *a_index;   // slot -> routed entry (GEMM 1) or nullptr (rows are slots)
    int a_div;            // routed entry / a_div = activation row
    const uint8_t *w_nib, *w_sc;
    int rows_per_expert;
    int K, Kp;
    int N;
    const int *tile_expert, *tile_row0, *tile_rows, *n_tiles;
    const int *tile_run0, *tile_runlen;
    int tiles_per_xcd;
    void *out;            // bf16 [R][N] (gated) or f32 [R][N]
};

// Tile and column block of this workgroup (by MoePlan::tiles_per_xcd).
// Within a run of tiles of one expert the workgroups are ordered column block by column block: the tiles that
// read the same weights are dispatched next to each other and share one fetch of them out of the XCD's L2.
__device__ __forceinline__ void exact_tile(const MoeExactArgs &g, int &tile, int &cb, int &expert, int &row0, int &rows) {
    const int linear = blockIdx.y * gridDim.x + blockIdx.x;
    const int turn = linear >> 3, cols = static_cast<int>(gridDim.x);
    const int base = (linear & 7) * g.tiles_per_xcd;
    const int entry = turn / cols;
    cb = turn - entry * cols;
    tile = base + entry;
    // (the entry's own tile is read in the same trip to memory; only a workgroup inside a run pays a second one,
    // and not for the expert, which the run shares)
    expert = g.tile_expert[tile];
    row0 = g.tile_row0[tile];
    rows = g.tile_rows[tile];
    const int run0 = g.tile_run0[tile], runlen = g.tile_runlen[tile];
    if (runlen > 1) {
        const int local = turn - (run0 - base) * cols;  // position among the run's runlen * cols workgroups
        cb = local / runlen;
        // (Tall tiles first in a run: dealt to 32 compute units in turn, a run of two would give every other one tall tiles only.
        // So the tiles trade places from one 32 to the next: T = 1024 241 -> 235 us.)
        tile = run0 + (local - cb * runlen + ((turn - local + cb * runlen) >> 5)) % runlen;
        row0 = g.tile_row0[tile];
        rows = g.tile_rows[tile];
    }
}

// mxfp4_moe_few.hip: the layer for up to kFewRows routed rows, without a plan; `act`, `out` and `slot_of` as the workspace holds them.
constexpr int kFewRows = 64;
struct MoeFewLayer {
    const uint8_t *gu, *gu_sc, *dn, *dn_sc;
    const __bf16 *x;
    const int *sel;
    const float *wts;
    __bf16 *y, *act;
    float *out;
    int *slot_of;
    int T, H, I, E, topk;
};
lhip_status moe_few_forward(const MoeFewLayer &l, hipStream_t s);

// mxfp4_moe_tall.hip.  Whether its 32-bit offsets reach everywhere for t tokens of width h and experts of width i.
constexpr int kTallRows = 96;
bool moe_tall_supports(int64_t t, int64_t h, int64_t i);
lhip_status moe_tall_gemm(const MoeExactArgs &a, bool gated, int max_tiles, hipStream_t s);

}  // namespace lhip
