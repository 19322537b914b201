// MXFP4 mixture-of-experts layer, exact form: the weights are expanded to bf16 in registers and multiplied on the
// bf16 matrix instruction with f32 accumulation.
//
// Not in the reference (it has neither MXFP4 nor MoE).  Its convention for quantised weights is "dequantise exactly,
// then multiply in f32" (examples/llama/src/loader.rs:227-241) and its expert MLP is luminal's SwiGLU
// down( up(x) * swish(gate(x)) ) (examples/llama/src/model.rs:24-32, src/hl_ops/unary.rs:169-177).  This form keeps
// to that: an e2m1 value times 2^(e8m0 - 127) has at most two significant bits and bf16 has the exponent range of
// f32, so every weight is a bf16 number exactly; the activations are the bf16 numbers the caller passed; products of
// two bf16 numbers are exact in f32, and v_mfma_f32_16x16x32_bf16 adds them at f32 accuracy.  The only roundings of a
// matmul are those of its f32 accumulation (and one to bf16 where the output is bf16).
//
// The expansion is one instruction per two weights: v_cvt_scalef32_pk_bf16_fp4 takes a byte of two e2m1 codes and a
// scale (an f32 whose exponent field is the block's e8m0 code) and returns the two scaled values as a bf16 pair.
//
// Operands.  The planar weights are tiled for a wavefront (common.h: lane (r, g) of a 16-row panel and 128-wide
// chunk holds the 32 codes of block g of row r as four dwords).  Dword d of that piece is codes k = 32g + 8d .. + 7,
// eight bf16 numbers after expansion, which is a lane's share of the weight operand of one 16x16x32 step; the
// hardware's k slot (g, e) of step d therefore stands for k = 32g + 8d + e, and the activation operand of that step
// is x[row][chunk*128 + 32g + 8d .. + 7] for lane (row, g): one 16-byte LDS read.  Four steps cover the chunk.
// In LDS an activation row of a chunk lies in two planes of 128 bytes (steps 0-1, steps 2-3), piece (g, d) at
// byte 16 (g + 4 (d & 1)) of plane d >> 1, which gives the fragment reads the addresses r * pitch + 16 g + 64 (d & 1)
// that were measured free of bank conflicts at a pitch of 160 bytes.
#include "mxfp4_moe_exact_device.h"

namespace lhip {

// LDS byte offset, inside a row's two planes of `plane_bytes` each, of 16-byte piece j (k = 8j .. 8j+7) of a chunk.
__device__ __forceinline__ int exact_piece_offset(int j, int plane_bytes) {
    const int g = j >> 2, d = j & 3;
    return (d >> 1) * plane_bytes + (g + 4 * (d & 1)) * 16;
}

// ---------------------------------------------------------------------------
// Planar MXFP4 -> bf16[N][K] through the expansion the GEMMs use.  One thread per block of 32 weights.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void mx_dequant_bf16_kernel(const uint8_t *__restrict__ nib, const uint8_t *__restrict__ sc,
                                                              __bf16 *__restrict__ out, size_t n_pieces, int n, int k,
                                                              int chunks) {
    const size_t piece = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (piece >= n_pieces) return;
    const size_t tile = piece >> 6;
    const int in_tile = static_cast<int>(piece & 63);
    const size_t panel = tile / chunks;
    const int chunk = static_cast<int>(tile - panel * chunks);
    const size_t row = panel * 16 + (in_tile & 15);
    const int kb = chunk * 4 + (in_tile >> 4);
    if (row >= static_cast<size_t>(n) || kb * 32 >= k) return;
    const mu32x4 q = *reinterpret_cast<const mu32x4 *>(nib + piece * 16);
    v8bf w[4];
    mx_expand_block(q, sc[piece], w);
    v8bf *o = reinterpret_cast<v8bf *>(out + row * k + kb * 32);
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = w[d];
}

// ---------------------------------------------------------------------------
// Grouped expert GEMM.  grid = (column blocks, max tiles); a workgroup of 4 * WR waves owns one row tile (up to
// BM = 16 MT routed rows of one expert) and 4 NT column fragments of 16.  Wave (column group, row group) holds the
// activation fragments of its MT / WR row fragments in registers for a whole chunk and walks its NT weight
// fragments: expand one (16 conversions), multiply it with every row fragment (4 matrix steps each).  So a weight
// is expanded once per row tile whatever the tile's height, and an activation fragment is read from LDS once per
// chunk.  GATED: fragments come in pairs, gate rows and the matching up rows; output bf16 up * swish(gate), else f32.
// ---------------------------------------------------------------------------
template <int MT, int NT, bool GATED, int WR, int D>
__global__ __launch_bounds__(256 * WR) void mx_moe_gemm_exact_kernel(MoeExactArgs g) {
    static_assert(!GATED || NT % 2 == 0, "gated tiles pair each gate fragment with its up fragment");
    static_assert(MT % WR == 0 && D % 2 == 0 && NT >= 2, "tile shape");
    constexpr int BM = 16 * MT;
    constexpr int MTW = MT / WR;  // row fragments per wave
    constexpr int THREADS = 256 * WR;
    constexpr int STG = MT / WR;  // 16-byte pieces of the activation tile staged per thread and chunk
    constexpr int A_PLANE = BM * kARow;
    constexpr int A_BUF = 2 * A_PLANE;

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // 3 x A_BUF

    int tile, cb, expert, row0, rows;
    exact_tile(g, tile, cb, expert, row0, rows);
    if (rows == 0) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_id & 3;
    const int wrow = WR == 1 ? 0 : wave_id >> 2;
    const int r = lane & 15, grp = lane >> 4;
    const int K = g.K, Kp = g.Kp;
    const int chunks = Kp / kChunk;
    const int steps = (chunks + D - 1) / D * D;
    const int frags = (rows + 15) >> 4;

    // ---- weight fragments: one contiguous KiB of codes and 64 scale bytes per fragment and chunk
    const uint8_t *w_tile[NT];
    const uint8_t *s_tile[NT];
    int col[NT];
#pragma unroll
    for (int f = 0; f < NT; ++f) {
        int n0, wrow0;
        if (GATED) {
            n0 = ((cb * 4 + wave) * (NT / 2) + (f >> 1)) * 16;
            wrow0 = ((f & 1) ? g.N : 0) + min(n0, g.N - 16);
        } else {
            n0 = ((cb * 4 + wave) * NT + f) * 16;
            wrow0 = min(n0, g.N - 16);
        }
        col[f] = n0 + r;
        const size_t panel = (static_cast<size_t>(expert) * g.rows_per_expert + wrow0) >> 4;
        w_tile[f] = g.w_nib + (panel * chunks * 64 + lane) * 16;
        s_tile[f] = g.w_sc + panel * chunks * 64 + lane;
    }
    BSet<MT, NT> bs[D];
    auto load_b = [&](int set, int c) __attribute__((always_inline)) {
        bs[set].valid = c < chunks;  // dead chunks (past the padded K; the refills of the last round) are not multiplied
        const int cc = min(c, chunks - 1);
#pragma unroll
        for (int f = 0; f < NT; ++f) {
            if (MT <= 2) {  // short tiles read every weight once: keep them out of the caches
                // (a dead chunk's request goes to one line for the whole wave: aimed at the last chunk it would pull
                // that kilobyte through the memory system again, D + 1 times per wave and fragment)
                const uint8_t *wq = c < chunks ? w_tile[f] + static_cast<size_t>(cc) * 1024 : g.w_nib;
                bs[set].q[f] = __builtin_nontemporal_load(reinterpret_cast<const mu32x4 *>(wq));
                bs[set].s[f] = s_tile[f][cc * 64];  // (cached: the 64 scale bytes of two consecutive chunks share a line)
            } else {
                bs[set].q[f] = *reinterpret_cast<const mu32x4 *>(w_tile[f] + static_cast<size_t>(cc) * 1024);
                bs[set].s[f] = s_tile[f][cc * 64];
            }
        }
    };

    // ---- activation tile: global (bf16 rows) -> registers -> LDS (three buffers), shared by all waves.
    // Threads take the tile's pieces in source order (16 consecutive threads = the 256 bytes of one row).
    const uint8_t *a_src[STG];
    int a_k[STG], a_dst[STG];
#pragma unroll
    for (int i = 0; i < STG; ++i) {
        const int q = tid + i * THREADS;
        const int row = q >> 4, j = q & 15;
        const int slot = row0 + min(row, rows - 1);  // rows past the tile re-read its last row (their results are not stored)
        const int arow = g.a_index ? g.a_index[slot] / g.a_div : slot;
        a_src[i] = reinterpret_cast<const uint8_t *>(g.a + static_cast<size_t>(arow) * K) + j * 16;
        a_k[i] = j * 8;
        a_dst[i] = row * kARow + exact_piece_offset(j, A_PLANE);
    }
    struct AStage {
        mu32x4 q[STG];
    };
    auto load_a = [&](AStage &st, int c) __attribute__((always_inline)) {
        const int cc = min(c, chunks - 1);
#pragma unroll
        for (int i = 0; i < STG; ++i) {
            // Pieces past K (the last chunk of a K that is no multiple of 128) are zeros: the padding weights are zero
            // too, but zero times whatever lies behind the row need not be.
            const bool in = cc * kChunk + a_k[i] < K;
            const uint8_t *p = in ? a_src[i] + cc * (kChunk * 2) : reinterpret_cast<const uint8_t *>(g.a);
            const mu32x4 v = *reinterpret_cast<const mu32x4 *>(p);
            const mu32x4 zero = {0, 0, 0, 0};
            st.q[i] = in ? v : zero;
        }
    };
    auto store_a = [&](AStage &st, unsigned char *base) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < STG; ++i) {
            asm volatile("" : "+v"(st.q[i]));
            *reinterpret_cast<mu32x4 *>(base + a_dst[i]) = st.q[i];
        }
    };

    v4f acc[MTW][NT];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int f = 0; f < NT; ++f) acc[i][f] = v4f{0.f, 0.f, 0.f, 0.f};

    // Row fragment n of this wave's row group is tile fragment n * WR + wrow.
    const int frag_lane = (wrow * 16 + r) * kARow + grp * 16;
    v8bf afr[MTW][4];
    auto load_frag = [&](const unsigned char *base, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        const unsigned char *p = base + frag_lane + i * (WR * 16 * kARow);
        afr[i][0] = *reinterpret_cast<const v8bf *>(p);
        afr[i][1] = *reinterpret_cast<const v8bf *>(p + 64);
        afr[i][2] = *reinterpret_cast<const v8bf *>(p + A_PLANE);
        afr[i][3] = *reinterpret_cast<const v8bf *>(p + A_PLANE + 64);
    };
    auto mfma_frag = [&](const v8bf (&wb)[4], auto ic, auto fc) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        constexpr int f = decltype(fc)::value;
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afr[i][d], wb[d], acc[i][f], 0, 0, 0);
        // Pin the accumulation here: nothing else reads acc until the epilogue, and without this the optimiser
        // sinks the matrix steps of the unrolled pipeline to its end and keeps every operand alive.
        asm volatile("" : "+a"(acc[i][f]));
    };

    // ---- pipeline: three LDS buffers, one barrier per chunk.  Chunk c multiplies out of buffer c % 3 (its
    // fragments are already in registers).  After the first weight fragment every wave passes the barrier and then
    // writes chunk c+2 (requested during chunk c-1) into buffer (c+2) % 3, which was last read when the fragments of
    // chunk c-1 were fetched; chunk c+1's buffer is complete behind that barrier, so its fragments are fetched into
    // the registers of each row fragment as soon as the chunk's last weight fragment has used them.
    // The prologue issues its loads in the loop's order (see mx_moe_gemm_kernel).
    AStage stage, stage2;
#pragma unroll
    for (int j = 0; j + 1 < D; ++j) load_b(j, j);
    load_a(stage, 0);
    load_a(stage2, 1);
    store_a(stage, lds);
    store_a(stage2, lds + A_BUF);
    load_a(stage, 2);
    load_b(D - 1, D - 1);
    __syncthreads();
    unsigned char *cur = lds, *nxt = lds + A_BUF, *fill = lds + 2 * A_BUF;
    static_for_n<MTW>([&](auto ic) __attribute__((always_inline)) { load_frag(cur, ic); });
    for (int c0 = 0; c0 < steps; c0 += D) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const int c = c0 + j;
            const bool live = bs[j].valid;
#pragma unroll
            for (int f = 0; f < NT; ++f) asm volatile("" : "+v"(bs[j].q[f]), "+v"(bs[j].s[f]));
            static_for_n<NT>([&](auto fc) __attribute__((always_inline)) {
                constexpr int f = decltype(fc)::value;
                v8bf wb[4];
                mx_expand_block(bs[j].q[f], bs[j].s[f], wb);
                static_for_n<MTW>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    if (live && i * WR + wrow < frags) mfma_frag(wb, ic, fc);  // wave-uniform
                    if (f == NT - 1) load_frag(nxt, ic);
                });
                if (f == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    __syncthreads();
                    store_a(stage, fill);
                    load_a(stage, c + 3);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            load_b(j, c + D);  // refill the set just consumed
            unsigned char *t = cur;
            cur = nxt;
            nxt = fill;
            fill = t;
        }
    }

    // ---- epilogue: acc[i][f][v] is row (i * WR + wrow) * 16 + 4 * grp + v, column fragment f, column r
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = (i * WR + wrow) * 16 + 4 * grp + v;
            if (m >= rows) continue;
            const size_t orow = static_cast<size_t>(row0 + m) * g.N;
            if (GATED) {
#pragma unroll
                for (int p = 0; p < NT / 2; ++p)
                    if (col[2 * p] < g.N)
                        static_cast<__bf16 *>(g.out)[orow + col[2 * p]] =
                            static_cast<__bf16>(exact_swiglu(acc[i][2 * p][v], acc[i][2 * p + 1][v]));
            } else {
#pragma unroll
                for (int f = 0; f < NT; ++f)
                    if (col[f] < g.N) static_cast<float *>(g.out)[orow + col[f]] = acc[i][f][v];
            }
        }
}

__global__ __launch_bounds__(1024) void moe_plan_kernel(const int *__restrict__ sel, int R, int E, int BM, MoePlan p) {
    moe_plan_block(sel, R, E, BM, p);
}

// act[r][k] = the bf16 activation the down GEMM consumed, down[r][h] = its f32 row, per routed entry.
__global__ __launch_bounds__(256) void moe_read_intermediates_exact_kernel(const int *__restrict__ slot_of,
                                                                           const __bf16 *__restrict__ a,
                                                                           const float *__restrict__ out,
                                                                           float *__restrict__ act, float *__restrict__ down,
                                                                           int R, int I, int H) {
    const int r = blockIdx.x;
    if (r >= R) return;
    const int slot = slot_of[r];
    if (act)
        for (int k = threadIdx.x; k < I; k += 256)
            act[static_cast<size_t>(r) * I + k] = slot >= 0 ? static_cast<float>(a[static_cast<size_t>(slot) * I + k]) : 0.f;
    if (down)
        for (int h = threadIdx.x; h < H; h += 256)
            down[static_cast<size_t>(r) * H + h] = slot >= 0 ? out[static_cast<size_t>(slot) * H + h] : 0.f;
}

template <int MT, int NT, bool GATED, int WR, int D>
static lhip_status launch_exact_gemm(const MoeExactArgs &a, int col_blocks, int max_tiles, hipStream_t s) {
    constexpr int BM = 16 * MT;
    const size_t lds_bytes = 3 * (2 * static_cast<size_t>(BM) * kARow);
    auto kern = mx_moe_gemm_exact_kernel<MT, NT, GATED, WR, D>;
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), lds_bytes)) return st;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(col_blocks), static_cast<unsigned>(max_tiles)), dim3(256 * WR),
                       lds_bytes, s, a);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

// Tile height of the exact form for R routed rows over E experts of H x I, in 16-row fragments: 16 or 32 rows where such a tile holds
// an expert with two standard deviations more rows than the average (so that nearly every expert is one tile and its weights are
// read and expanded once), else 64, or 96 (`tall`, mxfp4_moe_tall.hip), cut into equal parts for experts with more.
// A stage of the 96-row kernel takes longer when its workgroup is alone on a compute unit, and two of its workgroups end no
// sooner than two of 64 rows; it wins with the third.  So it is taken with two workgroups a compute unit in the first product and one
// and a half in the second, and there where its tiles are fewer (more than 46 rows an expert: some, then many are two tiles of 64) or
// hold one fragment of 32 (less than 30).  Measured on 16 layers (4 to 128 experts, H of 1024 to 4096, I of 512 to 14336) at 24 to
// 384 rows an expert: over 64 rows everywhere 0.974, the better of both 0.967, 96 rows everywhere 1.046.  us, 64 / 96 rows: 32 experts of
// 2880 x 2880, top 4, T = 192 115 / 106, T = 256 120 / 116, T = 384 142 / 142, T = 512 180 / 147, T = 1024 263 / 224; 8 experts of 4096 x
// 14336, top 2, T = 128 222 / 299, T = 384 329 / 445; 64 of 2048 x 1408, top 6, T = 512 99 / 97, T = 683 135 / 111; 12 of 2880 x 2880, top 3,
// T = 192 79 / 85.  16- / 32- / 64-row tiles of the first: T = 32 87 / 94 / 110, T = 64 90 / 95 / 110, T = 128 132 / 99 / 114.
static inline int exact_tile_fragments(int R, int E, int H, int I, bool tall) {
    const int avg = (R + E - 1) / E;
    const int need = avg + 2 * static_cast<int>(sqrtf(static_cast<float>(avg)) + 0.5f);
    if (need <= 32) return need <= 16 ? 1 : 2;
    const int64_t tiles = R / kTallRows + E / 2 > E ? R / kTallRows + E / 2 : E;  // about as many as there will be
    const bool filled = tiles * ((I + 127) / 128) >= 2 * 256 && tiles * ((H + 255) / 256) * 2 >= 3 * 256;
    return tall && filled && (avg < 30 || avg > 46) ? kTallRows / 16 : 4;
}

lhip_status moe_exact_forward(const uint8_t *gu, const uint8_t *dn, const __bf16 *x, const int32_t *sel_dev,
                              const float *wts_dev, __bf16 *y, int T, int H, int I, int E, int topk, MoeWorkspace &w,
                              hipStream_t s) {
    const int R = T * topk;
    const int Hp = static_cast<int>(pad128(H)), Ip = static_cast<int>(pad128(I));
    const uint8_t *gu_sc = gu + mx_scale_offset(static_cast<int64_t>(E) * 2 * I, H);
    const uint8_t *dn_sc = dn + mx_scale_offset(static_cast<int64_t>(E) * H, I);

    if (moe_few_takes(T, H, I, E, topk))
        return moe_few_forward(MoeFewLayer{gu, gu_sc, dn, dn_sc, x, sel_dev, wts_dev, y, w.act, w.out, w.plan.slot_of, T, H, I, E, topk}, s);

    const int mt = exact_tile_fragments(R, E, H, I, moe_tall_supports(T, H, I));
    const int BM = 16 * mt;
    const int max_tiles = (R / BM + E + 7) / 8 * 8;
    w.plan.max_tiles = max_tiles;
    w.plan.tiles_per_xcd = max_tiles / 8;
    // Experts listed by their rows, so that the XCDs have about as many: over own order, where these tiles are taken and an expert has more
    // than 50 rows on average, 0.986 (32 experts of 2880 x 2880), 0.989 (64 of 2048 x 1024, 48 of 4096 x 1024), 0.996 to 1.003 (16 of 4096 x
    // 4096, 64 and 60 of 2048 x 1408, 128 of 2048 x 768); at 24 and 28 rows 0.885 to 1.02.
    w.plan.by_rows = BM == kTallRows;
    w.plan.fragment = BM == kTallRows ? 32 : 16;
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), 0, s, sel_dev, R, E, BM, w.plan);
    LHIP_CHECK_LAUNCH();

    MoeExactArgs a1{};
    a1.a = x; a1.a_index = w.plan.slot_src; a1.a_div = topk;
    a1.w_nib = gu; a1.w_sc = gu_sc;
    a1.rows_per_expert = 2 * I; a1.K = H; a1.Kp = Hp; a1.N = I;
    a1.tile_expert = w.plan.tile_expert; a1.tile_row0 = w.plan.tile_row0; a1.tile_rows = w.plan.tile_rows;
    a1.n_tiles = w.plan.n_tiles; a1.tiles_per_xcd = w.plan.tiles_per_xcd; a1.out = w.act;
    a1.tile_run0 = w.plan.tile_run0; a1.tile_runlen = w.plan.tile_runlen;
    const int cb1 = (I + 127) / 128;  // 4 waves x two (gate, up) pairs of 16 columns
    lhip_status st;
    switch (mt) {
        case 1: st = launch_exact_gemm<1, 4, true, 1, 4>(a1, cb1, max_tiles, s); break;
        case 2: st = launch_exact_gemm<2, 4, true, 1, 4>(a1, cb1, max_tiles, s); break;
        case 4: st = launch_exact_gemm<4, 4, true, 1, 2>(a1, cb1, max_tiles, s); break;
        default: st = moe_tall_gemm(a1, true, max_tiles, s); break;
    }
    if (st) return st;
    MoeExactArgs a2{};
    a2.a = w.act; a2.a_index = nullptr; a2.a_div = 1;
    a2.w_nib = dn; a2.w_sc = dn_sc;
    a2.rows_per_expert = H; a2.K = I; a2.Kp = Ip; a2.N = H;
    a2.tile_expert = w.plan.tile_expert; a2.tile_row0 = w.plan.tile_row0; a2.tile_rows = w.plan.tile_rows;
    a2.n_tiles = w.plan.n_tiles; a2.tiles_per_xcd = w.plan.tiles_per_xcd; a2.out = w.out;
    a2.tile_run0 = w.plan.tile_run0; a2.tile_runlen = w.plan.tile_runlen;
    const int cb2 = (H + 127) / 128, cb2w = (H + 255) / 256;
    switch (mt) {
        case 1: st = launch_exact_gemm<1, 2, false, 1, 4>(a2, cb2, max_tiles, s); break;
        case 2: st = launch_exact_gemm<2, 2, false, 1, 4>(a2, cb2, max_tiles, s); break;
        case 4: st = launch_exact_gemm<4, 4, false, 1, 2>(a2, cb2w, max_tiles, s); break;
        default: st = moe_tall_gemm(a2, false, max_tiles, s); break;
    }
    if (st) return st;
    return moe_launch_combine(w.out, w.plan.slot_of, wts_dev, y, T, H, topk, s);
}

lhip_status moe_exact_read_intermediates(const MoeWorkspace &w, float *act_dev, float *down_dev, int R, int I, int H,
                                         hipStream_t s) {
    hipLaunchKernelGGL(moe_read_intermediates_exact_kernel, dim3(static_cast<unsigned>(R)), dim3(256), 0, s,
                       w.plan.slot_of, w.act, w.out, act_dev, down_dev, R, I, H);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

}  // namespace lhip

using namespace lhip;

extern "C" {

lhip_status lhip_mxfp4_dequant_bf16(const void *planar_dev, void *out_bf16_dev, int64_t n, int64_t k, void *stream) {
    if (!planar_dev || !out_bf16_dev) return LHIP_ERR_NULL_PTR;
    if (lhip_status s = check_q8_shape(n, k)) return s;
    if (!aligned(planar_dev, 256) || !aligned(out_bf16_dev, 16)) return LHIP_ERR_MISALIGNED;
    auto *base = static_cast<const uint8_t *>(planar_dev);
    const size_t n_pieces = mx_scale_offset(n, k) / 16;
    hipLaunchKernelGGL(mx_dequant_bf16_kernel, dim3(static_cast<unsigned>((n_pieces + 255) / 256)), dim3(256), 0,
                       as_stream(stream), base, base + mx_scale_offset(n, k), static_cast<__bf16 *>(out_bf16_dev), n_pieces,
                       static_cast<int>(n), static_cast<int>(k), static_cast<int>(mx_chunks(k)));
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

}  // extern "C"
