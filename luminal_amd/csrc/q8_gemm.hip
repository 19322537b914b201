// Q8_0 GEMM for prefill:  Y[M][N] = X[M][K] . W[N][K]^T, bf16 activations,
// f32 accumulation on the matrix cores, bf16 (or f32, or SwiGLU) output: the choice of the kernel per shape, and the
// tile kernel for small products.
//
// The reference has no such kernel on CUDA (its QuantizedMatmul re-runs the
// matvec once per activation row, crates/luminal_cuda/src/quantized.rs:146-164);
// the design precedent is the Metal backend's GEMM, which dequantises a weight
// tile into threadgroup memory and feeds the matrix unit
// (crates/luminal_metal/src/quantized.rs:54-61,63-199).  That kernel rounds
// q * d to the activation type first; these keep the weights exact: the int8
// codes go to the matrix cores as they are (exact in bf16) and the block's scale
// multiplies the f32 sum of the block's products.  Four kernels share the shapes:
//   * few rows, 128 at most: q8_gemm_skinny.hip, bound by streaming the weights;
//   * some dozens to hundreds of rows, or an odd N, and so few tiles that K would have to be sliced: q8_gemm_deep.hip;
//   * more rows: q8_gemm_wide.hip, tiles of 256x256 and 128x256, over slices of K
//     where those are few;
//   * more rows but too few such tiles and a K too short to slice: the kernel in
//     this file, tiles of 128x128 down to 64x64 by four waves.
// The kernel in this file walks K in steps of 64 (two Q8_0 blocks); activations go
// global -> registers -> LDS as bf16, codes global -> registers -> bf16 (one
// sign-extending byte conversion and a pack) -> LDS, the two block scales of the K
// tile to LDS as f32; LDS is double-buffered and the global loads run D tiles ahead
// in rotating register sets; a block is two chained v_mfma_f32_32x32x16_bf16 into a
// zeroed accumulator; LDS rows are padded by 16 bytes so the 16-byte operand reads
// of 8 consecutive lanes hit all banks once.
// With bf16 activations every product is exact, so the only roundings are those
// of the f32 additions (and the one of the bf16 store).  Rounding q * d to bf16
// instead leaves a relative error of 2^-9 per weight, proportional to the sum
// of |w x| and therefore large on every output that cancels: measured 3.5 to
// 5.1 under max |y - t| / max(|t|, 1e-3 rms(t)) on the Llama-3-8B shapes, where
// these kernels score 3.9e-3 (the bf16 store alone) and 1e-4 to 5e-4 on the f32 output.
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "q8_gemm_deep.h"
#include "q8_gemm_rows.h"
#include "q8_gemm_wide.h"
#include "q8_mma_device.h"

namespace lhip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t gu32x4 __attribute__((ext_vector_type(4)));

// x of lane ^ X, X = 1 or 2, within the vector pipe (a shuffle goes through LDS).
template <int X>
__device__ __forceinline__ float lane_xor(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), X == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true));
}

constexpr int kBK = 64;             // K per tile: two Q8_0 blocks
constexpr int kRowBytes = 144;      // 64 bf16 + 16 bytes of padding

// Tile BM x BN by WM x WN waves of at most 64 x 64 each (M tiles in groups of m_group per XCD, as in q8_gemm_wide.hip).
// LDS per buffer: activations BM x 64 bf16, codes BN x 64 as bf16 (rows of 144 bytes), and the BN x 2 block scales of the
// K tile as f32.  The lane that owns column n of a 32 x 32 accumulator tile needs one scale per block: it reads both
// scales of the K tile with one 8-byte LDS read.  The per-block fma costs one v_fma per output element and block on the
// vector ALU, the same number of cycles the block's two MFMAs take on the matrix pipe.
// D = register prefetch depth in K tiles (D > 1 needs K % (64*D) == 0 and D even).
// OutT = __bf16 (rounded to nearest even) or float (the accumulators as they are).
template <int BM, int BN, int WM, int WN, int D, typename OutT>
__global__ __launch_bounds__(WM *WN * 64) void q8_gemm_bf16_kernel(const int8_t *__restrict__ qs,
                                                                 const __half *__restrict__ ds,
                                                                 const __bf16 *__restrict__ x, OutT *__restrict__ y,
                                                                 int M, int N, int K, int m_tiles, int n_tiles,
                                                                 int swiglu, int m_group) {
    constexpr int T = WM * WN * 64;
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int FM = TM / 32, FN = TN / 32;  // 32x32 accumulator tiles per wave
    static_assert(FM >= 1 && FN >= 1 && FM <= 2 && FN <= 2, "wave tiles of at most 64 x 64");
    constexpr int A_CHUNKS = BM * 8 / T;
    constexpr int B_CHUNKS = BN * 4 / T;
    static_assert(A_CHUNKS >= 1 && B_CHUNKS >= 1 && BM * 8 % T == 0 && BN * 4 % T == 0, "tile/thread mismatch");
    constexpr int A_BYTES = BM * kRowBytes, B_BYTES = BN * kRowBytes, S_BYTES = BN * 8;
    constexpr int BUF = A_BYTES + B_BYTES + S_BYTES;

    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // 2 x (A tile, B tile, scales)

    int mt, nt;
    {
        // Workgroups are dealt to the eight XCDs in turn (id modulo 8) and an XCD runs its slots in order, 32 at a
        // time.  The XCD owns the N tiles xcd, xcd + 8, ...; its slots walk the M tiles in groups of m_group: within
        // a group N tile by N tile, the group's M tiles innermost.  The 32 workgroups in flight on an XCD are then
        // m_group M tiles x 32 / m_group N tiles: each of their weight tiles is fetched once and shared by m_group
        // workgroups out of the XCD's L2, each activation tile by 32 / m_group.
        const int id = blockIdx.x;
        const int xcd = id & 7, slot = id >> 3;
        const int npx = (n_tiles + 7) >> 3;                      // N tiles per XCD (the grid is padded to whole eights)
        const int full = m_tiles / m_group;                      // whole groups of M tiles
        const int in_full = full * m_group * npx;
        const int g0 = slot < in_full ? slot / (m_group * npx) : full;
        const int cur = slot < in_full ? m_group : m_tiles - full * m_group;
        const int rem = slot - g0 * m_group * npx;
        const int n_idx = rem / cur;
        mt = g0 * m_group + (rem - n_idx * cur);
        nt = n_idx * 8 + xcd;
        if (nt >= n_tiles) return;
    }
    const int m0 = mt * BM, n0 = nt * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int nblk = K >> 5;
    const int KT = K / kBK;

    const __bf16 *a_src[A_CHUNKS];
    int a_dst[A_CHUNKS];
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
        const int c = tid + i * T;
        const int row = c >> 3, col = (c & 7) * 8;
        a_src[i] = x + static_cast<size_t>(min(m0 + row, M - 1)) * K + col;
        a_dst[i] = row * kRowBytes + col * 2;
    }
    const int8_t *b_src[B_CHUNKS];
    const uint32_t *d_src[B_CHUNKS];  // the two scales of a K tile are one aligned dword (K/32 is even)
    int b_dst[B_CHUNKS];
    int s_dst[B_CHUNKS];              // where this thread leaves the row's scales, or -1: one thread in four does
#pragma unroll
    for (int i = 0; i < B_CHUNKS; ++i) {
        const int c = tid + i * T;
        const int row = c >> 2, q16 = c & 3;
        const int grow = min(n0 + row, N - 1);
        b_src[i] = qs + static_cast<size_t>(grow) * K + q16 * 16;
        d_src[i] = reinterpret_cast<const uint32_t *>(ds + static_cast<size_t>(grow) * nblk);
        b_dst[i] = row * kRowBytes + q16 * 32;
        s_dst[i] = q16 == 0 ? row * 8 : -1;
    }

    gu32x4 a_reg[D][A_CHUNKS], b_reg[D][B_CHUNKS];
    uint32_t d_reg[D][B_CHUNKS];
    auto load_tile = [&](int set, int kt, int p = 0, int P = 1) {
        const int k0 = min(kt, KT - 1) * kBK;  // tiles past the end re-read the last one (never used)
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i)
            if (i * P / A_CHUNKS == p) a_reg[set][i] = *reinterpret_cast<const gu32x4 *>(a_src[i] + k0);
#pragma unroll
        for (int i = 0; i < B_CHUNKS; ++i) {
            if (i * P / B_CHUNKS != p) continue;
            b_reg[set][i] = *reinterpret_cast<const gu32x4 *>(b_src[i] + k0);
            d_reg[set][i] = d_src[i][k0 >> 6];
        }
    };
    // two int8 of a dword (bytes 2h, 2h+1) -> two bf16, exactly: the sign-extending byte conversion gives an f32
    // whose upper half is the bf16 code
    auto store_tile = [&](int set, int buf, int p = 0, int P = 1) {
        unsigned char *A = lds + buf * BUF;
        unsigned char *B = A + A_BYTES;
        unsigned char *S = B + B_BYTES;
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i)
            if (i * P / A_CHUNKS == p) *reinterpret_cast<gu32x4 *>(A + a_dst[i]) = a_reg[set][i];
#pragma unroll
        for (int u = 0; u < 2 * B_CHUNKS; ++u) {
            if (u * P / (2 * B_CHUNKS) != p) continue;
            const int i = u >> 1;
            // Opaque to the optimiser: keeps the unpacking of this set here, at its use, instead of next to its loads
            asm volatile("" : "+v"(b_reg[set][i]), "+v"(d_reg[set][i]));
            if ((u & 1) == 0) {
                const gu32x4 lo = {codes2<false>(b_reg[set][i].x, 0), codes2<false>(b_reg[set][i].x, 1), codes2<false>(b_reg[set][i].y, 0),
                                   codes2<false>(b_reg[set][i].y, 1)};
                *reinterpret_cast<gu32x4 *>(B + b_dst[i]) = lo;
                if (s_dst[i] >= 0) {
                    const float d0 = __half2float(__ushort_as_half(static_cast<unsigned short>(d_reg[set][i] & 0xffffu)));
                    const float d1 = __half2float(__ushort_as_half(static_cast<unsigned short>(d_reg[set][i] >> 16)));
                    *reinterpret_cast<float2 *>(S + s_dst[i]) = make_float2(d0, d1);
                }
            } else {
                const gu32x4 hi = {codes2<false>(b_reg[set][i].z, 0), codes2<false>(b_reg[set][i].z, 1), codes2<false>(b_reg[set][i].w, 0),
                                   codes2<false>(b_reg[set][i].w, 1)};
                *reinterpret_cast<gu32x4 *>(B + b_dst[i] + 16) = hi;
            }
        }
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    const int frag_off = (lane & 31) * kRowBytes + (lane >> 5) * 16;
    // One K tile: two blocks of FM x FN slots; a slot is the two chained MFMAs of one accumulator tile's block sum.
    // The scheduler, left alone, issues every MFMA of the K tile first and every fma after (eight block sums live:
    // spills), so the order is fixed with scheduling fences: the sixteen fmas of the previous slot's block sum are
    // issued in two halves behind the two MFMAs of this slot and run on the vector ALU while the matrix pipe
    // works; the last slot's sum of a K tile is carried into the next tile (`pend`, zero before the first).  With STAGE the
    // dequantise-and-store of the next tile and the global loads of the tile after that are dealt out over the
    // slots.  The operand fragments of block 1 are requested during block 0 as their registers fall free (row i's
    // A fragments after its last column, column j's B fragments after its last row).
    f32x16 pend = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // block sum whose fmas are still to be issued
    float pend_d = 0.f;                                                                              // and its scale
    // Opaque to the optimiser, or it peels the first K tile off the loop (its fmas fold away) and schedules that
    // copy with all eight block sums live.
    asm volatile("" : "+v"(pend), "+v"(pend_d));
    auto k_tile = [&](int buf, bool stage, int set, int next_buf, int load_set, int load_kt) {
        const unsigned char *A = lds + buf * BUF + (wm * TM) * kRowBytes + frag_off;
        const unsigned char *B = lds + buf * BUF + A_BYTES + (wn * TN) * kRowBytes + frag_off;
        const unsigned char *S = lds + buf * BUF + A_BYTES + B_BYTES + (wn * TN + (lane & 31)) * 8;
        bf16x8 af[2][2][FM], bfr[2][2][FN];  // [block][k step][tile]
        auto load_a = [&](int b, int i) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                af[b][s][i] = *reinterpret_cast<const bf16x8 *>(A + i * 32 * kRowBytes + (2 * b + s) * 32);
        };
        auto load_b = [&](int b, int j) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
                bfr[b][s][j] = *reinterpret_cast<const bf16x8 *>(B + j * 32 * kRowBytes + (2 * b + s) * 32);
        };
        float2 sc[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) sc[j] = *reinterpret_cast<const float2 *>(S + j * 32 * 8);
#pragma unroll
        for (int i = 0; i < FM; ++i) load_a(0, i);
#pragma unroll
        for (int j = 0; j < FN; ++j) load_b(0, j);
        static_for<2 * FM * FN>([&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            constexpr int b = q / (FM * FN), r = q % (FM * FN), i = r / FN, j = r % FN;
            constexpr int rp = (r + FM * FN - 1) % (FM * FN), ip = rp / FN, jp = rp % FN;  // the slot before this one
            if (stage) {
                store_tile(set, next_buf, q, 2 * FM * FN);
                load_tile(load_set, load_kt, q, 2 * FM * FN);
            }
            __builtin_amdgcn_sched_barrier(0);
            f32x16 sum = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[b][0][i], bfr[b][0][j], sum, 0, 0, 0);
            // (the empty asm statements tie each result to its place between the fences: the fences hold the machine
            // scheduler, but arithmetic without side effects is moved past them before it ever gets there)
            asm volatile("" : "+v"(sum));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 8; ++v) acc[ip][jp][v] = fmaf(pend_d, pend[v], acc[ip][jp][v]);
            asm volatile("" : "+v"(acc[ip][jp]));
            __builtin_amdgcn_sched_barrier(0);
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[b][1][i], bfr[b][1][j], sum, 0, 0, 0);
            asm volatile("" : "+v"(sum));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 8; v < 16; ++v) acc[ip][jp][v] = fmaf(pend_d, pend[v], acc[ip][jp][v]);
            asm volatile("" : "+v"(acc[ip][jp]));
            if constexpr (b == 0) {  // this slot's MFMAs are issued: block 1's fragments into the registers that fell free
                if constexpr (j == FN - 1) load_a(1, i);
                if constexpr (i == FM - 1) load_b(1, j);
            }
            __builtin_amdgcn_sched_barrier(0);
            pend = sum;
            pend_d = b ? sc[j].y : sc[j].x;
        });
    };

#pragma unroll
    for (int j = 0; j < D; ++j) load_tile(j, j);
    store_tile(0, 0);
    __syncthreads();

    if constexpr (D == 1) {
        for (int kt = 0; kt < KT; ++kt) {
            load_tile(0, kt + 1);
            k_tile(kt & 1, false, 0, 0, 0, 0);
            store_tile(0, (kt + 1) & 1);
            __syncthreads();
        }
    } else {
        static_assert(D % 2 == 0, "LDS buffer parity must follow the register set");
        for (int kt = 0; kt < KT; kt += D) {
#pragma unroll
            for (int j = 0; j < D; ++j) {
                // set j held tile kt+j, already in LDS: refill it with tile kt+j+D
                k_tile(j & 1, true, (j + 1) % D, (j + 1) & 1, j, kt + j + D);
                __syncthreads();
            }
        }
    }

#pragma unroll
    for (int v = 0; v < 16; ++v) acc[FM - 1][FN - 1][v] = fmaf(pend_d, pend[v], acc[FM - 1][FN - 1][v]);

    // Epilogue: acc element v of lane l is row 8*(v/4) + 4*(l/32) + v%4, column l%32 of its 32x32 tile.
    if constexpr (sizeof(OutT) == 2) {
        if (swiglu) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int col = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int row = m0 + wm * TM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                        const float mine = acc[i][j][v], other = lane_xor<1>(mine);
                        const float act = (lane & 1) ? swiglu_value(other, mine) : swiglu_value(mine, other);
                        const float act2 = lane_xor<2>(act);
                        if ((lane & 3) == 0 && row < M && col < N) {
                            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                            const bf16x2 pk = {static_cast<__bf16>(act), static_cast<__bf16>(act2)};
                            *reinterpret_cast<bf16x2 *>(reinterpret_cast<__bf16 *>(y) +
                                                        static_cast<size_t>(row) * (N >> 1) + (col >> 1)) = pk;
                        }
                    }
                }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int col = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm * TM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row < M && col < N) y[static_cast<size_t>(row) * N + col] = static_cast<OutT>(acc[i][j][v]);
            }
        }
}

// What the epilogue writes: bf16 (m, N), f32 (m, N), or bf16 (m, N/2) = up * swish(gate) of (gate, up) column pairs.
enum { kOutBf16 = 0, kOutF32 = 1, kOutSwiglu = 2 };

// q8_gemm_skinny.hip: the weight-streaming kernel for at most 128 activation rows.
bool q8_gemm_skinny_supports(int m, int n, int k, int out, const void *y);
int q8_gemm_skinny_splits(int m, int n, int k, size_t room);
double q8_gemm_skinny_us(int m, int n, int k, size_t room);
lhip_status q8_gemm_skinny_launch(const int8_t *qs, const __half *ds, const void *x_bf16, void *y, int m, int n, int k,
                                  int out, int splits, hipStream_t s, bool own_workspace = false, float *ws = nullptr,
                                  size_t ws_floats = 0);
float *q8_gemm_scratch(size_t *floats);  // the library's partial-sum array on the current device
constexpr size_t kGemmScratchFloats = size_t{8} << 20;  // its size (q8_gemm_skinny.hip: kSkScratchFloats)

// Where the partial planes of a K-sliced product go: the library's per-device scratch array (shared by every call on
// the device), or the caller's workspace (the re-entrant entry points).  A workspace smaller than the plan with all its
// slices needs means fewer or no slices.
struct GemmScratch {
    bool own = false;       // true: `ws` / `floats` below, never the library's array
    float *ws = nullptr;
    size_t floats = 0;
    size_t room() const { return own ? (ws ? (floats < kGemmScratchFloats ? floats : kGemmScratchFloats) : 0) : kGemmScratchFloats; }
};
lhip_status q8_gemm_reduce_launch(const float *part, void *y, int m, int n, int slices, int out, hipStream_t s, int ldy = 0);
constexpr int kTileSkinny = 5;        // K slices chosen by the library
constexpr int kTileSkinnySplit = 50;  // + number of K slices
constexpr int kTileSliced = 120;      // + number of K slices: the large tile over slices of K, then a reduction
constexpr int kTileTail = 200;        // more than one round of large tiles, whatever ends its last round first
constexpr int kTileDeep = 1000;       // + 10 mt + nt: q8_gemm_deep.hip; not by name from outside

// A product of more than 256 tiles of 128x256 runs in rounds of 256 workgroups (one per CU), and a last round that
// is partly filled takes as long as a full one.  The plan below gives whole rounds to one launch and the remaining
// column tiles to a K-sliced one (f32 partial planes in the scratch array, added in slice order), so that the
// remainder fills the chip for 1 / slices of a round: `n_main` leading weight rows in whole rounds, `slices` K slices
// for the rest (0: no such plan).  Needs the M tiles to divide 256, K long enough, and room for the planes.
// Mixing 256x256 and 128x256 tiles in one launch (q8_gemm_wide.hip) is the other way to end a last round early, and the
// better one unless the remainder is small; gemm_tail_pays compares them.
struct GemmTail {
    int n_main = 0, slices = 0;
};
static GemmTail gemm_tail_plan(int64_t m, int64_t n, int64_t k, int out, const void *y, size_t room) {
    GemmTail none;
    if (m <= 128 || k < 2048 || n % 4 != 0 || !aligned(y, out == kOutF32 ? 16 : (out == kOutBf16 ? 8 : 4))) return none;
    const int64_t m_tiles = (m + 255) / 256, n_tiles = (n + 127) / 128;  // halves of a 256x256 tile: 256x128 or 128x256
    if (m_tiles * n_tiles <= 256 || 256 % m_tiles != 0) return none;
    const int64_t per_round = 256 / m_tiles;                 // column tiles of one round
    const int64_t main_tiles = n_tiles / per_round * per_round;
    const int64_t tail_tiles = (n_tiles - main_tiles) * m_tiles;
    if (tail_tiles == 0) return none;
    const int64_t n_tail = n - main_tiles * 128, kt = k / kBK;
    for (int slices = 8; slices >= 2; slices >>= 1)
        if (tail_tiles * slices <= 256 && kt % slices == 0 && (kt / slices) % 4 == 0 &&
            static_cast<size_t>(slices) * m * n_tail <= room) {
            GemmTail t;
            t.n_main = static_cast<int>(main_tiles * 128);
            t.slices = slices;
            return t;
        }
    return none;
}

// Whether the sliced remainder ends before one launch of mixed tiles: half units of a 128x256 tile over all of K (0.64
// us per 64 of K), the remainder's share of a round, and its launch, its planes and their sum: 25 us behind several rounds, where the two
// are level at 1.06 of the one launch's time; behind a single one, whose planes are few, 2 us, unless 25 are a fifth of it.  Measured, us,
// sliced and one launch: 2023 x 17016 x 4096 321 and 335, 916 x 25056 x 4096 245 and 225; behind a single round 439 x 16896 x 5120 136 and 126,
// 794 x 8352 x 14336 320 and 282, 952 x 9028 x 2048 73 and 62, 479 x 16540 x 8192 194 and 212, 1906 x 4456 x 8192 194 and 197, 960 x 8196 x 4096 106
// and 106, 1024 x 8692 x 4096 111 and 108, 1962 x 4356 x 4096 113 and 107 (these three are sliced).
static bool gemm_tail_pays(const GemmTail &t, int64_t m, int64_t n, int64_t k) {
    if (t.slices < 2) return false;
    const double unit = 0.64 * static_cast<double>(k / kBK);
    const bool one_round = (m + 255) / 256 * (t.n_main / 128) <= 256;
    const double one = q8_gemm_wide_ends(m, n) * unit, sliced = q8_gemm_wide_ends(m, t.n_main) * unit + 2.0 * unit / t.slices;
    return one_round ? sliced + 2.0 < one && sliced + 25.0 < 1.22 * one : sliced + 25.0 < 1.06 * one;
}

// M tiles per group of the raster: the activation tiles of a group of rows stay in an XCD's L2 while its N tiles pass.
constexpr int kGemmMGroup = 8;
static int gemm_m_group(int m_tiles) { return m_tiles < kGemmMGroup ? m_tiles : kGemmMGroup; }

template <int BM, int BN, int WM, int WN, int D, typename OutT>
static lhip_status launch_gemm_t(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k,
                               int swiglu, hipStream_t s) {
    const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + BN - 1) / BN;
    const int n_tiles_pad = (n_tiles + 7) / 8 * 8;
    if (static_cast<int64_t>(m_tiles) * n_tiles_pad > 0x7fffffff) return LHIP_ERR_INVALID_SHAPE;  // the grid's x extent
    const size_t lds_bytes = 2 * (static_cast<size_t>(BM + BN) * kRowBytes + static_cast<size_t>(BN) * 8);
    auto kern = q8_gemm_bf16_kernel<BM, BN, WM, WN, D, OutT>;
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), lds_bytes)) return st;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(m_tiles * n_tiles_pad)), dim3(WM * WN * 64), lds_bytes, s, qs, ds,
                       static_cast<const __bf16 *>(x), static_cast<OutT *>(y), m, n, k, m_tiles, n_tiles, swiglu,
                       gemm_m_group(m_tiles));
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

template <int BM, int BN, int WM, int WN, int D>
static lhip_status launch_gemm(int out, const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k,
                             hipStream_t s) {
    return out == kOutF32 ? launch_gemm_t<BM, BN, WM, WN, D, float>(qs, ds, x, y, m, n, k, 0, s)
                          : launch_gemm_t<BM, BN, WM, WN, D, __bf16>(qs, ds, x, y, m, n, k, out == kOutSwiglu, s);
}

static lhip_status gemm_dispatch(const void *planar_dev, const void *x_dev, void *y_dev, int64_t m, int64_t n, int64_t k,
                                 int tile, int out, void *stream, const GemmScratch &scratch = GemmScratch{}) {
    if (!planar_dev || !x_dev || !y_dev) return LHIP_ERR_NULL_PTR;
    if (lhip_status s = check_q8_shape(n, k)) return s;
    if (m <= 0 || m > kMaxDim) return LHIP_ERR_INVALID_SHAPE;
    if (k % kBK != 0) return LHIP_ERR_UNSUPPORTED;
    if (out == kOutSwiglu && n % 4 != 0) return LHIP_ERR_INVALID_SHAPE;  // pairs, stored two at a time
    if (!aligned(planar_dev, 256) || !aligned(x_dev, 16) || !aligned(y_dev, out == kOutBf16 ? 2 : 4)) return LHIP_ERR_MISALIGNED;
    auto *base = static_cast<const uint8_t *>(planar_dev);
    auto *qs = reinterpret_cast<const int8_t *>(base);
    auto *ds = reinterpret_cast<const __half *>(base + q8_scale_offset(n, k));
    const int mi = static_cast<int>(m), ni = static_cast<int>(n), ki = static_cast<int>(k);
    hipStream_t s = as_stream(stream);
    const bool wide = q8_gemm_wide_supports(k);  // where not, asked for by name: the same product by tiles of 128x128
    if (tile == kTileSkinny || (tile > kTileSkinnySplit && tile <= kTileSkinnySplit + 64)) {
        if (!q8_gemm_skinny_supports(mi, ni, ki, out, y_dev)) return LHIP_ERR_UNSUPPORTED;
        // (a plain call of a K that is no multiple of 512 has no room: gemm_plain_room)
        return q8_gemm_skinny_launch(qs, ds, x_dev, y_dev, mi, ni, ki, out, tile == kTileSkinny ? 0 : tile - kTileSkinnySplit, s,
                                     scratch.own || k % 512 != 0, scratch.ws, scratch.floats);
    }
    if (tile > kTileDeep)
        return q8_gemm_deep_launch(qs, ds, x_dev, kWdBf16, y_dev, mi, ni, ki, out, DeepPlan{(tile - kTileDeep) / 10, tile % 10}, s);
    if (tile > kTileSliced && tile <= kTileSliced + 16) {
        // Few output tiles (the down projection of a 512-token prompt: 64 tiles of 128x256): slices of K fill the chip,
        // f32 partial planes go to the scratch array and are added in slice order.
        const int slices = tile - kTileSliced;
        const int kt = ki / kBK;
        size_t cap = scratch.room();
        float *part = scratch.own ? scratch.ws : q8_gemm_scratch(&cap);
        if (!part) return scratch.own ? LHIP_ERR_UNSUPPORTED : LHIP_ERR_HIP;
        if (slices < 2 || (slices - 1) * ((kt + slices - 1) / slices) >= kt ||
            static_cast<size_t>(slices) * mi * ni > cap || ni % 4 != 0 || !aligned(y_dev, out == kOutF32 ? 16 : (out == kOutBf16 ? 8 : 4)))
            return LHIP_ERR_UNSUPPORTED;
        if (wide) {
            if (lhip_status st = q8_gemm_wide_launch(qs, ds, x_dev, kWdBf16, part, mi, ni, ki, kOutF32, s, slices)) return st;
            return q8_gemm_reduce_launch(part, y_dev, mi, ni, slices, out, s);
        }
        tile = 0;
    }
    if (tile == kTileTail) {
        size_t cap = scratch.room();
        float *part = scratch.own ? scratch.ws : q8_gemm_scratch(&cap);
        if (!part) return scratch.own ? LHIP_ERR_UNSUPPORTED : LHIP_ERR_HIP;
        const GemmTail t = gemm_tail_plan(m, n, k, out, y_dev, cap);
        if (t.slices < 2) return LHIP_ERR_UNSUPPORTED;
        if (wide && gemm_tail_pays(t, m, n, k)) {
            const int n_tail = ni - t.n_main;
            // whole rounds: the leading n_main weight rows, written into the full-width output
            if (lhip_status st = q8_gemm_wide_launch(qs, ds, x_dev, kWdBf16, y_dev, mi, t.n_main, ki, out, s, 1, ni)) return st;
            // the rest: K slices of the trailing weight rows into the planes, then their sum into the trailing columns
            const int8_t *qs_tail = qs + static_cast<size_t>(t.n_main) * ki;
            const __half *ds_tail = ds + static_cast<size_t>(t.n_main) * (ki / 32);
            if (lhip_status st = q8_gemm_wide_launch(qs_tail, ds_tail, x_dev, kWdBf16, part, mi, n_tail, ki, kOutF32, s, t.slices)) return st;
            const size_t col0 = out == kOutSwiglu ? t.n_main / 2 : t.n_main;
            void *y_tail = out == kOutF32 ? static_cast<void *>(static_cast<float *>(y_dev) + col0)
                                          : static_cast<void *>(static_cast<__bf16 *>(y_dev) + col0);
            return q8_gemm_reduce_launch(part, y_tail, mi, n_tail, t.slices, out, s, ni);
        }
        tile = 0;
    }
    // Register prefetch four (two) K tiles ahead needs K to be a whole number of 4-tile (2-tile) rounds.
    const int depth = (k % (kBK * 4)) == 0 ? 4 : ((k % (kBK * 2)) == 0 ? 2 : 1);
#define LHIP_TILE(BM, BN, WM, WN)                                                                          \
    return depth == 4   ? launch_gemm<BM, BN, WM, WN, 4>(out, qs, ds, x_dev, y_dev, mi, ni, ki, s)      \
           : depth == 2 ? launch_gemm<BM, BN, WM, WN, 2>(out, qs, ds, x_dev, y_dev, mi, ni, ki, s)      \
                        : launch_gemm<BM, BN, WM, WN, 1>(out, qs, ds, x_dev, y_dev, mi, ni, ki, s)
    switch (tile) {
        case 0:
            if (wide) return q8_gemm_wide_launch(qs, ds, x_dev, kWdBf16, y_dev, mi, ni, ki, out, s);
            [[fallthrough]];
        case 1: LHIP_TILE(128, 128, 2, 2);
        case 2: LHIP_TILE(128, 64, 2, 2);
        case 3: LHIP_TILE(64, 64, 2, 2);
        default: return LHIP_ERR_UNSUPPORTED;
    }
#undef LHIP_TILE
}

// Room that the plain entry points plan with: the scratch array for K in steps of 512 only, as in the f32 / f16 operators.
// For every other K they keep nothing outside their outputs, so that their calls may overlap on several streams.
static size_t gemm_plain_room(int64_t k) { return k % 512 == 0 ? kGemmScratchFloats : 0; }

// What a product of more than 32 rows takes without K slices, us, and by which tiles: 64x64 where 128x64 are fewer than 64,
// 128x64 where the large ones are fewer than 32 or end later.  Up to 256 tiles of this file's kernel run one to a CU and up to
// 512 two, 128x64 at 1.0 and 1.22 us per 64 of K, 64x64 at 0.6 (an eighth more where the loads run one tile ahead only); a
// 128x256 tile takes 1.07 with most of the chip idle; and each launch some microseconds, more for an odd N.  Measured, large ->
// 128x64, us: 128 x 8190 x 4096 75 -> 69, 512 x 2001 x 14336 246 -> 227, 300 x 2879 x 256 11.7 -> 8.1, 777 x 2001 x 256 12.0 ->
// 8.5, 512 x 4095 x 256 11.9 -> 8.7; the other way 512 x 8190 x 1024 24.7 <- 26.2, 300 x 8190 x 4096 75 <- 83.
// (The output form has no part in the choice: the SwiGLU form has the bits of the f32 one.)
static double gemm_unsliced_us(int64_t m, int64_t n, int64_t k, int *tile) {
    const int64_t large = (m + 127) / 128 * ((n + 255) / 256), small = (m + 127) / 128 * ((n + 63) / 64);
    const double kt = static_cast<double>(k / kBK), ahead = k % (kBK * 2) != 0 ? 1.12 : 1.0;
    double us = small < 64 ? 3.0 + 0.6 * ahead * kt : small <= 256 ? 4.3 + 1.0 * ahead * kt : 5.9 + 1.22 * ahead * kt;
    *tile = small < 64 ? 3 : 2;
    if (large >= 32 && q8_gemm_wide_supports(k)) {
        const double wide = (n % 2 != 0 ? 7.7 : 5.4) + q8_gemm_wide_ends(m, n) * 0.535 * kt;
        if (small > 512 || wide <= us) us = wide, *tile = 0;
    }
    return us;
}
// And over slices of `per` 64-wide tiles: two launches, a workgroup's walk, and the planes written and read once more.
// Measured, sliced -> not, us: 512 x 4096 x 1024 over four 24.1 -> 21.8, 364 x 10496 x 512 over two 25.9 -> 11, 72 x 2600 x 768
// over three 11.8 -> 9.9; the other way 4096 x 4096 at 512 rows 38 <- 73, 2880 x 2880 at 128 rows 21 <- 33.  The small tiles
// exchange SwiGLU's pairs between lanes, 128x64 for 4 us and 64x64 for 3: half of that stands against them for every form.
static double gemm_sliced_us(int64_t m, int64_t n, int64_t slices, int64_t per, int64_t workgroups) {
    return 8.3 + static_cast<double>(per) * (1.03 + 0.06 * static_cast<double>(workgroups) / 256.0) + (per < 5 ? 0.3 : 0.0) +
           0.33e-6 * 4.0 * static_cast<double>(slices * m) * static_cast<double>(n);
}

// The tiles (kTile...) for a product that the weight-streaming kernel does not take, and their time, us.
static int gemm_tiles(int64_t m, int64_t n, int64_t k, int out, const void *y, size_t room, double *us) {
    const int64_t kt = k / kBK, b0 = (m + 127) / 128 * ((n + 255) / 256);
    if (m <= 32) {
        const int tile = (m + 127) / 128 * ((n + 63) / 64) >= 64 ? 2 : 3;
        *us = tile == 2 ? 4.3 + static_cast<double>(kt) : 3.0 + 0.6 * (k % (kBK * 2) != 0 ? 1.12 : 1.0) * static_cast<double>(kt);
        return tile;
    }
    int tile;
    *us = gemm_unsliced_us(m, n, k, &tile);
    const double unsliced = *us + (tile == 2 ? 2.2 : tile == 3 ? 1.3 : 0.0);
    // Few 128x256 tiles: slices of K until the chip is full (at most eight, of at least four 64-wide tiles), when the
    // partial planes fit the scratch array and cost less than the shorter walk saves (measured, us, whole K -> sliced: 4096 x
    // 4096 at 512 rows 73 -> 36, 4096 x 14336 at 512 rows 244 -> 85, 2880 x 2880 at 777 rows 54 -> 33 over three uneven
    // slices).  Up to 128 rows only what the weight-streaming kernel does not cover.
    if (q8_gemm_wide_supports(k)) {
        if (n % 4 == 0 && aligned(y, out == kOutF32 ? 16 : (out == kOutBf16 ? 8 : 4)))
            for (int64_t slices = 256 / b0 < 8 ? 256 / b0 : 8; slices >= 2; --slices) {
                const int64_t per = (kt + slices - 1) / slices;
                if (per < 4 || (slices - 1) * per >= kt || static_cast<size_t>(slices) * m * n > room) continue;
                const double sliced = gemm_sliced_us(m, n, slices, per, b0 * slices);
                if (sliced < unsliced) {
                    *us = sliced;
                    return kTileSliced + static_cast<int>(slices);
                }
            }
        if (gemm_tail_plan(m, n, k, out, y, room).slices >= 2) return kTileTail;
    }
    return tile;
}

// The weight-streaming kernel, or slices or tiles; *us: what the latter take.
static int gemm_slices_or_tiles(int64_t m, int64_t n, int64_t k, int out, const void *y, size_t room, double *us) {
    *us = 0.0;
    // Few activation rows: the product is bound by the weight stream.  A K that is no multiple of 512 is one for that kernel
    // unless the tiles end within a tenth of it, which they do for a K of one step and for many weight rows.  Measured, us,
    // tiles -> streamed, without and with a workspace: 16 x 2880 x 2880 33 -> 9.9 and 33 -> 8.6, 45 x 2880 x 2880 33 -> 17 and 15.9 ->
    // 13.4, 128 x 4096 x 4160 79 -> 36 and 22.5 -> 20, 16 x 28672 x 960 24 -> 10.7; the other way 128 x 28672 x 320 11.5 <- 13.7,
    // 80 x 28672 x 4160 with one 54 <- 60.
    if (m <= 128 && n <= kMaxDim && k <= kMaxDim &&
        q8_gemm_skinny_supports(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), out, y)) {
        if (k % 512 == 0) return kTileSkinny;
        const int tile = gemm_tiles(m, n, k, out, y, room, us);
        return 1.1 * q8_gemm_skinny_us(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), room) < *us ? kTileSkinny : tile;
    }
    return gemm_tiles(m, n, k, out, y, room, us);
}

// Those, or the kernel whose workgroups walk all of K, where it ends a twentieth sooner, the spread of the estimates.  Measured, us,
// tiles and slices -> that kernel: 192 x 6000 x 1536 23.3 -> 11.7, 256 x 4096 x 4096 27.0 -> 20.5, 1024 x 1024 x 4096 28.6 -> 22.6, 352 x
// 3067 x 12288 (no slices for an odd N) 191 -> 69; the other way 256 x 14336 x 4096 54 <- 66, 592 x 9820 x 768 23 <- 38.  The slices that the
// header promises a long K stay: at 8192 and more they are ahead for most sizes (350 x 6364 x 10688 82 <- 119, 207 x 2276 x 12992 40
// <- 43), though not for few weight rows (171 x 544 x 8192 26.3 -> 19.8).  From 6144 on a seventh, for weights from memory: 141 x 3540 x 6144 28.0 <-
// 30.0, 167 x 3528 x 7552 31.2 <- 34.0, 312 x 1928 x 7424 31.3 <- 33.6.
// Up to 128 rows the streaming kernel stays for K below three of its steps of 512 and, where it is ahead of tiles and slices, for every
// K outside those steps.  Where they are ahead of it, the other kernel takes what it ends a seventh sooner; us, weights from memory (from the
// cache), tiles or slices -> it: 128 x 2880 x 2880 22.0 -> 13.9 (20.6 -> 10.9), 101 x 468 x 576 9.1 -> 4.2, 57 x 6512 x 5760 27.3 -> 25.4 (26.3 ->
// 20.0); mean of 62 sizes 1.55 (1.72) times as fast, none slower; at a twentieth 124 x 14128 x 4480 39.3 <- 41.3.  From three steps on the
// other kernel takes what it ends a fifth sooner above 64 rows, for which the strips are bound by their reads of the activations and no
// longer by the weights, and a quarter sooner from 33 on: the estimates are of weights that the memory-side cache holds, and from memory
// that kernel loses 1.5 to 2 us more.  Measured, us, strips -> that kernel, weights from memory: 80 x 4096 x 4096 16.8 -> 14.8, 80 x 6144 x
// 4096 21.9 -> 20.4, 48 x 6144 x 4096 18.8 -> 15.2, the other way 100 x 4096 x 4096 17.7 <- 19.1; from the cache: 80 x 4096 x 4096 16.8 ->
// 12.7, 96 x 14336 x 4096 33.7 -> 29.8, 128 x 6000 x 1536 13.8 -> 9.9, 96 x 8148 x 2048 15.8 -> 11.4, 45 x 14336 x 4096 27.6 -> 22.6.
static int gemm_auto_tile(int64_t m, int64_t n, int64_t k, int out, const void *y, size_t room) {
    double us;
    const int tile = gemm_slices_or_tiles(m, n, k, out, y, room, &us);
    const bool streams = m <= 128 && q8_gemm_skinny_supports(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), out, y);
    const bool sliced = tile > kTileSliced && tile < kTileTail;
    double margin = streams || (sliced && k >= 6144) ? 1.15 : 1.05;
    if (streams && tile == kTileSkinny) {
        if (m <= 32 || k % 512 != 0 || k < 1536) return tile;
        us = q8_gemm_skinny_us(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), room);
        margin = m > 64 ? 1.2 : 1.25;
    }
    if ((sliced && k >= 8192) || k < 256 || !q8_gemm_deep_supports(k, nullptr)) return tile;
    const DeepPlan deep = q8_gemm_deep_plan(m, n, k, us / margin);
    return deep.mt ? kTileDeep + 10 * deep.mt + deep.nt : tile;
}

void q8_gemm_describe(int64_t m, int64_t n, int64_t k, size_t room, int32_t plan[3]) {
    room = room == SIZE_MAX ? gemm_plain_room(k) : room < kGemmScratchFloats ? room : kGemmScratchFloats;
    const int tile = gemm_auto_tile(m, n, k, kOutBf16, nullptr, room);
    if (tile == kTileSkinny) return q8_gemm_skinny_describe(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), room, plan);
    if (tile > kTileDeep) {
        plan[0] = 4, plan[1] = 32 * (tile % 10), plan[2] = 1;
        return;
    }
    plan[0] = 3, plan[1] = tile == 0 && q8_gemm_wide_supports(k) ? q8_gemm_wide_special_height(m, n) : 0;
    plan[2] = tile == kTileTail ? 0 : tile > kTileSliced ? tile - kTileSliced : 1;
}

}  // namespace lhip

using namespace lhip;

extern "C" {

lhip_status lhip_q8_0_matmul_bf16_cfg(const void *planar_dev, const void *x_dev, void *y_dev, int64_t m, int64_t n,
                                      int64_t k, int tile, void *stream) {
    if (tile > kTileTail) return LHIP_ERR_UNSUPPORTED;
    if (tile > kTileSliced && tile <= kTileSliced + 16 && k % (kBK * 4 * (tile - kTileSliced)) != 0) return LHIP_ERR_UNSUPPORTED;
    if ((tile == kTileSkinny || (tile > kTileSkinnySplit && tile <= kTileSkinnySplit + 64)) && k % 512 != 0) return LHIP_ERR_UNSUPPORTED;
    return gemm_dispatch(planar_dev, x_dev, y_dev, m, n, k, tile, kOutBf16, stream);
}

lhip_status lhip_q8_0_matmul_bf16(const void *planar_dev, const void *x_dev, void *y_dev, int64_t m, int64_t n,
                                  int64_t k, void *stream) {
    return gemm_dispatch(planar_dev, x_dev, y_dev, m, n, k, gemm_auto_tile(m, n, k, kOutBf16, y_dev, gemm_plain_room(k)), kOutBf16, stream);
}

lhip_status lhip_q8_0_matmul_bf16_f32out(const void *planar_dev, const void *x_dev, float *y_dev, int64_t m, int64_t n,
                                         int64_t k, void *stream) {
    return gemm_dispatch(planar_dev, x_dev, y_dev, m, n, k, gemm_auto_tile(m, n, k, kOutF32, y_dev, gemm_plain_room(k)), kOutF32, stream);
}

lhip_status lhip_q8_0_matmul_bf16_swiglu(const void *planar_dev, const void *x_dev, void *out_dev, int64_t m, int64_t n,
                                         int64_t k, void *stream) {
    return gemm_dispatch(planar_dev, x_dev, out_dev, m, n, k, gemm_auto_tile(m, n, k, kOutSwiglu, out_dev, gemm_plain_room(k)), kOutSwiglu, stream);
}

size_t lhip_q8_0_matmul_bf16_workspace_nbytes(int64_t m, int64_t n, int64_t k, int32_t out_form) {
    if (check_q8_shape(n, k) != LHIP_OK || m <= 0 || m > kMaxDim || k % kBK != 0) return 0;
    if (out_form < kOutBf16 || out_form > kOutSwiglu) return 0;
    // the plan with all its slices (an aligned output is assumed: K is sliced for aligned outputs only), also where the kernel that
    // needs no planes is ahead of it: callers' sizes stay what they were
    double us;
    const int tile = gemm_slices_or_tiles(m, n, k, out_form, nullptr, kGemmScratchFloats, &us);
    size_t floats = 0;
    if (tile > kTileSliced && tile <= kTileSliced + 16)
        floats = static_cast<size_t>(tile - kTileSliced) * m * n;
    else if (tile == kTileTail) {
        const GemmTail t = gemm_tail_plan(m, n, k, out_form, nullptr, kGemmScratchFloats);
        floats = static_cast<size_t>(t.slices) * m * (n - t.n_main);
    }
    else if (tile == kTileSkinny) {
        const int splits = q8_gemm_skinny_splits(static_cast<int>(m), static_cast<int>(n), static_cast<int>(k), kGemmScratchFloats);
        if (splits > 1) floats = static_cast<size_t>(splits) * m * n;
    }
    return floats * sizeof(float);
}

lhip_status lhip_q8_0_matmul_bf16_ws(const void *planar_dev, const void *x_dev, void *y_dev, int64_t m, int64_t n, int64_t k,
                                     int32_t out_form, void *workspace_dev, size_t workspace_nbytes, void *stream) {
    if (out_form < kOutBf16 || out_form > kOutSwiglu) return LHIP_ERR_INVALID_SHAPE;
    if (workspace_dev && !aligned(workspace_dev, 256)) return LHIP_ERR_MISALIGNED;
    GemmScratch scratch;
    scratch.own = true;
    scratch.ws = static_cast<float *>(workspace_dev);
    scratch.floats = workspace_dev ? workspace_nbytes / sizeof(float) : 0;
    return gemm_dispatch(planar_dev, x_dev, y_dev, m, n, k, gemm_auto_tile(m, n, k, out_form, y_dev, scratch.room()), out_form,
                         stream, scratch);
}

}  // extern "C"
