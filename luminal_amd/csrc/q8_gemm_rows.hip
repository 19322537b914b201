// Q8_0 weights x several activation rows, f32 or f16, on the matrix cores: the operators behind lhip_q8_0_matmul_f32 and
// _f16 for more rows than the weight-streaming kernel of q8_gemm_skinny.hip serves well, and for every K that is a
// multiple of 32 only (that kernel walks K in steps of 512).
//
// The arithmetic is that of q8_gemm_skinny.hip and q8_gemm_wide.hip: int8 codes exact in bf16 / f16, an f32 activation as
// three bf16 limbs whose sum is the value exactly (one chained matrix step per limb), an f16 one as it is (one step), the
// f32 sum of a block's products scaled by the block's d on the vector ALU.
//
// Three limbs make the matrix pipe the bound (192 of its cycles per 32 x 32 outputs and block; a register-only loop of
// the mix takes 207), so everything else is kept out of the way of the matrix steps:
//   * a wave owns 16 activation rows and all 256 weight rows of the tile: it loads its rows straight into registers, in
//     operand order, two blocks ahead, and splits them there - each value once per workgroup, no planes in memory, no
//     LDS for activations (planes brought to LDS: 24 operand reads per block and wave instead of 16);
//   * the codes are the shared operand: four loader waves, one per SIMD, bring a group of four blocks into LDS as bf16 /
//     f16 while the eight compute waves multiply the group before, one barrier per group.  Dealt out among the compute
//     waves instead, that work stands in front of their matrix steps (512 x 14336 x 4096 f32: 176 -> 161 us);
//   * the operand reads run two pairs of fragments ahead, the scaling of a pair runs under the next pair's steps.
// Measured, whole operator, passes of 64 rows of q8_gemm_skinny.hip -> this kernel: f32 14336 x 4096 at 256 / 512 rows
// 120 -> 83 / 239 -> 145 us; 2880 x 2880 at 45 rows (K is no multiple of 512: one matvec per row before) 97 -> 13, of which
// the sum of the slices takes 3.  Tiles of 224 weight rows fill the chip at 256 x 14336 (128 tiles x 2 slices, 85 -> 83), of 128 at 45
// x 2880 (23 tiles x 8 slices for 12 x 12, 14.6 -> 12.2).
#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "q8_gemm_rows.h"
#include "q8_mma_device.h"

namespace lhip {

constexpr int kRwBN = 256;                      // weight rows per workgroup, at most
constexpr int kRwPlane = kRwBN * 64 + 64;       // bytes of one block's codes as bf16 / f16, and a shift of the banks
constexpr int kRwBuf = 4 * kRwPlane + 4 * kRwBN * 4;  // a group of four blocks and its scales as f32
constexpr int kRwLds = 2 * kRwBuf;
enum { kRwOutF32 = 1, kRwOutF16 = 4 };  // as in q8_gemm_skinny.hip

// Workgroup tile: 128 activation rows (a compute wave: 16) x 16 FR weight rows (256, or fewer where these end sooner: a tile's time
// goes nearly with its weight rows, and the launch's with its rounds of 256 tiles; the LDS is laid out for 256), over slice_blocks blocks of K; with more than one
// slice each goes into an f32 plane of (M, N) of its own.  ldy = row pitch of y (N, or more when the launch fills some columns
// of a wider output).
template <typename XT, int OUT, int FR>
__global__ __launch_bounds__(768) void q8_gemm_rows_kernel(const int8_t *__restrict__ qs, const unsigned short *__restrict__ ds,
                                                           const XT *__restrict__ x, void *__restrict__ y, int M, int N, int K,
                                                           int m_tiles, int n_tiles, int slices, int slice_blocks, int ldy) {
    constexpr bool kF16 = !std::is_same<XT, float>::value;
    constexpr int L = kF16 ? 1 : 3;                            // operands per value
    constexpr int XW = sizeof(XT) == 4 ? 2 : 1;                // 16-byte loads per 8 values
    constexpr int BN = 16 * FR, PP = FR / 2;                   // weight rows; pairs of fragments
    static_assert(FR % 2 == 0 && BN <= kRwBN, "pairs of fragments");
    extern __shared__ __attribute__((aligned(16))) unsigned char rw_lds[];
    int mt, nt, slice;
    {
        const int u = xcd_item(blockIdx.x, m_tiles * n_tiles * slices);
        if (u < 0) return;
        mt = u % m_tiles;
        const int ns = u / m_tiles;
        nt = ns / slices;
        slice = ns - nt * slices;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int nblk = K >> 5;
    const int blk0 = slice * slice_blocks, nb = min(slice_blocks, nblk - blk0);  // this slice's blocks
    const int groups = (nb + 3) >> 2;
    const int m0 = mt * 128 + wave * 16, n0 = nt * BN;
    const bool idle = m0 >= M;  // a wave without rows only stages

    auto swz = [](int row) { return (4 - (row >> 2)) & 3; };
    if (wave >= 8) {
        // ---- loaders: a group's codes -> registers -> bf16 / f16 in LDS, two groups ahead of their use.  Thread
        // (row lt / 8 + 32 q, piece lt % 8) holds 16 codes of a group's 128.
        const int lt = tid - 512, wp = lt & 7, wrow = lt >> 3;
        const int8_t *w_src[PP];
#pragma unroll
        for (int q = 0; q < PP; ++q)
            w_src[q] = qs + static_cast<size_t>(min(n0 + q * 32 + wrow, N - 1)) * K + static_cast<size_t>(blk0) * 32;
        const int w_dst = (wp >> 1) * kRwPlane + wrow * 64 + (((wp & 1) * 2) ^ swz(wrow)) * 16;  // second half: ^ 16; pass q: + 32 rows
        const unsigned short *s_src = ds + static_cast<size_t>(min(n0 + lt, N - 1)) * nblk + blk0;
        const int s_dst = 4 * kRwPlane + ((lt >> 5) * 16 + (lt & 15)) * 8 + ((lt >> 4) & 1) * 4;
        mma_u32x4 wreg[2][PP];
        unsigned short sreg[2][4];
        auto load_w = [&](int set, int grp) __attribute__((always_inline)) {
            // pieces of blocks past the slice's end repeat its last block's (never multiplied)
            const int b = min(grp * 4 + (wp >> 1), nb - 1);
#pragma unroll
            for (int q = 0; q < PP; ++q) wreg[set][q] = *reinterpret_cast<const mma_u32x4 *>(w_src[q] + b * 32 + (wp & 1) * 16);
#pragma unroll
            for (int h = 0; h < 4; ++h) sreg[set][h] = s_src[min(grp * 4 + h, nb - 1)];
        };
        auto store_w = [&](int set, unsigned char *buf) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < PP; ++q) {
                asm volatile("" : "+v"(wreg[set][q]));
                const mma_u32x4 &w = wreg[set][q];
                const mma_u32x4 lo = {codes2<kF16>(w[0], 0), codes2<kF16>(w[0], 1), codes2<kF16>(w[1], 0), codes2<kF16>(w[1], 1)};
                const mma_u32x4 hi = {codes2<kF16>(w[2], 0), codes2<kF16>(w[2], 1), codes2<kF16>(w[3], 0), codes2<kF16>(w[3], 1)};
                *reinterpret_cast<mma_u32x4 *>(buf + w_dst + q * 32 * 64) = lo;
                *reinterpret_cast<mma_u32x4 *>(buf + (w_dst ^ 16) + q * 32 * 64) = hi;
            }
#pragma unroll
            for (int h = 0; h < 4; ++h)
                *reinterpret_cast<float *>(buf + s_dst + h * kRwBN * 4) = __half2float(__ushort_as_half(sreg[set][h]));
        };
        load_w(0, 0);
        load_w(1, 1);
        store_w(0, rw_lds);
        load_w(0, 2);
        __syncthreads();
        for (int grp = 0; grp < groups; grp += 2) {
            store_w(1, rw_lds + kRwBuf);
            load_w(1, grp + 3);
            __syncthreads();
            if (grp + 1 >= groups) return;
            store_w(0, rw_lds);
            load_w(0, grp + 4);
            __syncthreads();
        }
        return;
    }

    // ---- activations: lane (r, g) loads values 8 g .. 8 g + 7 of a block of row r, two blocks ahead
    const XT *x_src = x + static_cast<size_t>(min(m0 + r, M - 1)) * K + static_cast<size_t>(blk0) * 32 + g * 8;
    mma_u32x4 xraw[2][XW], xop[L];
    auto load_x = [&](int set, int b) __attribute__((always_inline)) {
        const int bb = min(b, nb - 1);
#pragma unroll
        for (int w = 0; w < XW; ++w) xraw[set][w] = reinterpret_cast<const mma_u32x4 *>(x_src + static_cast<size_t>(bb) * 32)[w];
    };
    auto split_x = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < XW; ++w) asm volatile("" : "+v"(xraw[set][w]));  // the arithmetic stays here, behind the loads' wait
        if constexpr (L == 1) {
            xop[0] = xraw[set][0];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t limb[L];
                split_limbs2<L>(__uint_as_float(xraw[set][e >> 1][(e & 1) * 2]), __uint_as_float(xraw[set][e >> 1][(e & 1) * 2 + 1]), limb);
#pragma unroll
                for (int l = 0; l < L; ++l) xop[l][e] = limb[l];
            }
        }
    };

    mma_f32x4 acc[FR];
#pragma unroll
    for (int j = 0; j < FR; ++j) acc[j] = mma_f32x4{0.f, 0.f, 0.f, 0.f};

    const int b_lane = r * 64 + ((g ^ swz(r)) * 16);
    const int s_lane = 4 * kRwPlane + r * 8;
    // NB blocks of a group, from block B0 on: PP pairs of weight fragments each against the wave's rows.
    auto blocks = [&](const unsigned char *buf, int blk, auto nbc, auto first) __attribute__((always_inline)) {
        constexpr int NB = decltype(nbc)::value, B0 = decltype(first)::value, RING = 4, AHEAD = 2;
        mma_u32x4 br[RING][2];
        float sc[RING][2];
        auto read_b = [&](int p) __attribute__((always_inline)) {
            const int b = B0 + p / PP;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                br[p % RING][j] = *reinterpret_cast<const mma_u32x4 *>(buf + b * kRwPlane + b_lane + (2 * (p % PP) + j) * 16 * 64);
            const float2 s2 = *reinterpret_cast<const float2 *>(buf + s_lane + b * kRwBN * 4 + (p % PP) * 128);
            sc[p % RING][0] = s2.x;
            sc[p % RING][1] = s2.y;
        };
#pragma unroll
        for (int p = 0; p < AHEAD; ++p) read_b(p);
        mma_f32x4 last[2];
        auto scale = [&](int p, int j) __attribute__((always_inline)) {  // the sums of pair p
            mma_f32x4 &a = acc[2 * (p % PP) + j];
#pragma unroll
            for (int v = 0; v < 4; ++v) a[v] = fmaf(sc[p % RING][j], last[j][v], a[v]);
            asm volatile("" : "+v"(a));
        };
        static_for<PP * NB>([&](auto pc) __attribute__((always_inline)) {
            constexpr int p = decltype(pc)::value, b = B0 + p / PP;
            if constexpr (p % PP == 0) {
                split_x(b & 1);
                load_x(b & 1, blk + b + 2);
            }
            if constexpr (p + AHEAD < PP * NB) read_b(p + AHEAD);
            mma_f32x4 s[2];
            // The fences hold this order: the two fragments' chains alternate, small limbs first, and the scaling of the
            // pair before stands in the middle of them.
            static_for<L>([&](auto lc) __attribute__((always_inline)) {
                constexpr int l = L - 1 - decltype(lc)::value;
                static_for<2>([&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value;
                    const mma_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                    __builtin_amdgcn_sched_barrier(0);
                    s[j] = mma_16x16x32<kF16>(xop[l], br[p % RING][j], l == L - 1 ? zero : s[j]);
                    asm volatile("" : "+v"(s[j]));
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (p > 0 && l == L / 2) scale(p - 1, j);
                });
            });
            last[0] = s[0];
            last[1] = s[1];
        });
        scale(PP * NB - 1, 0);
        scale(PP * NB - 1, 1);
    };
    if (idle) {
        for (int grp = 0; grp <= groups; ++grp) __syncthreads();
        return;
    }
    load_x(0, 0);
    load_x(1, 1);
    __syncthreads();
    const int whole_groups = nb >> 2;
    for (int grp = 0; grp < whole_groups; ++grp) {
        const unsigned char *buf = rw_lds + (grp & 1) * kRwBuf;
        blocks(buf, grp * 4, std::integral_constant<int, 4>{}, std::integral_constant<int, 0>{});
        __syncthreads();
    }
    const unsigned char *buf = rw_lds + (whole_groups & 1) * kRwBuf;
    constexpr std::integral_constant<int, 1> one{};
    if ((nb & 3) >= 1) blocks(buf, whole_groups * 4, one, std::integral_constant<int, 0>{});
    if ((nb & 3) >= 2) blocks(buf, whole_groups * 4, one, std::integral_constant<int, 1>{});
    if ((nb & 3) >= 3) blocks(buf, whole_groups * 4, one, std::integral_constant<int, 2>{});
    if (nb & 3) __syncthreads();

    // ---- epilogue: element v of lane (r, g) is row 4 g + v, column r of its 16 x 16 tile; rows of 16 FR through LDS
    constexpr int EP = 260;
    float *ep = reinterpret_cast<float *>(rw_lds) + wave * (16 * EP);
    static_assert(8 * 16 * EP * 4 <= kRwLds, "epilogue buffer");
    using OT = std::conditional_t<OUT == kRwOutF32, float, _Float16>;
    OT *yo = static_cast<OT *>(y) + static_cast<size_t>(slice) * M * N;
    const int col = n0 + lane * 4;
    const bool whole = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(yo) & (4 * sizeof(OT) - 1)) == 0;
#pragma unroll
    for (int j = 0; j < FR; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) ep[(4 * g + v) * EP + j * 16 + r] = acc[j][v];
    if (lane * 4 >= BN) return;  // the next tile's columns
#pragma unroll 4
    for (int q = 0; q < 16; ++q) {
        const int row = m0 + q;
        const mma_f32x4 v = *reinterpret_cast<const mma_f32x4 *>(ep + q * EP + lane * 4);
        if (row >= M) break;
        OT *p = yo + static_cast<size_t>(row) * ldy + col;
        if (whole && col + 4 <= N) {
            typedef OT otx4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<otx4 *>(p) = otx4{static_cast<OT>(v[0]), static_cast<OT>(v[1]), static_cast<OT>(v[2]), static_cast<OT>(v[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < N) p[e] = static_cast<OT>(v[e]);
        }
    }
}

// Sum of the K slices in slice order, for rows that do not start on 16 bytes.
template <typename OT>
__global__ __launch_bounds__(256) void q8_gemm_rows_reduce_kernel(const float *__restrict__ part, OT *__restrict__ y, int M, int N,
                                                                  int slices, int ldy) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x, count = static_cast<size_t>(M) * N;
    if (i >= count) return;
    float v = part[i];
    int s = 1;
    auto add = [&](auto batch) __attribute__((always_inline)) {  // the next planes: their loads first
        constexpr int C = decltype(batch)::value;
        float p[C];
#pragma unroll
        for (int u = 0; u < C; ++u) p[u] = part[(s + u) * count + i];
#pragma unroll
        for (int u = 0; u < C; ++u) v += p[u];
        s += C;
    };
    while (s + 6 <= slices) add(std::integral_constant<int, 6>{});
    if (s + 3 <= slices) add(std::integral_constant<int, 3>{});
    while (s < slices) add(std::integral_constant<int, 1>{});
    const size_t m = i / N;
    y[m * ldy + (i - m * N)] = static_cast<OT>(v);
}

template <typename XT, int OUT, int FR>
static lhip_status rw_launch_w(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, int slices, int ldy,
                               hipStream_t s) {
    const int m_tiles = (m + 127) / 128, n_tiles = (n + 16 * FR - 1) / (16 * FR);
    const int64_t total = static_cast<int64_t>(m_tiles) * n_tiles * slices;
    if (total > 0x7ffffff0) return LHIP_ERR_INVALID_SHAPE;  // the grid's x extent
    const int per = q8_gemm_rows_slice_blocks(k, slices);
    if (static_cast<int64_t>(slices - 1) * per >= k / 32) return LHIP_ERR_UNSUPPORTED;  // an empty slice
    auto kern = q8_gemm_rows_kernel<XT, OUT, FR>;
    static LdsOptIn opt;
    if (lhip_status st = lds_opt_in(opt, reinterpret_cast<const void *>(kern), kRwLds)) return st;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((total + 7) / 8 * 8)), dim3(768), kRwLds, s, qs,
                       reinterpret_cast<const unsigned short *>(ds), static_cast<const XT *>(x), y, m, n, k, m_tiles, n_tiles, slices,
                       per, ldy);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

template <typename XT, int OUT>
static lhip_status rw_launch_t(int width, const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, int slices,
                               int ldy, hipStream_t s) {
    switch (width) {
        case 128: return rw_launch_w<XT, OUT, 8>(qs, ds, x, y, m, n, k, slices, ldy, s);
        case 192: return rw_launch_w<XT, OUT, 12>(qs, ds, x, y, m, n, k, slices, ldy, s);
        case 224: return rw_launch_w<XT, OUT, 14>(qs, ds, x, y, m, n, k, slices, ldy, s);
        default: return rw_launch_w<XT, OUT, 16>(qs, ds, x, y, m, n, k, slices, ldy, s);
    }
}

int q8_gemm_rows_slice_blocks(int64_t k, int slices) {
    return static_cast<int>(((k / 32 + slices - 1) / slices + 3) / 4 * 4);
}

lhip_status q8_gemm_reduce_launch(const float *part, void *y, int m, int n, int slices, int out, hipStream_t s, int ldy = 0);

lhip_status q8_gemm_rows_launch(const int8_t *qs, const __half *ds, const void *x, void *y, int m, int n, int k, bool f16, int width,
                                int slices, float *part, int ldy, hipStream_t s) {
    if (slices == 1)
        return f16 ? rw_launch_t<__half, kRwOutF16>(width, qs, ds, x, y, m, n, k, 1, ldy, s)
                   : rw_launch_t<float, kRwOutF32>(width, qs, ds, x, y, m, n, k, 1, ldy, s);
    if (lhip_status st = f16 ? rw_launch_t<__half, kRwOutF32>(width, qs, ds, x, part, m, n, k, slices, n, s)
                             : rw_launch_t<float, kRwOutF32>(width, qs, ds, x, part, m, n, k, slices, n, s))
        return st;
    if (n % 4 == 0 && ldy % 4 == 0 && aligned(y, f16 ? 8 : 16))
        return q8_gemm_reduce_launch(part, y, m, n, slices, f16 ? kRwOutF16 : kRwOutF32, s, ldy);
    const dim3 grid(static_cast<unsigned>((static_cast<size_t>(m) * n + 255) / 256));
    if (f16)
        hipLaunchKernelGGL(q8_gemm_rows_reduce_kernel<_Float16>, grid, dim3(256), 0, s, part, static_cast<_Float16 *>(y), m, n, slices, ldy);
    else
        hipLaunchKernelGGL(q8_gemm_rows_reduce_kernel<float>, grid, dim3(256), 0, s, part, static_cast<float *>(y), m, n, slices, ldy);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

}  // namespace lhip
