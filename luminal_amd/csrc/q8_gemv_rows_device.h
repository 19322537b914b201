// Device code of the Q8_0 matvec for several activation rows (host side: q8_gemv_rows.hip).
#pragma once

#include "q8_gemv_device.h"

namespace lhip {

// How the activations lie in LDS: f32 as floats, f16 as halves (v_fma_mix takes a half as an operand, so they are read in half
// the LDS time and converted for nothing).  A piece is 16 bytes: `per` pieces hold a lane's 16 activations of a slice, piece j of
// lane l at  slice * per * 64 + j * 64 + l, so that the reads of a wave are contiguous.
template <typename XT>
struct RowsX;
template <>
struct RowsX<float> {
    static constexpr int kPer = 4;  // pieces per lane and slice
    typedef float4 Piece;
    static __device__ __forceinline__ Piece load(const float *x, int i) { return reinterpret_cast<const float4 *>(x)[i]; }
    static __device__ __forceinline__ float fma16(const float (&c)[16], const Piece (&x)[kPer]) {
        float s = c[0] * x[0].x;
        s = fmaf(c[1], x[0].y, s);
        s = fmaf(c[2], x[0].z, s);
        s = fmaf(c[3], x[0].w, s);
#pragma unroll
        for (int j = 1; j < 4; ++j) {
            s = fmaf(c[4 * j], x[j].x, s);
            s = fmaf(c[4 * j + 1], x[j].y, s);
            s = fmaf(c[4 * j + 2], x[j].z, s);
            s = fmaf(c[4 * j + 3], x[j].w, s);
        }
        return s;
    }
};
template <>
struct RowsX<__half> {
    static constexpr int kPer = 2;
    typedef uint4 Piece;
    // (rows of halves are 8-byte aligned, not 16)
    static __device__ __forceinline__ Piece load(const __half *x, int i) {
        const uint2 a = reinterpret_cast<const uint2 *>(x)[2 * i], b = reinterpret_cast<const uint2 *>(x)[2 * i + 1];
        return make_uint4(a.x, a.y, b.x, b.y);
    }
    static __device__ __forceinline__ float half_of(uint32_t w, int i) {
        const __half2 h = *reinterpret_cast<const __half2 *>(&w);
        return i ? __high2float(h) : __low2float(h);
    }
    static __device__ __forceinline__ float fma16(const float (&c)[16], const Piece (&x)[kPer]) {
        const uint32_t w[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
        float s = c[0] * half_of(w[0], 0);
#pragma unroll
        for (int i = 1; i < 16; ++i) s = fmaf(c[i], half_of(w[i / 2], i & 1), s);
        return s;
    }
};

// y (m, n) = x (m, k) W^T by matvecs of MR activation rows each: grid.y passes of MR rows, in each of which a wave walks row groups
// of R weight rows as q8_gemv_pipe_body does, converts a code once for all MR rows and adds up every row's products in that
// kernel's order, so a row's result is bit for bit that of a call with this row alone.
//
// Bound: the weight stream, up to some rows; the vector pipe takes (16 + 16 MR) instructions per 16 codes of a lane, the LDS
// MR * kPer reads per R * 16 codes.
//
// RAG: K is no multiple of S * 1024.  The activations are zero behind K, the lanes that lie there read the row's first bytes
// again and take a scale of zero.
template <int R, int S, int W, int MR, bool RAG, typename XT>
__global__ __launch_bounds__(W * 64) void q8_gemv_rows_kernel(const int8_t *__restrict__ qs, const unsigned short *__restrict__ ds,
                                                              const XT *__restrict__ x, XT *__restrict__ y, int m, int n, int k,
                                                              int grid_blocks,
                                                              unsigned inv_groups) {
    typedef RowsX<XT> X;
    typedef typename X::Piece Piece;
    constexpr int kPer = X::kPer;
    constexpr int kStage = 8;  // pieces a thread stages from registers, requested ahead of the weights
    extern __shared__ uint4 staged_lds[];
    Piece *xs = reinterpret_cast<Piece *>(staged_lds);
    const unsigned lane = threadIdx.x & 63u;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_global = blockIdx.x * W + wave;
    const int total_waves = grid_blocks * W;
    const int m0 = blockIdx.y * MR;
    const int nblk = k >> 5;

    const int n_groups = (n + R - 1) / R;
    const int chunks = RAG ? (k + S * 1024 - 1) / (S * 1024) : k / (S * 1024);
    const int my_groups = wave_global < n_groups ? (n_groups - wave_global + total_waves - 1) / total_waves : 0;
    const int T = my_groups * chunks;
    const int row_pieces = chunks * S * kPer * 64;  // of one staged row of activations

    // Group i of 64 pieces of the staged rows (wave-uniform): row i / row_groups, of whose groups it is slice * kPer + j.
    const int row_groups = chunks * S * kPer, groups_all = MR * row_groups;
    auto piece = [&](int i) {
        const int row = MR == 1 ? 0 : static_cast<int>(static_cast<unsigned>(i) * inv_groups >> 16);
        const int p = MR == 1 ? i : i - row * row_groups;
        const int slice = p / kPer, j = p % kPer;
        const bool in = !RAG || slice * 1024 + static_cast<int>(lane) * 16 < k;
        Piece v = X::load(x + static_cast<size_t>(min(m0 + row, m - 1)) * k, in ? slice * (kPer * 64) + static_cast<int>(lane) * kPer + j : 0);
        if (RAG && !in) v = Piece{};
        return v;
    };
    Piece xr[kStage];
#pragma unroll
    for (int j = 0; j < kStage; ++j) xr[j] = piece(wave + j * W < groups_all ? wave + j * W : 0);
    __builtin_amdgcn_sched_barrier(0);

    struct Buf {
        u32x4 q[S][R];
        unsigned d[S][R];
    } a, b;
    auto load = [&](Buf &buf, int gg, int cc, bool live) {
        const unsigned kbase = live ? static_cast<unsigned>(cc) * (S * 1024u) : 0u;
        unsigned qoff[S], doff[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const unsigned ko = s * 1024u + lane * 16u;
            const bool in = live && (!RAG || kbase + ko < static_cast<unsigned>(k));
            qoff[s] = in ? kbase + ko : 0u;
            doff[s] = in ? ((kbase + ko) >> 5) * 2u : 0u;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = live ? min(gg * R + r, n - 1) : 0;
            const char *qrow = reinterpret_cast<const char *>(qs) + static_cast<size_t>(row) * k;
            const char *drow = reinterpret_cast<const char *>(ds) + static_cast<size_t>(row) * nblk * 2;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                buf.q[s][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(qrow + qoff[s]));
                buf.d[s][r] = __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(drow + doff[s]));
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) asm volatile("" ::"v"(qoff[s]), "v"(doff[s]));
    };
    float acc[MR][R];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[i][r] = 0.f;
    auto compute = [&](Buf &buf, int cc) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int slice = cc * S + s;
            float c[R][16], d[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                asm volatile("" : "+v"(buf.q[s][r]), "+v"(buf.d[s][r]));
#pragma unroll
                for (int i = 0; i < 16; ++i) c[r][i] = sb(buf.q[s][r][i / 4], i & 3);
                d[r] = __half2float(__ushort_as_half(static_cast<unsigned short>(buf.d[s][r])));
                if (RAG && slice * 1024 + static_cast<int>(lane) * 16 >= k) d[r] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < MR; ++i) {
                const Piece *xp = xs + i * row_pieces + slice * (kPer * 64) + lane;
                Piece xv[kPer];
#pragma unroll
                for (int j = 0; j < kPer; ++j) xv[j] = xp[j * 64];
#pragma unroll
                for (int r = 0; r < R; ++r) acc[i][r] = fmaf(X::fma16(c[r], xv), d[r], acc[i][r]);
            }
        }
    };
    int t = 0, g = wave_global, c = 0, g1 = wave_global, c1 = 0;
    auto next = [&]() {
        if (++c1 == chunks) {
            c1 = 0;
            g1 += total_waves;
        }
    };
    next();
    load(a, T > 0 ? wave_global : 0, 0, T > 0);
    __builtin_amdgcn_sched_barrier(0);
    load(b, g1, c1, T > 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kStage; ++j)
        if (wave + j * W < groups_all) xs[(wave + j * W) * 64 + lane] = xr[j];
    for (int i = wave + kStage * W; i < groups_all; i += W) xs[i * 64 + lane] = piece(i);
    __syncthreads();
    if (T == 0) return;

    // Whether a step was the wave's last; otherwise on to the next.
    auto done = [&]() {
        if (c == chunks - 1) {
            float out = 0.f;
#pragma unroll
            for (int i = 0; i < MR; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float s = wave_sum(acc[i][r]);
                    if (lane == static_cast<unsigned>(i * R + r)) out = s;
                    acc[i][r] = 0.f;
                }
            const int row = m0 + static_cast<int>(lane) / R, col = g * R + static_cast<int>(lane) % R;
            if (lane < static_cast<unsigned>(MR * R) && row < m && col < n) store_y(y + static_cast<size_t>(row) * n, col, out);
        }
        if (++t >= T) return true;
        g = g1;
        c = c1;
        next();
        return false;
    };
    compute(a, c);
    if (done()) return;
    while (true) {
        load(a, g1, c1, t + 1 < T);
        __builtin_amdgcn_sched_barrier(0);
        compute(b, c);
        if (done()) return;
        load(b, g1, c1, t + 1 < T);
        __builtin_amdgcn_sched_barrier(0);
        compute(a, c);
        if (done()) return;
    }
}

}  // namespace lhip
