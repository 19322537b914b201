// Causal grouped-query attention for a block of prompt tokens on the f32 matrix cores.
//
// Same operator as attention_kernel in llama_ops.hip (examples/llama/src/model.rs:112-139: scores = q.k/sqrt(hd),
// causal mask, softmax, times V, over the KV cache that already holds the new tokens), for many query tokens:
// a flash-attention sweep with v_mfma_f32_16x16x4_f32, so inputs, products and sums stay f32 and the result meets
// the same bar as the scalar kernel.
//
// Work split: one workgroup per (KV head, block of 16 query tokens); its G waves are the G query heads that share
// the KV head, so they walk the same key tiles (32 keys each, staged once in LDS for all of them) under the same
// causal limit.
//
// Per wave and key tile, with lane = (r, g), r = lane % 16, g = lane / 16:
//   S^T = K Q^T   (two halves of 16 keys x 16 queries): A = K, B = Q^T.  The summation index of an MFMA step is free to name
//                 any head-dim element as long as A and B agree; lane group g takes elements 16*j + 4*g + e, e = 0..3, so a
//                 lane keeps HD/4 floats of Q in registers for the whole sweep and its K values come from LDS as 16-byte reads.
//                 Result layout: lane (r, g) holds query r, keys 16*kh + 4*g + v, v = 0..3 - a query's
//                 scores are in four lanes' registers, so the running max and sum need two exchanges per tile and no LDS.
//   O^T += V^T P^T (HD x 16 queries): B = P^T is exactly the score registers (step (kh, v) uses key 16*kh + 4*g + v of lane
//                 group g); A = V^T: lane (r, g) reads V[key][OB*r ..] as 16-byte LDS reads for the OB output blocks of 16
//                 rows, i.e. output row q of block j is head-dim OB*q + j.
// The accumulators of O^T have the query in the lane as well, so rescaling by exp(m_old - m_new) is per lane.
//
// What bounds it: the matrix pipe (128 steps of 32 cycles a tile and wave at HD = 128) and, for a prompt of a few hundred tokens, the
// serial chain of the last block's tiles, with most of the chip idle.  Hence blocks of 16 queries (with v_mfma_f32_32x32x2 and blocks of 32,
// as before, twice the chain on half the workgroups), operands requested from LDS ahead of their use (the compiler waited
// for each where it was read: 49 us and not 34 at 300 tokens), two buffers and one barrier a tile (but see BUFS).  32 heads on 8 of 128, us, before ->
// now: 16 tokens 11.9 -> 6.7, 100 31 -> 14.8, 300 69 -> 34, 512 109 -> 53, 1000 207 -> 129, 2000 575 -> 350 (94 TFLOP/s of 157).
#include "common.h"

namespace lhip {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kPfTileK = 32;  // keys per tile
constexpr int kPfTileQ = 16;  // queries per workgroup

template <int G, int HD, typename OutT>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(1, 2))) void attention_prefill_kernel(
    const float *__restrict__ qkv, const float *__restrict__ k_cache, const float *__restrict__ v_cache, OutT *__restrict__ out,
    const int *__restrict__ pos_dev, int tokens, int hkv, int max_seq) {
    constexpr int THREADS = 64 * G;
    constexpr int PART = HD / 4;           // head-dim elements per lane group
    constexpr int OB = HD / 16;            // output blocks of 16 rows of O^T
    constexpr int TILE_F4 = kPfTileK * HD / 4;
    constexpr int LD = TILE_F4 / THREADS;  // float4 per thread and tile and matrix
    static_assert(TILE_F4 % THREADS == 0 && THREADS % (HD / 4) == 0, "whole rounds of whole rows");
    constexpr bool PREFETCH = LD <= 4;     // keep the next tile in registers during the sweep of this one
    // Two buffers of a tile, and one for a single wave: it waits for nobody, so the second gives it nothing, and with twice the LDS half
    // the waves fit a CU (32 heads on 32 of 128, two buffers -> one, us: 300 tokens 39 -> 37, 1000 232 -> 150, 2000 876 -> 517; two waves,
    // 32 on 16: 1000 tokens 112 <- 141).
    constexpr int BUFS = G == 1 ? 1 : 2;
    static_assert(BUFS == 2 || !PREFETCH, "a tile requested ahead is stored in the other buffer");
    // 16-byte piece p of a K row lies at p ^ (key % 16), of a V row at p ^ (key / 4 % 2), which gives the operand reads below
    // 16 lanes on 16 different slots.
    __shared__ __attribute__((aligned(16))) float k_s[BUFS][kPfTileK * HD];
    __shared__ __attribute__((aligned(16))) float v_s[BUFS][kPfTileK * HD];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int block = static_cast<int>(blockIdx.x / static_cast<unsigned>(hkv)), kvh = static_cast<int>(blockIdx.x) - block * hkv;
    const int qb = (tokens + kPfTileQ - 1) / kPfTileQ - 1 - block;  // the longest blocks first
    const int hq = hkv * G;
    const int pos0 = *pos_dev;
    const int q0 = qb * kPfTileQ;
    const int head = kvh * G + wave;
    const int my_q = q0 + r;
    const int my_pos = pos0 + my_q;
    const int n_keys = min(pos0 + min(tokens, q0 + kPfTileQ), max_seq);
    const int n_tiles = (n_keys + kPfTileK - 1) / kPfTileK;
    const float inv_sqrt = 1.0f / sqrtf(static_cast<float>(HD));

    float qreg[PART];
    {
        const float *qrow = qkv + (static_cast<size_t>(min(my_q, tokens - 1)) * (hq + 2 * hkv) + head) * HD + g * 4;
#pragma unroll
        for (int j = 0; j < PART / 4; ++j) {
            const v4f t = reinterpret_cast<const v4f *>(qrow)[4 * j];
            qreg[4 * j] = t.x * inv_sqrt; qreg[4 * j + 1] = t.y * inv_sqrt;
            qreg[4 * j + 2] = t.z * inv_sqrt; qreg[4 * j + 3] = t.w * inv_sqrt;
        }
    }

    const v4f *kc4 = reinterpret_cast<const v4f *>(k_cache) + static_cast<size_t>(kvh) * max_seq * (HD / 4);
    const v4f *vc4 = reinterpret_cast<const v4f *>(v_cache) + static_cast<size_t>(kvh) * max_seq * (HD / 4);
    // Piece i of a thread is row i * STEP + row0, column col0 of a tile.
    constexpr int STEP = THREADS / (HD / 4), NST = PREFETCH ? LD : 1;
    const int row0 = tid / (HD / 4), col0 = tid % (HD / 4);
    auto k_at = [](int row, int col) { return row * HD + (col ^ (row & 15)) * 4; };
    auto v_at = [](int row, int col) { return row * HD + (col ^ ((row >> 2) & 1)) * 4; };
    auto source = [&](int t, int i) { return static_cast<size_t>(min(t * kPfTileK + i * STEP + row0, n_keys - 1)) * (HD / 4) + col0; };  // rows past the end repeat the last key (masked)
    v4f kst[NST], vst[NST];
    auto load_tile = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            kst[i] = kc4[source(t, i)];
            vst[i] = vc4[source(t, i)];
        }
    };
    auto store_tile = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            *reinterpret_cast<v4f *>(&k_s[buf][k_at(i * STEP + row0, col0)]) = kst[i];
            *reinterpret_cast<v4f *>(&v_s[buf][v_at(i * STEP + row0, col0)]) = vst[i];
        }
    };
    auto copy_tile = [&](int t, int buf) {  // few waves: too many registers per thread to hold, copied through in pieces
        for (int i = 0; i < LD; ++i) {
            *reinterpret_cast<v4f *>(&k_s[buf][k_at(i * STEP + row0, col0)]) = kc4[source(t, i)];
            *reinterpret_cast<v4f *>(&v_s[buf][v_at(i * STEP + row0, col0)]) = vc4[source(t, i)];
        }
    };

    v4f o_acc[OB];
#pragma unroll
    for (int j = 0; j < OB; ++j) o_acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    if (PREFETCH) {
        load_tile(0);
        store_tile(0);
    } else {
        copy_tile(0, 0);
    }
    __syncthreads();
    for (int t = 0; t < n_tiles; ++t) {
        const float *kb = k_s[t % BUFS], *vb = v_s[t % BUFS];
        if (PREFETCH && t + 1 < n_tiles) load_tile(t + 1);
        v4f s_acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
        // Operands are requested from LDS ahead of their use; the fences hold that order.
        constexpr int NK = PART / 4, RING = 3;
        v4f kr[RING][2];
        auto read_k = [&](int j) __attribute__((always_inline)) {
            kr[j % RING][0] = *reinterpret_cast<const v4f *>(kb + k_at(r, 4 * j + g));
            kr[j % RING][1] = *reinterpret_cast<const v4f *>(kb + k_at(16 + r, 4 * j + g));
        };
#pragma unroll
        for (int j = 0; j < RING - 1; ++j) read_k(j);
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            if (j + RING - 1 < NK) read_k(j + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)
                    s_acc[kh] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[j % RING][kh][e], qreg[4 * j + e], s_acc[kh], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the first V operands come while the weights are formed
        constexpr int NV = 8 * (OB / 4);  // (key, four output blocks)
        v4f vr[RING];
        auto read_v = [&](int u) __attribute__((always_inline)) {
            const int step = u / (OB / 4), key = 16 * (step >> 2) + 4 * g + (step & 3);
            vr[u % RING] = *reinterpret_cast<const v4f *>(vb + v_at(key, OB / 4 * r + u % (OB / 4)));
        };
#pragma unroll
        for (int u = 0; u < RING - 1; ++u) read_v(u);
        float tmax = -INFINITY;
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int key = t * kPfTileK + 16 * kh + 4 * g + v;
                if (key > my_pos || key >= n_keys) s_acc[kh][v] = -INFINITY;
                tmax = fmaxf(tmax, s_acc[kh][v]);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float m_new = fmaxf(m_run, tmax);  // finite from the first tile on: key 0 is visible to every query
        const float corr = expf(m_run - m_new);
        float psum = 0.f;
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                s_acc[kh][v] = expf(s_acc[kh][v] - m_new);
                psum += s_acc[kh][v];
            }
        psum += __shfl_xor(psum, 16);
        psum += __shfl_xor(psum, 32);
        l_run = l_run * corr + psum;
        m_run = m_new;
#pragma unroll
        for (int j = 0; j < OB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) o_acc[j][v] *= corr;
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            if (u + RING - 1 < NV) read_v(u + RING - 1);
            __builtin_amdgcn_sched_barrier(0);
            const int step = u / (OB / 4), j0 = u % (OB / 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o_acc[j0 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[u % RING][e], s_acc[step >> 2][step & 3], o_acc[j0 + e], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (BUFS == 1) __syncthreads();  // the only buffer has been read
        if (t + 1 < n_tiles) {           // (of two, the other was last read a tile ago, behind a barrier)
            if (PREFETCH) store_tile((t + 1) % BUFS);
            else copy_tile(t + 1, (t + 1) % BUFS);
        }
        __syncthreads();
    }

    // ---- out[q][head*HD + OB*row + j] = O^T[j][row][q] / l, row = 4 g + v
    if (my_q < tokens) {
        const float inv = 1.0f / l_run;
        OutT *orow = out + (static_cast<size_t>(my_q) * hq + head) * HD;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            typedef OutT otx4 __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int j = 0; j < OB; j += 4) {
                otx4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = static_cast<OutT>(o_acc[j + e][v] * inv);
                *reinterpret_cast<otx4 *>(orow + OB * (4 * g + v) + j) = o;
            }
        }
    }
}

// Launcher used by lhip_attention_f32 for prompt-sized calls; false if this shape is not built.
bool attention_prefill_launch(const float *qkv, const float *kc, const float *vc, void *out, bool out_bf16, const int *pos,
                              int tokens, int q_heads, int kv_heads, int head_dim, int max_seq, hipStream_t s) {
    if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return false;
    const int g = q_heads / kv_heads;
    const int64_t blocks = (static_cast<int64_t>(tokens) + kPfTileQ - 1) / kPfTileQ * kv_heads;
    if (blocks > 0x7fffffff) return false;
    const dim3 grid(static_cast<unsigned>(blocks));
#define LHIP_CASE(G, HD)                                                                                            \
    if (g == G && head_dim == HD) {                                                                                 \
        if (out_bf16)                                                                                               \
            hipLaunchKernelGGL((attention_prefill_kernel<G, HD, __bf16>), grid, dim3(64 * G), 0, s, qkv, kc, vc,    \
                               static_cast<__bf16 *>(out), pos, tokens, kv_heads, max_seq);                         \
        else                                                                                                        \
            hipLaunchKernelGGL((attention_prefill_kernel<G, HD, float>), grid, dim3(64 * G), 0, s, qkv, kc, vc,     \
                               static_cast<float *>(out), pos, tokens, kv_heads, max_seq);                          \
        return true;                                                                                                \
    }
    LHIP_CASE(1, 64) LHIP_CASE(2, 64) LHIP_CASE(4, 64) LHIP_CASE(8, 64)
    LHIP_CASE(1, 128) LHIP_CASE(2, 128) LHIP_CASE(4, 128) LHIP_CASE(8, 128)
#undef LHIP_CASE
    return false;
}

}  // namespace lhip
