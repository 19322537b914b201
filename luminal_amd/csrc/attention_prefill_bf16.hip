// Causal grouped-query attention for a block of prompt tokens on the bf16 matrix cores.
//
// Same operator and work split as attention_prefill.hip (one workgroup per (KV head, 32 query tokens), one wave
// per query head of the group, 32-key tiles staged once in LDS for all of them), for callers whose attention
// output feeds a bf16 GEMM anyway: Q (pre-scaled), K, V and the soft-max weights are rounded to bf16 for
// v_mfma_f32_32x32x16_bf16, sums and the soft-max itself stay f32.  Sixteen MFMAs per wave and tile instead of 128.
//
// Per wave and key tile, lane = (c, h), c = lane % 32, h = lane / 32:
//   S^T = K Q^T   : A = K tile (row = key c, 8 consecutive head-dim elements per step and lane half, 16-byte LDS
//                   reads of the bf16 K rows), B = Q^T from registers.  Result layout as in the f32 kernel: lane
//                   (c, h) holds query c, keys 8*(v/4) + 4*h + v%4, v = 0..15.
//   O^T += V^T P^T: B = P^T is those registers, converted: MFMA step s (16 keys) takes registers 8s .. 8s+7, i.e.
//                   lane half h supplies keys 16s + 8a + 4h + b (a = 0..1, b = 0..3) in slots 4a + b.  A = V^T
//                   must present the same keys in the same slots, so V is stored transposed in LDS with bits 2
//                   and 3 of the key index swapped: a lane's eight keys are then one 16-byte read.
//
// What bounds it is the serial chain of a tile in a wave (scores -> maximum -> weights -> O), with one or two waves per
// SIMD to hide it: the longest query block's tiles one after the other are the operator's time.  So the scores of the NEXT
// tile are computed between the exponentials of this one (one matrix step beside two weights; K is staged a tile further
// ahead than V), the exponentials are the hardware's exp2, a tile's sum is a dot product of the rounded weights with ones,
// only the tiles that reach past a block's first query are masked, the accumulators are rescaled only where a maximum
// moved, and the longest query blocks start first.
// Measured (32 query heads on 8, head_dim 128): 300 / 512 / 1024 / 2000 tokens from position 0 in 14.3 / 20.6 / 35.5 / 72.6 us
// (23.0 / 35.6 / 66.1 / 154.7 before), 1000 tokens behind 3000 in 120 (234).  Of the 72.6, 20 are the staging (f32 loads 13,
// conversion and LDS stores 7) and 10 the rescaling.  Not kept: the keys of a block shared by two waves a head (each wave's
// weights are then rounded against its own maximum and not the row's).
#include <type_traits>
#include <utility>

#include "common.h"

namespace lhip {

typedef float pv16f __attribute__((ext_vector_type(16)));
typedef __bf16 pbf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 pbf16x4 __attribute__((ext_vector_type(4)));
typedef float pf32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 pbf16x2 __attribute__((ext_vector_type(2)));

constexpr int kBfTileK = 32;  // keys per tile
constexpr int kBfTileQ = 32;  // queries per workgroup
constexpr float kLog2e = 1.44269504088896340736f;
// Bytes per row of V^T in LDS (four 16-byte granules used).  Five granules a row spread the operand reads of 16 rows over
// all banks; the granule is further exchanged by the row's bits 4 and 5, so that the transposing writes (rows 4 apart from
// lane to lane) meet a bank twice and not eight times.
constexpr int kBfVPitch = 80;

// Two waves per SIMD at least: with the registers of one, the compiler keeps the accumulators in the other half of the file
// and moves all of them back and forth in every tile.
template <int G, int HD>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(2))) void attention_prefill_bf16_kernel(
    const float *__restrict__ qkv, const float *__restrict__ k_cache, const float *__restrict__ v_cache, __bf16 *__restrict__ out,
    const int *__restrict__ pos_dev, int tokens, int hkv, int max_seq) {
    constexpr int THREADS = 64 * G;
    constexpr int KPITCH = HD * 2 + 16;            // bytes: 16 rows of a read start in different banks
    constexpr int STEPS = HD / 16;                 // MFMA steps of S^T
    constexpr int OB = HD / 32;                    // 32-row blocks of O^T
    constexpr int K_F4 = kBfTileK * HD / 4;        // float4 of a K tile
    constexpr int KLD = K_F4 / THREADS;            // float4 of K per thread and tile
    constexpr int V_UNITS = (kBfTileK / 4) * (HD / 4);  // (4 keys) x (4 head-dim) blocks of a V tile
    constexpr int VU = V_UNITS >= THREADS ? V_UNITS / THREADS : 1;
    static_assert(K_F4 % THREADS == 0 && KLD >= 1 && KLD <= 8 && (V_UNITS % THREADS == 0 || V_UNITS < THREADS), "staging split");
    constexpr int K_BYTES = kBfTileK * KPITCH, V_BYTES = HD * kBfVPitch;
    __shared__ __attribute__((aligned(16))) unsigned char k_s[2][K_BYTES];
    __shared__ __attribute__((aligned(16))) unsigned char v_s[2][V_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, h = lane >> 5;
    const int kvh = blockIdx.x, qb = gridDim.y - 1 - blockIdx.y;  // the longest query blocks first
    const int hq = hkv * G;
    const int pos0 = *pos_dev;
    const int q0 = qb * kBfTileQ;
    const int head = kvh * G + wave;
    const int my_q = q0 + c;
    const int my_pos = pos0 + my_q;
    const int n_keys = min(pos0 + min(tokens, q0 + kBfTileQ), max_seq);
    const int n_tiles = (n_keys + kBfTileK - 1) / kBfTileK;
    const float inv_sqrt = 1.0f / sqrtf(static_cast<float>(HD));

    // ---- Q^T operand of every step: Q[my_q][16 step + 8 h .. + 8) / sqrt(HD), bf16
    pbf16x8 qv[STEPS];
    {
        const float *qrow = qkv + (static_cast<size_t>(min(my_q, tokens - 1)) * (hq + 2 * hkv) + head) * HD + 8 * h;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const float4 a = *reinterpret_cast<const float4 *>(qrow + 16 * s), b = *reinterpret_cast<const float4 *>(qrow + 16 * s + 4);
            qv[s] = pbf16x8{static_cast<__bf16>(a.x * inv_sqrt), static_cast<__bf16>(a.y * inv_sqrt),
                            static_cast<__bf16>(a.z * inv_sqrt), static_cast<__bf16>(a.w * inv_sqrt),
                            static_cast<__bf16>(b.x * inv_sqrt), static_cast<__bf16>(b.y * inv_sqrt),
                            static_cast<__bf16>(b.z * inv_sqrt), static_cast<__bf16>(b.w * inv_sqrt)};
        }
    }

    // ---- tile staging: global f32 -> registers -> bf16 in LDS (K row-major, V transposed)
    const float4 *kc4 = reinterpret_cast<const float4 *>(k_cache) + static_cast<size_t>(kvh) * max_seq * (HD / 4);
    const float4 *vc4 = reinterpret_cast<const float4 *>(v_cache) + static_cast<size_t>(kvh) * max_seq * (HD / 4);
    const bool v_thread = V_UNITS >= THREADS || tid < V_UNITS;  // THREADS > V_UNITS: the first V_UNITS threads transpose V
    // tiles in flight: two, where the registers are there for them (one step is shorter than a trip to memory under load)
    constexpr int SETS = G == 2 ? 1 : 2;
    pf32x4 kst[SETS][KLD], vst[SETS][VU][4];
    // (rows past the end come as zeros, by the bounds check of the buffer loads; their keys are masked)
    auto tile_of = [&](const float4 *base, int t) __attribute__((always_inline)) {
        const int rows = __builtin_amdgcn_readfirstlane(max(min(n_keys - t * kBfTileK, kBfTileK), 0));
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(base + static_cast<size_t>(t) * (kBfTileK * HD / 4)), 0,
                                                 rows * HD * 4, 0x00020000);
    };
    auto load_k = [&](pf32x4 (&st)[KLD], int t) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t tile = tile_of(kc4, t);
#pragma unroll
        for (int i = 0; i < KLD; ++i)
            st[i] = __builtin_bit_cast(pf32x4, __builtin_amdgcn_raw_buffer_load_b128(tile, (tid + i * THREADS) * 16, 0, 0));
    };
    auto load_v = [&](pf32x4 (&st)[VU][4], int t) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t tile = tile_of(vc4, t);
        // (no branch around the loads: the wait for K would have to assume them skipped, i.e. wait for younger loads too)
#pragma unroll
        for (int u = 0; u < VU; ++u) {
            const int unit = tid * VU + u;
            const int kg = unit / (HD / 4), dq = unit - kg * (HD / 4);
            const int off = v_thread ? 4 * kg * (HD * 4) + dq * 16 : kBfTileK * HD * 4;  // else past the bounds
#pragma unroll
            for (int i = 0; i < 4; ++i)
                st[u][i] = __builtin_bit_cast(pf32x4, __builtin_amdgcn_raw_buffer_load_b128(tile, off + i * (HD * 4), 0, 0));
        }
    };
    auto store_k = [&](pf32x4 (&st)[KLD], int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KLD; ++i) {
            const int f = tid + i * THREADS;
            const int row = f / (HD / 4), col = f - row * (HD / 4);
            asm volatile("" : "+v"(st[i]));  // (holds the conversion, and so the wait for the load, here)
            const pbf16x4 w = {static_cast<__bf16>(st[i].x), static_cast<__bf16>(st[i].y), static_cast<__bf16>(st[i].z),
                               static_cast<__bf16>(st[i].w)};
            *reinterpret_cast<pbf16x4 *>(&k_s[buf][row * KPITCH + col * 8]) = w;
        }
    };
    auto store_v = [&](pf32x4 (&st)[VU][4], int buf) __attribute__((always_inline)) {
        if (v_thread) {
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int unit = tid * VU + u;
                const int kg = unit / (HD / 4), dq = unit - kg * (HD / 4);
                const int key = 4 * kg;  // first of four consecutive keys; V^T column = key with bits 2 and 3 swapped
                const int pos = (key & 16) | ((key & 4) << 1) | ((key & 8) >> 1);
                asm volatile("" : "+v"(st[u][0]), "+v"(st[u][1]), "+v"(st[u][2]), "+v"(st[u][3]));
#pragma unroll
                for (int dd = 0; dd < 4; ++dd) {
                    const pbf16x4 w = {static_cast<__bf16>(st[u][0][dd]), static_cast<__bf16>(st[u][1][dd]),
                                       static_cast<__bf16>(st[u][2][dd]), static_cast<__bf16>(st[u][3][dd])};
                    *reinterpret_cast<pbf16x4 *>(&v_s[buf][(4 * dq + dd) * kBfVPitch + (((pos >> 3) ^ (dq >> 2)) & 3) * 16 + (pos & 7) * 2]) = w;
                }
            }
        }
    };

    pv16f o_acc[OB], s_acc;
#pragma unroll
    for (int j = 0; j < OB; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) o_acc[j][v] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    pv16f zero;
#pragma unroll
    for (int v = 0; v < 16; ++v) zero[v] = 0.f;
    auto k_step = [&](int buf, int s, const pv16f &acc) __attribute__((always_inline)) {
        const unsigned char *krow = &k_s[buf][c * KPITCH + h * 16];
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const pbf16x8 *>(krow + s * 32), qv[s], acc, 0, 0, 0);
    };

    {
        pf32x4 first[KLD];
        load_k(first, 0);
        load_v(vst[0], 0);
        load_k(kst[0], 1);
        store_k(first, 0);
        store_v(vst[0], 0);
        store_k(kst[0], 1);
    }
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
        load_k(kst[i], 2 + i);
        load_v(vst[i], 1 + i);
    }
    __syncthreads();
    s_acc = zero;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) s_acc = k_step(0, s, s_acc);
    __syncthreads();
    // Tile t: s_acc holds its scores, LDS K of tile t + 1 and V of tile t, the staging registers (in flight) K of t + 2 and V of
    // t + 1, which go into the buffers that every wave left at the last barrier, and with two sets those of the tile behind.
    auto step = [&](int t, auto masked, auto parity) __attribute__((always_inline)) {
        constexpr int buf = decltype(parity)::value, set = buf % SETS;  // buf = t & 1
        store_k(kst[set], buf);
        store_v(vst[set], buf ^ 1);
        load_k(kst[set], t + 2 + SETS);
        load_v(vst[set], t + 1 + SETS);
        // ---- causal mask, running max
        if constexpr (decltype(masked)::value) {
            const int seen = min(my_pos, n_keys - 1) - t * kBfTileK - 4 * h;
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (8 * (v >> 2) + (v & 3) > seen) s_acc[v] = -INFINITY;
        }
        float tmax = s_acc[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) tmax = fmaxf(tmax, s_acc[v]);
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
            tmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        }
        // finite from the first tile on: key 0 is visible to every query.  Where no query's maximum moved, the factor is 1.
        if (__any(!(tmax <= m_run))) {
            const float m_new = fmaxf(m_run, tmax);
            const float corr = __builtin_amdgcn_exp2f((m_run - m_new) * kLog2e);
            l_run *= corr;
            m_run = m_new;
#pragma unroll
            for (int j = 0; j < OB; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) o_acc[j][v] *= corr;
        }
        // ---- weights, rounded to bf16 once, and the running sum (this lane's keys only, until the end) of the rounded values:
        // the result stays a convex combination of the (rounded) V rows.  Beside them the scores of the next tile.
        const float m_scaled = m_run * kLog2e;
        pbf16x8 pb[2];
        pv16f s_next = zero;
        auto weights = [&](int v) __attribute__((always_inline)) {
            const pbf16x2 w = {static_cast<__bf16>(__builtin_amdgcn_exp2f(fmaf(s_acc[v], kLog2e, -m_scaled))),
                               static_cast<__bf16>(__builtin_amdgcn_exp2f(fmaf(s_acc[v + 1], kLog2e, -m_scaled)))};
            pb[v >> 3][v & 7] = w[0];
            pb[v >> 3][(v & 7) + 1] = w[1];
            l_run = __builtin_amdgcn_fdot2_f32_bf16(w, pbf16x2{static_cast<__bf16>(1.f), static_cast<__bf16>(1.f)}, l_run, false);
        };
        constexpr int PER = 16 / STEPS;  // weights beside a matrix step
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            s_next = k_step(buf ^ 1, s, s_next);
#pragma unroll
            for (int v = s * PER; v < (s + 1) * PER; v += 2) weights(v);
            __builtin_amdgcn_sched_barrier(0x3f4);  // the matrix steps and the weights keep this order; loads, stores, scalars move
        }
        // ---- O^T += V^T P^T
        const unsigned char *vrow = &v_s[buf][c * kBfVPitch + (h ^ (c >> 4)) * 16];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < OB; ++j)
                o_acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    *reinterpret_cast<const pbf16x8 *>(vrow + j * 32 * kBfVPitch + (s ^ (j & 1)) * 32), pb[s], o_acc[j], 0, 0, 0);
        s_acc = s_next;
        __syncthreads();
    };
    // only the tiles that reach past the block's first query need the mask
    const int whole = min((pos0 + q0 + 1) / kBfTileK, n_tiles);
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    int t = 0;
    for (; t + 1 < whole; t += 2) {
        step(t, std::false_type{}, even);
        step(t + 1, std::false_type{}, odd);
    }
    if (t < whole) {
        step(t, std::false_type{}, even);
        if (++t < n_tiles) step(t++, std::true_type{}, odd);
    }
    for (; t < n_tiles; t += 2) {
        step(t, std::true_type{}, even);
        if (t + 1 < n_tiles) step(t + 1, std::true_type{}, odd);
    }

    // ---- out[q][head*HD + 32 j + 8 a + 4 h + b] = O^T[..][q] / l: four consecutive head-dim elements per store
    const auto l_sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
    if (my_q < tokens) {
        const float inv = 1.0f / (__uint_as_float(l_sw[0]) + __uint_as_float(l_sw[1]));
        __bf16 *orow = out + (static_cast<size_t>(my_q) * hq + head) * HD;
#pragma unroll
        for (int j = 0; j < OB; ++j)
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const pbf16x4 w = {static_cast<__bf16>(o_acc[j][4 * a] * inv), static_cast<__bf16>(o_acc[j][4 * a + 1] * inv),
                                   static_cast<__bf16>(o_acc[j][4 * a + 2] * inv), static_cast<__bf16>(o_acc[j][4 * a + 3] * inv)};
                *reinterpret_cast<pbf16x4 *>(orow + 32 * j + 8 * a + 4 * h) = w;
            }
    }
}

// Launches the kernel for the head shapes it is built for; false if (q_heads / kv_heads, head_dim) is not one.
bool attention_prefill_bf16_launch(const float *qkv, const float *kc, const float *vc, void *out, const int *pos, int tokens,
                                   int q_heads, int kv_heads, int head_dim, int max_seq, hipStream_t s) {
    if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return false;
    const int g = q_heads / kv_heads;
    const dim3 grid(static_cast<unsigned>(kv_heads), static_cast<unsigned>((tokens + kBfTileQ - 1) / kBfTileQ));
    if (kv_heads > 65535 || grid.y > 65535) return false;
#define LHIP_CASE(G, HD)                                                                                              \
    if (g == G && head_dim == HD) {                                                                                   \
        hipLaunchKernelGGL((attention_prefill_bf16_kernel<G, HD>), grid, dim3(64 * G), 0, s, qkv, kc, vc,             \
                           static_cast<__bf16 *>(out), pos, tokens, kv_heads, max_seq);                               \
        return true;                                                                                                  \
    }
    LHIP_CASE(2, 64) LHIP_CASE(4, 64) LHIP_CASE(8, 64)
    LHIP_CASE(2, 128) LHIP_CASE(4, 128) LHIP_CASE(8, 128)
#undef LHIP_CASE
    return false;
}

}  // namespace lhip
