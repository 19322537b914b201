// Batch-1 decode attention with rotary embedding and KV append folded in.
//
// What the reference's graph does for one new token (examples/llama/src/model.rs:52-72
// rotary, :108-110 cache concat, :112-139 grouped-query attention) as ONE launch:
//   q, k of the new token are rotated; k and v are appended to the caches at *pos;
//   out[h] = softmax(q_h . K / sqrt(hd)) V over positions 0..*pos.
//
// Shape of the launch (short caches: attention_decode_short_kernel).  At batch 1 the work
// is a read of the two caches, which one workgroup per head cannot pull fast enough (it exposes several dependent memory round
// trips on a handful of CUs).  So the keys of each KV head are cut into `splits` ranges,
// one workgroup each (grid = kv_heads x splits, about one workgroup per CU), and the G
// query heads that share a KV head are served by the same workgroup, which therefore
// reads every cache row once.  Each workgroup writes its partial softmax state (max, sum,
// weighted V) to a workspace and a second, small kernel (one workgroup per query head) merges
// the partials into the output rows.  The bodies of both kernels live in
// attention_decode_device.h, which describes the work inside a workgroup.
#include "attention_decode_device.h"
#include "common.h"

namespace lhip {

template <int G, int HD>
__global__ __launch_bounds__(kDecThreads) void attention_decode_kernel(
    const float *__restrict__ qkv, float *__restrict__ k_cache, float *__restrict__ v_cache,
    const int *__restrict__ pos_dev, int hkv, int max_seq, float theta, int n_splits,
    float *__restrict__ ws_ml, float4 *__restrict__ ws_acc, bool few_ranges) {
    __shared__ AttnShared<G, HD> sh;
    attention_decode_body<G, HD, kDecThreads>(PlainIO{}, sh, blockIdx.x, blockIdx.y, qkv, k_cache, v_cache, *pos_dev, hkv,
                                                     max_seq, theta, n_splits, ws_ml, ws_acc, few_ranges);
}

// One workgroup per query head.
template <int G, int HD>
__global__ __launch_bounds__(kDecThreads) void attention_merge_kernel(float *__restrict__ out,
                                                                      const int *__restrict__ pos_dev, int max_seq,
                                                                      int n_splits, const float *__restrict__ ws_ml,
                                                                      const float4 *__restrict__ ws_acc, bool few_ranges) {
    __shared__ MergeShared sh;
    attention_merge_body<G, HD, kDecThreads>(PlainIO{}, sh, blockIdx.x, out, *pos_dev, max_seq, n_splits, ws_ml, ws_acc,
                                             nullptr, few_ranges);
}

// The same in one launch, for caches of at most kShortKeys positions: grid (query heads, kShortParts), a workgroup takes all keys of
// its head and a quarter of the output columns.  The arithmetic is that of the two launches, range by range and in their order
// (ranges of at most 16 keys, one tile each), so the results are theirs bit for bit.
//
// What bounds it: a launch and its dependent trips up to some 200 keys (6.2 us at 32), then what one CU reads, 28 bytes a clock:
// every key row is read by the workgroups of all its query heads and parts, 200 KB each at 300 keys, which up to some 400 keys costs
// less than the second launch.  The first 256 rows are asked for ahead of the position.  Eight layers in turn from a graph, two
// launches -> one, us: 32 heads on 8 of 128 at 32 / 100 / 200 / 300 / 400 / 510 keys 8.7 / 9.0 / 9.2 / 9.2 / 9.2 / 9.2 -> 6.2 / 6.4 /
// 6.9 / 7.9 / 9.0 / 9.3; 64 on 8 of 64 10.3 / 10.5 / 10.7 / 10.8 / 10.8 / 10.7 -> 6.1 / 6.4 / 6.7 / 7.1 / 7.7 / 8.0; 32 on 16 of 64 in a
// cache of 256 7.5 -> 5.5 to 6.1.
constexpr int kShortKeys = 512;
constexpr int kShortParts = 4;       // workgroups a head
constexpr int kShortThreads = 1024;
constexpr int kShortRange = 16;      // keys of a range, at most
constexpr int kShortRanges = 32;     // ranges, at most

template <int HD>
__global__ __launch_bounds__(kShortThreads) void attention_decode_short_kernel(
    const float *__restrict__ qkv, float *__restrict__ k_cache, float *__restrict__ v_cache, const int *__restrict__ pos_dev,
    int group, int hkv, int max_seq, float theta, int n_splits, float *__restrict__ out) {
    constexpr int C4 = HD / 4, PC = C4 / kShortParts;       // float4 columns of a row, of a part
    constexpr int KG = kDecThreads / C4;                    // key groups of a range in P.V (the two launches')
    constexpr int KPG = kShortRange / KG;                   // keys of one
    constexpr int J = HD / 32;                              // float4 per lane and key in the scores
    constexpr int KEYS = kShortThreads / 8, PASSES = kShortKeys / KEYS;
    constexpr int SLOTS = kShortRanges * KG * PC / kShortThreads;  // (range, key group, column) per thread
    constexpr int SG = kDecThreads / C4;                    // sub-groups of the merge
    static_assert(KPG * KG == kShortRange && SLOTS >= 1 && kShortRanges * kShortRange == kShortKeys, "shape");
    __shared__ float4 q_s[C4], knew[C4], vnew[C4];
    __shared__ float p_s[kShortRanges][kShortRange];
    __shared__ float m_s[kShortRanges], l_s[kShortRanges], w_s[kShortRanges];
    __shared__ float4 part[kShortRanges][KG][PC];
    __shared__ float4 acc_s[kShortRanges][PC];
    __shared__ float4 num_s[SG][PC];
    __shared__ float den_s[SG];

    const int tid = threadIdx.x;
    const int head = blockIdx.x, kvh = head / group, c0 = blockIdx.y * PC;
    const int hq = hkv * group;
    // ---- this head's q, the new key and value: they do not wait for the position
    const int pr = tid >> 1;  // of q and k: pairs 0 .. HD - 1, both lanes of two the same (one stores)
    const int prow = pr / (HD / 2), pj = pr - prow * (HD / 2);
    float2 xr = make_float2(0.f, 0.f);
    float4 vn = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tid < 2 * HD) {
        const lhip_f32x2 v = *as_global(reinterpret_cast<const lhip_f32x2 *>(qkv + static_cast<size_t>(prow == 0 ? head : hq + kvh) * HD + 2 * pj));
        xr = make_float2(v.x, v.y);
    }
    if (tid < C4) vn = ldg4(reinterpret_cast<const float4 *>(qkv + static_cast<size_t>(hq + hkv + kvh) * HD) + tid);

    // ---- cache rows, all of them; the row of the new position is replaced from LDS below.  The first keys' are asked for ahead of the
    // position too: what lies behind it is not used.
    const float4 *kc4 = reinterpret_cast<const float4 *>(k_cache) + static_cast<size_t>(kvh) * max_seq * C4;
    const float4 *vc4 = reinterpret_cast<const float4 *>(v_cache) + static_cast<size_t>(kvh) * max_seq * C4;
    const int sub = tid & 7, kslot = tid >> 3;
    float4 kreg[PASSES][J];
    auto load_k = [&](int i) __attribute__((always_inline)) {
        const float4 *row = kc4 + static_cast<size_t>(min(kslot + i * KEYS, max_seq - 1)) * C4;
#pragma unroll
        for (int j = 0; j < J; ++j) kreg[i][j] = ldg4(row + j * 8 + sub);
    };
    constexpr int EARLY = 2;
#pragma unroll
    for (int i = 0; i < EARLY; ++i) load_k(i);
    asm volatile("" ::: "memory");  // (they stay ahead of the wait for the position)
    const int pos = *pos_dev;
    const int n_keys = min(pos + 1, max_seq);
    const int chunk = (n_keys + n_splits - 1) / n_splits;
    const int n_active = (n_keys + chunk - 1) / chunk;
    const float inv_sqrt = 1.0f / sqrtf(static_cast<float>(HD));
#pragma unroll
    for (int i = EARLY; i < PASSES; ++i)
        if (i * KEYS < n_keys) load_k(i);  // uniform
    float4 vreg[SLOTS][KPG];
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        const int item = t * kShortThreads + tid, c = item % PC, kg = (item / PC) % KG, range = item / (PC * KG);
        const int k0 = min(range, n_active - 1) * chunk, k1 = min(n_keys, k0 + chunk);
        if (t * (kShortThreads / (PC * KG)) < n_active) {  // uniform
#pragma unroll
            for (int u = 0; u < KPG; ++u) {
                const int key = k0 + kg + KG * u;
                vreg[t][u] = ldg4(vc4 + static_cast<size_t>(key < k1 ? key : k0) * C4 + c0 + c);
            }
        }
    }
    // ---- rotary (adjacent pairs, the products rounded one by one; the operator of prompts, lhip_rope_kv_append_f32, fuses one of the two)
    if (tid < 2 * HD && (tid & 1) == 0) {
        const float2 sc = rope_sin_cos(theta, 2 * pj, HD, pos);
        const float sn = sc.x, cs = sc.y;
        float *dst = reinterpret_cast<float *>(prow == 0 ? q_s : knew);
        dst[2 * pj] = __fsub_rn(__fmul_rn(xr.x, cs), __fmul_rn(xr.y, sn));
        dst[2 * pj + 1] = __fadd_rn(__fmul_rn(xr.x, sn), __fmul_rn(xr.y, cs));
    }
    if (tid < C4) vnew[tid] = vn;
    if (tid < kShortKeys) p_s[tid / kShortRange][tid % kShortRange] = -INFINITY;
    __syncthreads();
    if (blockIdx.y == 0 && head == kvh * group && pos < max_seq && tid < C4) {  // one workgroup a KV head appends
        stg4(reinterpret_cast<float4 *>(k_cache) + (static_cast<size_t>(kvh) * max_seq + pos) * C4 + tid, knew[tid]);
        stg4(reinterpret_cast<float4 *>(v_cache) + (static_cast<size_t>(kvh) * max_seq + pos) * C4 + tid, vnew[tid]);
    }
    // ---- scores
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const int key = kslot + i * KEYS;
        if (i * KEYS < n_keys) {
            float d = 0.f;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const float4 qv = q_s[j * 8 + sub];
                const float4 kv = key == pos ? knew[j * 8 + sub] : kreg[i][j];
                d = fmaf(qv.x, kv.x, d);
                d = fmaf(qv.y, kv.y, d);
                d = fmaf(qv.z, kv.z, d);
                d = fmaf(qv.w, kv.w, d);
            }
            sum_of_eight_lanes<1>(&d, sub);
            const int range = key / chunk;
            if (sub == 0 && key < n_keys) p_s[range][key - range * chunk] = d * inv_sqrt;
        }
    }
    __syncthreads();
    // ---- softmax of every range: 16 lanes each
    if (tid < n_active * kShortRange) {
        const int range = tid / kShortRange, slot = tid % kShortRange;
        const float sv = p_s[range][slot];
        float m = sv;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        const float p = expf(sv - m);
        float sum = p;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        p_s[range][slot] = p;
        if (slot == 0) m_s[range] = m, l_s[range] = sum;
    }
    __syncthreads();
    // ---- weights of the ranges in the merge, by the last wave; P.V
    if (tid >= kShortThreads - 64) {
        const int range = tid & 63;
        const float m = m_s[min(range, n_active - 1)], mx = wave_max64(m);
        if (range < n_active) w_s[range] = dec_merge_weight(m, mx);
    }
#pragma unroll
    for (int t = 0; t < SLOTS; ++t) {
        const int item = t * kShortThreads + tid, c = item % PC, kg = (item / PC) % KG, range = item / (PC * KG);
        if (range < n_active) {
            const int k0 = range * chunk;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int u = 0; u < KPG; ++u) {
                const int key = k0 + kg + KG * u;
                const float w = p_s[range][kg + KG * u];
                // behind the new position, the last key, nothing is multiplied, not even by zero (as in attention_decode_body): the row
                // read there may be the new position's, which the workgroup that appends it has written by now or not
                const float4 v = key < pos ? vreg[t][u] : key == pos && key < min(n_keys, k0 + chunk) ? vnew[c0 + c] : make_float4(0.f, 0.f, 0.f, 0.f);
                a.x = fmaf(w, v.x, a.x); a.y = fmaf(w, v.y, a.y);
                a.z = fmaf(w, v.z, a.z); a.w = fmaf(w, v.w, a.w);
            }
            part[range][kg][c] = a;
        }
    }
    __syncthreads();
    // ---- merge: the ranges' sums, then a sub-group of ranges and a column per thread
    if (tid < n_active * PC) {
        const int c = tid % PC, range = tid / PC;
        float4 av = part[range][0][c];
#pragma unroll
        for (int q = 1; q < KG; ++q) {
            const float4 u = part[range][q][c];
            av.x += u.x; av.y += u.y; av.z += u.z; av.w += u.w;
        }
        acc_s[range][c] = av;
    }
    __syncthreads();
    if (tid < SG * PC) {
        const int c = tid % PC, sg = tid / PC;
        float den = 0.f;
        float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < kShortRanges / SG; ++u) {
            const int range = sg + u * SG;
            if (range < n_active) {
                const float wgt = w_s[range];
                const float4 av = acc_s[range][c];
                den = fmaf(l_s[range], wgt, den);
                num.x = fmaf(av.x, wgt, num.x); num.y = fmaf(av.y, wgt, num.y);
                num.z = fmaf(av.z, wgt, num.z); num.w = fmaf(av.w, wgt, num.w);
            }
        }
        num_s[sg][c] = num;
        if (c == 0) den_s[sg] = den;
    }
    __syncthreads();
    if (tid < PC) {
        float4 num = num_s[0][tid];
        float den = den_s[0];
#pragma unroll
        for (int q = 1; q < SG; ++q) {
            const float4 u = num_s[q][tid];
            num.x += u.x; num.y += u.y; num.z += u.z; num.w += u.w;
            den += den_s[q];
        }
        const float inv = 1.0f / den;
        stg4(reinterpret_cast<float4 *>(out) + static_cast<size_t>(head) * C4 + c0 + tid,
             make_float4(num.x * inv, num.y * inv, num.z * inv, num.w * inv));
    }
}

// out == nullptr: the partial states stay in the workspace for a consumer that merges them itself
// (lhip_q8_0_matvec_attn_merge_f32).
template <int G, int HD>
static lhip_status launch_decode(const float *qkv, float *kc, float *vc, float *out, const int *pos, int hkv, int max_seq,
                                 float theta, void *workspace, bool few, hipStream_t s) {
    const int splits = dec_splits(hkv);
    auto *base = static_cast<uint8_t *>(workspace);
    float *ml = reinterpret_cast<float *>(base);
    float4 *acc = reinterpret_cast<float4 *>(base + dec_ml_bytes(hkv, splits, G));
    // One launch where no range has more than its tile of 16 keys and all rows of the cache are taken at once.  By the cache and not by
    // the position, which a graph replays through; at 510 keys the two forms are level (above).
    if (out && !few && splits <= kShortRanges && max_seq <= kShortKeys && max_seq <= splits * kShortRange) {
        hipLaunchKernelGGL(attention_decode_short_kernel<HD>, dim3(static_cast<unsigned>(hkv * G), kShortParts), dim3(kShortThreads), 0,
                           s, qkv, kc, vc, pos, G, hkv, max_seq, theta, splits, out);
        LHIP_CHECK_LAUNCH();
        return LHIP_OK;
    }
    hipLaunchKernelGGL((attention_decode_kernel<G, HD>), dim3(static_cast<unsigned>(hkv), static_cast<unsigned>(splits)),
                       dim3(kDecThreads), 0, s, qkv, kc, vc, pos, hkv, max_seq, theta, splits, ml, acc, few);
    LHIP_CHECK_LAUNCH();
    if (!out) return LHIP_OK;
    hipLaunchKernelGGL((attention_merge_kernel<G, HD>), dim3(static_cast<unsigned>(hkv * G)), dim3(kDecThreads), 0, s, out,
                       pos, max_seq, splits, ml, acc, few);
    LHIP_CHECK_LAUNCH();
    return LHIP_OK;
}

lhip_status attention_decode_impl(const float *qkv_dev, float *k_cache_dev, float *v_cache_dev, float *out_dev,
                                  bool with_merge, bool few, const int32_t *pos_dev, int64_t q_heads, int64_t kv_heads,
                                  int64_t head_dim, int64_t max_seq, float theta, void *workspace_dev, void *stream);

static bool dec_supported(int64_t q_heads, int64_t kv_heads, int64_t head_dim) {
    if (kv_heads <= 0 || q_heads <= 0 || q_heads % kv_heads != 0) return false;
    const int64_t g = q_heads / kv_heads;
    return (g == 1 || g == 2 || g == 4 || g == 8) && (head_dim == 64 || head_dim == 128);
}

}  // namespace lhip

using namespace lhip;

extern "C" {

size_t lhip_attention_decode_workspace_nbytes(int64_t q_heads, int64_t kv_heads, int64_t head_dim) {
    if (!dec_supported(q_heads, kv_heads, head_dim) || kv_heads > 65535) return 0;
    const size_t g = static_cast<size_t>(q_heads / kv_heads);
    const int splits = dec_splits(kv_heads);
    const size_t slots = static_cast<size_t>(kv_heads) * splits * g;
    return dec_ml_bytes(kv_heads, splits, static_cast<int64_t>(g)) +
           slots * static_cast<size_t>(head_dim) * sizeof(float);
}

lhip_status lhip_attention_decode_partial_f32(const float *qkv_dev, float *k_cache_dev, float *v_cache_dev,
                                              const int32_t *pos_dev, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                                              int64_t max_seq, float theta, void *workspace_dev, void *stream) {
    return attention_decode_impl(qkv_dev, k_cache_dev, v_cache_dev, nullptr, false, true, pos_dev, q_heads, kv_heads,
                                 head_dim, max_seq, theta, workspace_dev, stream);
}

lhip_status lhip_attention_decode_few_ranges_f32(const float *qkv_dev, float *k_cache_dev, float *v_cache_dev,
                                                 float *out_dev, const int32_t *pos_dev, int64_t q_heads, int64_t kv_heads,
                                                 int64_t head_dim, int64_t max_seq, float theta, void *workspace_dev,
                                                 void *stream) {
    return attention_decode_impl(qkv_dev, k_cache_dev, v_cache_dev, out_dev, true, true, pos_dev, q_heads, kv_heads,
                                 head_dim, max_seq, theta, workspace_dev, stream);
}

lhip_status lhip_attention_decode_f32(const float *qkv_dev, float *k_cache_dev, float *v_cache_dev, float *out_dev,
                                      const int32_t *pos_dev, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                                      int64_t max_seq, float theta, void *workspace_dev, void *stream) {
    return attention_decode_impl(qkv_dev, k_cache_dev, v_cache_dev, out_dev, true, false, pos_dev, q_heads, kv_heads,
                                 head_dim, max_seq, theta, workspace_dev, stream);
}

}  // extern "C"

namespace lhip {

lhip_status attention_decode_impl(const float *qkv_dev, float *k_cache_dev, float *v_cache_dev, float *out_dev,
                                  bool with_merge, bool few, const int32_t *pos_dev, int64_t q_heads, int64_t kv_heads,
                                  int64_t head_dim, int64_t max_seq, float theta, void *workspace_dev, void *stream) {
    if (!qkv_dev || !k_cache_dev || !v_cache_dev || (with_merge && !out_dev) || !pos_dev || !workspace_dev)
        return LHIP_ERR_NULL_PTR;
    if (q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || max_seq <= 0 || q_heads % kv_heads != 0 ||
        max_seq > kMaxDim || kv_heads > 65535)
        return LHIP_ERR_INVALID_SHAPE;
    if (!dec_supported(q_heads, kv_heads, head_dim)) return LHIP_ERR_UNSUPPORTED;
    if (!aligned(qkv_dev, 16) || !aligned(k_cache_dev, 16) || !aligned(v_cache_dev, 16) ||
        (with_merge && !aligned(out_dev, 16)) || !aligned(workspace_dev, 256))
        return LHIP_ERR_MISALIGNED;
    const int g = static_cast<int>(q_heads / kv_heads);
    const int hkv = static_cast<int>(kv_heads), ms = static_cast<int>(max_seq);
    hipStream_t s = as_stream(stream);
#define LHIP_CASE(G, HD) \
    if (g == G && head_dim == HD) \
        return launch_decode<G, HD>(qkv_dev, k_cache_dev, v_cache_dev, out_dev, pos_dev, hkv, ms, theta, workspace_dev, few, s);
    LHIP_CASE(1, 64) LHIP_CASE(2, 64) LHIP_CASE(4, 64) LHIP_CASE(8, 64)
    LHIP_CASE(1, 128) LHIP_CASE(2, 128) LHIP_CASE(4, 128) LHIP_CASE(8, 128)
#undef LHIP_CASE
    return LHIP_ERR_UNSUPPORTED;
}

}  // namespace lhip
