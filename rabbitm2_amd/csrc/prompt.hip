// A prompt read in as blocks of positions (rabbit2/src/rabbit2.c:703-714 runs it token by token; the tokens
// of a block only meet in the attention, :472-498, which reads the keys and values of the positions before
// them): QK-norm + RoPE + cache rows for a block, and causal attention of the block over the cache. The
// matrix products of a block are grouped_full.hip's, the MoE block is the one of any batch of tokens.
#include <math.h>

#include "rbt2_internal.h"

namespace rbt {
namespace {

// x[t] = the embedding row of the token at position p0 + t (embed_kernel's clamp of the id).
template <int DT>
__global__ __launch_bounds__(256) void prompt_embed_kernel(const void *__restrict__ emb, int D, int vocab,
                                                           const int32_t *__restrict__ seq, float *__restrict__ x) {
    const int i = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (i >= D) return;
    const int tok = min(max(seq[t], 0), vocab - 1);
    x[(size_t)t * D + i] = load_w<DT>(emb, (size_t)tok * D + i);
}

// grid (T), 256 threads. The arithmetic of attn_kernel (model.hip) for each token: QK-norm over the whole q
// and k rows (rabbit2.c:475-478), RoPE from the table at p0 + t (:479-480), k and v into the cache
// (:482-484).
__global__ __launch_bounds__(256) void prompt_rope_kernel(float *__restrict__ q, const float *__restrict__ k,
                                                          const float *__restrict__ v, const float *__restrict__ qw,
                                                          const float *__restrict__ kw, int qk_norm, float eps,
                                                          int n_heads, int n_kv, int hd, int p0, float *__restrict__ kc,
                                                          float *__restrict__ vc, const float2 *__restrict__ rope_cs) {
    __shared__ float red[8];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int qd = n_heads * hd, kvd = n_kv * hd, half = hd / 2, pos = p0 + t;
    q += (size_t)t * qd;
    k += (size_t)t * kvd;
    v += (size_t)t * kvd;
    kc += (size_t)pos * kvd;
    vc += (size_t)pos * kvd;
    float inv_q = 1.0f, inv_k = 1.0f;
    if (qk_norm) {
        float sq = 0.0f, sk = 0.0f;
        for (int i = tid; i < qd; i += 256) sq += q[i] * q[i];
        for (int i = tid; i < kvd; i += 256) sk += k[i] * k[i];
        sq = wave_sum(sq);
        sk = wave_sum(sk);
        if (lane == 0) {
            red[wv] = sq;
            red[4 + wv] = sk;
        }
        __syncthreads();
        sq = (red[0] + red[1]) + (red[2] + red[3]);
        sk = (red[4] + red[5]) + (red[6] + red[7]);
        inv_q = 1.0f / sqrtf(sq / (float)qd + eps);
        inv_k = 1.0f / sqrtf(sk / (float)kvd + eps);
    }
    const float2 *cs = rope_cs + (size_t)pos * half;
    auto rotate = [&](const float *src, const float *w, float inv, float *dst, int rows) {
        for (int u = tid; u < rows * half; u += 256) {  // pair u: elements i and i + half of one head
#pragma clang fp contract(off)
            const int h = u / half, i = u - h * half, lo = h * hd + i, hi = lo + half;
            float a = src[lo], b = src[hi];
            if (qk_norm) {
                a = a * inv * w[lo];
                b = b * inv * w[hi];
            }
            const float2 c = cs[i];
            dst[lo] = a * c.x - b * c.y;
            dst[hi] = b * c.x + a * c.y;
        }
    };
    rotate(q, qw, inv_q, q, n_heads);
    rotate(k, kw, inv_k, kc, n_kv);
    for (int i = tid; i < kvd; i += 256) vc[i] = v[i];
}

// Head dim 128: a block per (head, 16 queries), its four waves each taking every fourth group of 32 keys
// with an online softmax of their own, merged through LDS at the end. Products are v_mfma_f32_16x16x4_f32
// on f32 operands, transposed so that no operand is moved between lanes: S^T = K Q^T leaves lane l the keys
// 4 (l / 16) + i of query l % 16, which is the B operand of O^T = V^T P^T as it stands (step i takes key
// 4 (l / 16) + i in k-slot l / 16). K and Q rows enter 16 bytes per lane (dims 16 s + 4 (l / 16) + i), V
// rows 32 (dims 8 (l % 16) + d), straight from the cache.
// Bound: the serial chain of a wave's key groups (products 128 x 32 clocks per group); 16 queries per
// block, its keys split over four waves, keep the longest chain at a quarter of the keys and fill the chip
// (16 heads, 400 positions: 400 blocks, 25.5 us; with the kernel below 16 layers take 1.4 ms longer).
// A position's output depends on the rows up to its own only, whatever the later ones hold.
constexpr int kPaQ = 16, kPaKeys = 32, kPaHd = 128;
constexpr uint32_t kInfBits = 0x7F800000u;
__global__ __launch_bounds__(256) void prompt_attn_kernel(const float *__restrict__ q, int n_heads, int n_kv, int p0,
                                                          int T, const float *__restrict__ kc,
                                                          const float *__restrict__ vc, float *__restrict__ ao) {
    __shared__ float s_m[4][kPaQ], s_l[4][kPaQ];
    __shared__ __align__(16) float s_o[4][kPaQ][kPaHd + 4];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x, kvh = h / (n_heads / n_kv), kvd = n_kv * kPaHd, qd = n_heads * kPaHd;
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kPaQ;  // the longest blocks first
    const int c = lane & 15, g = lane >> 4;
    const int tq = min(t0 + c, T - 1), last = p0 + tq;  // this lane's query and its last key
    const int n = p0 + min(t0 + kPaQ, T);               // keys of the block
    const float *kb = kc + (size_t)kvh * kPaHd, *vb = vc + (size_t)kvh * kPaHd;
    f32x4 qv[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) qv[s] = ld_f4(q + (size_t)tq * qd + (size_t)h * kPaHd + 16 * s + 4 * g);
    const float scale = 1.0f / sqrtf((float)kPaHd);
    f32x4 o[8];  // o[d][ii]: dim 8 (4 g + ii) + d of query c
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;
    for (int j0 = wv * kPaKeys; j0 < n; j0 += 4 * kPaKeys) {  // wave-uniform
        f32x4 kr[2][8], vr[2][4][2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float *kp = kb + (size_t)min(j0 + 16 * b + c, n - 1) * kvd + 4 * g;
#pragma unroll
            for (int s = 0; s < 8; ++s) kr[b][s] = ld_f4(kp + 16 * s);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float *vp = vb + (size_t)min(j0 + 16 * b + 4 * g + i, n - 1) * kvd + 8 * c;
                vr[b][i][0] = ld_f4(vp);
                vr[b][i][1] = ld_f4(vp + 4);
            }
        f32x4 sc[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            sc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 8; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[b][s][i], qv[s][i], sc[b], 0, 0, 0);
        }
        float mx = m;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[b][i] = j0 + 16 * b + 4 * g + i <= last ? sc[b][i] * scale : -INFINITY;
                mx = fmaxf(mx, sc[b][i]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float ref = mx == -INFINITY ? 0.0f : mx;  // no key of this query yet: all weights 0
        const float alpha = expf(m - ref);
        m = mx;
        l *= alpha;
#pragma unroll
        for (int d = 0; d < 8; ++d) o[d] *= alpha;
        // A key behind a query has weight 0 there, but 0 times an infinity or NaN is NaN, so values that are not
        // finite stay out of the products and are added below, to the queries that may see them.
        uint32_t top = 0;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[b][i] = expf(sc[b][i] - ref);
                l += sc[b][i];
                const bool none = j0 + 16 * b + 4 * g + i >= n;  // (clamped) rows past the block's keys
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    const float v = vr[b][i][d >> 2][d & 3];
                    const uint32_t mag = none ? 0u : __float_as_uint(v) & 0x7FFFFFFFu;
                    top = max(top, mag);
                    o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(none || mag >= kInfBits ? 0.0f : v, sc[b][i], o[d], 0,
                                                                0, 0);
                }
            }
        if (__any(top >= kInfBits)) {  // key by key; the weights change lanes through this wave's s_o
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) s_o[wv][c][16 * b + 4 * g + i] = sc[b][i];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            for (int k = 0; k < kPaKeys && j0 + k < n; ++k) {
                if (j0 + k > last) continue;
                const float p = s_o[wv][c][k], *vp = vb + (size_t)(j0 + k) * kvd + 32 * g;
#pragma unroll
                for (int ii = 0; ii < 4; ++ii)
#pragma unroll
                    for (int d = 0; d < 8; ++d)
                        if (!__builtin_isfinite(vp[8 * ii + d])) o[d][ii] += p * vp[8 * ii + d];
            }
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) {
        s_m[wv][c] = m;
        s_l[wv][c] = l;
    }
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
        float *dst = &s_o[wv][c][8 * (4 * g + ii)];
        *reinterpret_cast<f32x4 *>(dst) = f32x4{o[0][ii], o[1][ii], o[2][ii], o[3][ii]};
        *reinterpret_cast<f32x4 *>(dst + 4) = f32x4{o[4][ii], o[5][ii], o[6][ii], o[7][ii]};
    }
    __syncthreads();
    // 16 threads per query, 8 dims each
    const int mq = tid >> 4, d0 = 8 * (tid & 15);
    if (t0 + mq >= T) return;
    float M = -INFINITY, L = 0.0f, a[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, s_m[w][mq]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        a[w] = s_l[w][mq] > 0.0f ? expf(s_m[w][mq] - M) : 0.0f;
        L += a[w] * s_l[w][mq];
    }
    const float inv = 1.0f / L;
    float *dst = ao + (size_t)(t0 + mq) * qd + (size_t)h * kPaHd + d0;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        f32x4 r = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; ++w) r += a[w] * *reinterpret_cast<const f32x4 *>(&s_o[w][mq][d0 + 4 * x]);
        *reinterpret_cast<f32x4 *>(dst + 4 * x) = r * inv;
    }
}

// Any head dim up to 256: a block per (head, query); 256 keys at a time, a thread per key for the scores
// and a thread per dim for the weighted sum of the values.
__global__ __launch_bounds__(256) void prompt_attn_any_kernel(const float *__restrict__ q, int n_heads, int n_kv,
                                                              int hd, int p0, const float *__restrict__ kc,
                                                              const float *__restrict__ vc, float *__restrict__ ao) {
    __shared__ float s_q[256], s_p[256], red[8];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, h = blockIdx.x, t = blockIdx.y;
    const int kvh = h / (n_heads / n_kv), kvd = n_kv * hd, n = p0 + t + 1;
    if (tid < hd) s_q[tid] = q[((size_t)t * n_heads + h) * hd + tid];
    __syncthreads();
    const float scale = 1.0f / sqrtf((float)hd);
    float m = -INFINITY, l = 0.0f, o = 0.0f;
    for (int j0 = 0; j0 < n; j0 += 256) {
        const int j = j0 + tid;
        float s = -INFINITY;
        if (j < n) {
            const float *kp = kc + (size_t)j * kvd + (size_t)kvh * hd;
            s = 0.0f;
            for (int i = 0; i < hd; ++i) s += s_q[i] * kp[i];
            s *= scale;
        }
        const float wm = wave_max(s);
        if (lane == 0) red[wv] = wm;
        __syncthreads();
        const float mn = fmaxf(fmaxf(m, fmaxf(red[0], red[1])), fmaxf(red[2], red[3]));
        const float ref = mn == -INFINITY ? 0.0f : mn;
        const float p = j < n ? expf(s - ref) : 0.0f;
        s_p[tid] = p;
        const float ps = wave_sum(p);
        if (lane == 0) red[4 + wv] = ps;
        __syncthreads();
        const float alpha = expf(m - ref);
        l = l * alpha + ((red[4] + red[5]) + (red[6] + red[7]));
        o *= alpha;
        if (tid < hd) {
            const float *vp = vc + (size_t)j0 * kvd + (size_t)kvh * hd + tid;
            const int nk = min(256, n - j0);
            for (int jj = 0; jj < nk; ++jj) o += s_p[jj] * vp[(size_t)jj * kvd];
        }
        m = mn;
        __syncthreads();  // red and s_p are rewritten
    }
    if (tid < hd) ao[((size_t)t * n_heads + h) * hd + tid] = o / l;
}

__global__ __launch_bounds__(256) void prompt_record_kernel(const int32_t *__restrict__ routing, int layer,
                                                            int n_layers, int K, int p0, int n,
                                                            int32_t *__restrict__ hist) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) hist[((size_t)(p0 + i / K) * n_layers + layer) * K + i % K] = routing[i];
}

}  // namespace

hipError_t launch_prompt_embed(const Launch &L, int dtype, const void *emb, int D, int vocab, const int32_t *seq, int T,
                               float *x) {
    if (T < 1) return hipSuccess;
    if (T > 65535) return hipErrorInvalidValue;
    const dim3 g((unsigned)((D + 255) / 256), (unsigned)T);
    return dtype == RBT_DT_BF16 ? launch(L, prompt_embed_kernel<RBT_DT_BF16>, g, dim3(256), 0, emb, D, vocab, seq, x)
                                : launch(L, prompt_embed_kernel<RBT_DT_F32>, g, dim3(256), 0, emb, D, vocab, seq, x);
}

hipError_t launch_prompt_rope(const Launch &L, float *q, const float *k, const float *v, const float *qw,
                              const float *kw, int qk_norm, float eps, int n_heads, int n_kv, int hd, int p0, int T,
                              float *kc, float *vc, const float2 *rope_cs) {
    if (T < 1) return hipSuccess;
    return launch(L, prompt_rope_kernel, dim3((unsigned)T), dim3(256), 0, q, k, v, qw, kw, qk_norm, eps, n_heads, n_kv,
                  hd, p0, kc, vc, rope_cs);
}

hipError_t launch_prompt_attention(const Launch &L, const float *q, int n_heads, int n_kv, int hd, int p0, int T,
                                   const float *kc, const float *vc, float *ao) {
    if (T < 1) return hipSuccess;
    if (T > 65535 || hd > 256 || n_heads % n_kv != 0) return hipErrorInvalidValue;
    const auto a16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (hd == kPaHd && a16(q) && a16(kc) && a16(vc) && a16(ao))
        return launch(L, prompt_attn_kernel, dim3((unsigned)n_heads, (unsigned)((T + kPaQ - 1) / kPaQ)), dim3(256), 0, q,
                      n_heads, n_kv, p0, T, kc, vc, ao);
    return launch(L, prompt_attn_any_kernel, dim3((unsigned)n_heads, (unsigned)T), dim3(256), 0, q, n_heads, n_kv, hd, p0,
                  kc, vc, ao);
}

hipError_t launch_prompt_record(const Launch &L, const int32_t *routing, int layer, int n_layers, int K, int p0, int T,
                                int32_t *hist) {
    const int n = T * K;
    return launch(L, prompt_record_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, routing, layer, n_layers, K,
                  p0, n, hist);
}

}  // namespace rbt
