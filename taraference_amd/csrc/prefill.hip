// Prefill (n_tok > 1) for gfx950: causal tiled attention and the batched glue
// of the n_tok-row forward (the GEMMs are in prefill_gemm.hip).
//
// Replaces kernels/attn/fast_v2.cu attn_fast_v2 / attn_fast_v2_d (:12, :103).
#include "dequant.hpp"
#include "prefill.hpp"
#include "tf_common.hpp"
#include "tf_host.hpp"

typedef float tf_f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 tf_h8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------- attention
//
// Causal attention of n_q queries (positions pos0 .. pos0+n_q-1) over the
// f16 cache, fp32 arithmetic.  A workgroup (256 threads) owns one head and
// 16 consecutive queries; K/V tiles of T keys (64, 32, 16 for head_dim 64,
// 128, 256: about 45 KB of LDS) are staged in LDS as f32 and shared by the
// 16 queries.  Thread (query qi = tid / 16, m = tid % 16): scores of keys
// m, m+16, ... of the tile (a DPP row holds one query, so the row max and
// sum are row reductions), then output dims DPT m .. DPT m + DPT-1 with
// DPT = head_dim / 16.  Online softmax as
// the reference: m_new = max(m, tile max), alpha = e^(m - m_new),
// l = l alpha + tile sum, out = acc / max(l, 1e-20).

#define TF_PA_Q 16

template <int HD>
__global__ __launch_bounds__(256) void tf_attn_prefill_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    float* __restrict__ out, int n_head, int n_kv, int pos0_arg, const int* __restrict__ pos0_ptr,
    int n_q, float scale) {
    constexpr int DPT = HD / 16;  // output dims per thread
    constexpr int TF_PA_T = HD == 64 ? 64 : (HD == 128 ? 32 : 16);  // keys per tile
    constexpr int NS = TF_PA_T / 16;                                // scores per thread
    __shared__ __align__(16) float qs[TF_PA_Q * (HD + 4)];
    __shared__ __align__(16) float ks[TF_PA_T * (HD + 4)];
    __shared__ __align__(16) float vs[TF_PA_T * HD];
    __shared__ float ps[TF_PA_Q * (TF_PA_T + 1)];
    const int pos0 = pos0_ptr ? pos0_ptr[0] : pos0_arg;
    const int h = blockIdx.y, q0 = blockIdx.x * TF_PA_Q;
    const int tid = threadIdx.x, qi = tid >> 4, m = tid & 15;
    const int kv_h = h / (n_head / n_kv), stride = n_kv * HD;
    const int qn = q0 + qi;
    const bool qvalid = qn < n_q;
    const int my_len = pos0 + (qvalid ? qn : q0) + 1;           // keys this query sees
    const int last_q = (q0 + TF_PA_Q < n_q ? q0 + TF_PA_Q : n_q) - 1;
    const int seq_len = pos0 + last_q + 1;                         // keys of the workgroup
    for (int i = tid; i < TF_PA_Q * HD / 4; i += 256) {
        const int r = i / (HD / 4), c4 = i % (HD / 4);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (q0 + r < n_q)
            v = *reinterpret_cast<const float4*>(q + (size_t)(q0 + r) * n_head * HD + h * HD + 4 * c4);
        *reinterpret_cast<float4*>(qs + r * (HD + 4) + 4 * c4) = v;
    }
    float mx = -1e30f, l = 0.f, acc[DPT];
    for (int i = 0; i < DPT; i++) acc[i] = 0.f;
    for (int t0 = 0; t0 < seq_len; t0 += TF_PA_T) {
        const int tlen = seq_len - t0 < TF_PA_T ? seq_len - t0 : TF_PA_T;
        __syncthreads();  // q staged / previous tile consumed
        for (int i = tid; i < TF_PA_T * HD / 4; i += 256) {
            const int r = i / (HD / 4), c4 = i % (HD / 4);
            float4 kf = make_float4(0.f, 0.f, 0.f, 0.f), vf = kf;
            if (r < tlen) {
                const size_t off = (size_t)(t0 + r) * stride + (size_t)kv_h * HD + 4 * c4;
                const uint2 kb = *reinterpret_cast<const uint2*>(kc + off);
                const uint2 vb = *reinterpret_cast<const uint2*>(vc + off);
                kf = make_float4(tf_h2f(kb.x), tf_h2f(kb.x >> 16), tf_h2f(kb.y), tf_h2f(kb.y >> 16));
                vf = make_float4(tf_h2f(vb.x), tf_h2f(vb.x >> 16), tf_h2f(vb.y), tf_h2f(vb.y >> 16));
            }
            *reinterpret_cast<float4*>(ks + r * (HD + 4) + 4 * c4) = kf;
            *reinterpret_cast<float4*>(vs + r * HD + 4 * c4) = vf;
        }
        __syncthreads();
        // scores of keys m + 16 j
        float s[NS];
        const float* qrow = qs + qi * (HD + 4);
#pragma unroll
        for (int j = 0; j < NS; j++) {
            const float* krow = ks + (m + 16 * j) * (HD + 4);
            float a0 = 0.f, a1 = 0.f;
            for (int d = 0; d < HD; d += 8) {
                const float4 qa = *reinterpret_cast<const float4*>(qrow + d);
                const float4 qb = *reinterpret_cast<const float4*>(qrow + d + 4);
                const float4 ka = *reinterpret_cast<const float4*>(krow + d);
                const float4 kb = *reinterpret_cast<const float4*>(krow + d + 4);
                a0 += qa.x * ka.x + qa.y * ka.y + qa.z * ka.z + qa.w * ka.w;
                a1 += qb.x * kb.x + qb.y * kb.y + qb.z * kb.z + qb.w * kb.w;
            }
            const int key = t0 + m + 16 * j;
            s[j] = key < my_len ? (a0 + a1) * scale : -1e30f;
        }
        float tmax = s[0];
#pragma unroll
        for (int j = 1; j < NS; j++) tmax = fmaxf(tmax, s[j]);
        tmax = tf_row16_max(tmax);
        const float m_new = fmaxf(mx, tmax);
        const float alpha = __expf(mx - m_new);
        float ls = 0.f;
#pragma unroll
        for (int j = 0; j < NS; j++) {
            const float e = s[j] > -1e29f ? __expf(s[j] - m_new) : 0.f;
            ps[qi * (TF_PA_T + 1) + m + 16 * j] = e;
            ls += e;
        }
        ls = tf_row16_sum(ls);
        l = l * alpha + ls;
        mx = m_new;
        for (int i = 0; i < DPT; i++) acc[i] *= alpha;
        __syncthreads();  // ps complete (the row's other lanes wrote it)
        const float* prow = ps + qi * (TF_PA_T + 1);
        for (int t = 0; t < tlen; t++) {
            const float p = prow[t];
            const float* vrow = vs + t * HD + DPT * m;
#pragma unroll
            for (int i = 0; i < DPT; i += 4) {
                const float4 v = *reinterpret_cast<const float4*>(vrow + i);
                acc[i] += p * v.x;
                acc[i + 1] += p * v.y;
                acc[i + 2] += p * v.z;
                acc[i + 3] += p * v.w;
            }
        }
    }
    if (qvalid) {
        const float inv = 1.f / fmaxf(l, 1e-20f);
        float* o = out + (size_t)qn * n_head * HD + h * HD + DPT * m;
        for (int i = 0; i < DPT; i += 4)
            *reinterpret_cast<float4*>(o + i) =
                make_float4(acc[i] * inv, acc[i + 1] * inv, acc[i + 2] * inv, acc[i + 3] * inv);
    }
}

// Matrix-core form for head_dim 128.  A workgroup (4 waves) owns one head
// and 16 queries; the waves split the 32-key tiles round-robin, each staging
// its own tiles in LDS, and merge their (m, l, O) with the log-sum-exp rule
// at the end (a wave with no keys for a query contributes e^(-1e30 - M) = 0).
// Per tile, on v_mfma_f32_16x16x32_f16:
//   S^T = K q^T: A = K rows (A row i of key block b is key
//       8 (i / 4) + 4 b + i % 4, so the C values a lane holds, key rows
//       4g .. 4g+3 of blocks 0 and 1, are the tile's keys 8g .. 8g+7), B =
//       q^T, q split into two f16 parts after a power-of-two scale (2^-22
//       relative per product; K is f16, the products are exact);
//   O += P V: A = P (query l16, keys 8g .. 8g+7: the lane's own S values
//       after the softmax, split into two f16 parts), B = V gathered from
//       the row-major f16 tile (8 u16 reads per fragment).
// Softmax per query: the lane's 8 values, then the 4 lanes of the query
// (xor 16, 32).  Keys past the workgroup's last query are staged as zeros.

#define TF_PM_T 32              // keys per tile
#define TF_PM_KROW 272          // K tile row bytes (128 f16 + 16)
#define TF_PM_VROW 264          // V tile row bytes (128 f16 + 8): 8-row gathers on distinct banks
#define TF_PM_WAVE_BYTES (TF_PM_T * TF_PM_KROW + TF_PM_T * TF_PM_VROW)

__global__ __launch_bounds__(256) void tf_attn_prefill_mfma_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    float* __restrict__ out, int n_head, int n_kv, int pos0_arg, const int* __restrict__ pos0_ptr,
    int n_q, float scale) {
    constexpr int HD = 128;
    __shared__ __align__(16) uint8_t lds[4 * TF_PM_WAVE_BYTES];
    __shared__ float ml[2][4][16];
    const int pos0 = pos0_ptr ? pos0_ptr[0] : pos0_arg;
    const int h = blockIdx.y, q0 = blockIdx.x * 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, l16 = lane & 15;
    const int kv_h = h / (n_head / n_kv), stride = n_kv * HD;
    const int last_q = (q0 + 16 < n_q ? q0 + 16 : n_q) - 1;
    const int kv_len = pos0 + last_q + 1;  // keys the workgroup reads
    const int n_t = (kv_len + TF_PM_T - 1) / TF_PM_T;
    uint8_t* kt = lds + wave * TF_PM_WAVE_BYTES;
    uint8_t* vt = kt + TF_PM_T * TF_PM_KROW;

    // q^T fragments: query l16, dims 32 st + 8 g .. +7, two f16 parts
    const int my_q = q0 + l16 < n_q ? q0 + l16 : last_q;
    const int qpos = pos0 + my_q;
    float qv[32];
    {
        const float* qr = q + (size_t)my_q * n_head * HD + (size_t)h * HD;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const float4 a = *reinterpret_cast<const float4*>(qr + 32 * st + 8 * g);
            const float4 b = *reinterpret_cast<const float4*>(qr + 32 * st + 8 * g + 4);
            qv[8 * st] = a.x; qv[8 * st + 1] = a.y; qv[8 * st + 2] = a.z; qv[8 * st + 3] = a.w;
            qv[8 * st + 4] = b.x; qv[8 * st + 5] = b.y; qv[8 * st + 6] = b.z; qv[8 * st + 7] = b.w;
        }
    }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(qv[i]));
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    const int eb = (int)((__float_as_uint(amax) >> 23) & 0xff);
    int fe = amax > 0.f ? 141 - eb : 0;
    fe = fe > 126 ? 126 : fe;
    const float f = __uint_as_float((uint32_t)(fe + 127) << 23);
    const float sscale = scale * __uint_as_float((uint32_t)(127 - fe) << 23);
    tf_h8 qb[4][2];
#pragma unroll
    for (int st = 0; st < 4; st++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float a = qv[8 * st + i] * f;
            const _Float16 hi = (_Float16)a;
            qb[st][0][i] = hi;
            qb[st][1][i] = (_Float16)(a - (float)hi);
        }

    float mx = -1e30f, l = 0.f;
    tf_f32x4 o[8];
#pragma unroll
    for (int nb = 0; nb < 8; nb++) o[nb] = tf_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int ti = wave; ti < n_t; ti += 4) {
        const int t0 = ti * TF_PM_T;
        // stage K and V rows t0 .. t0+31 (zeros past kv_len)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int idx = lane + 64 * j, r = idx >> 4, c = idx & 15;
            tf_u32x4 kb = {0, 0, 0, 0}, vb = {0, 0, 0, 0};
            if (t0 + r < kv_len) {
                const size_t off = (size_t)(t0 + r) * stride + (size_t)kv_h * HD + 8 * c;
                kb = *reinterpret_cast<const tf_u32x4*>(kc + off);
                vb = *reinterpret_cast<const tf_u32x4*>(vc + off);
            }
            *reinterpret_cast<tf_u32x4*>(kt + r * TF_PM_KROW + 16 * c) = kb;
            uint32_t* vw = reinterpret_cast<uint32_t*>(vt + r * TF_PM_VROW + 16 * c);
            vw[0] = vb.x; vw[1] = vb.y; vw[2] = vb.z; vw[3] = vb.w;  // 8-byte aligned rows
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // LDS stores of the wave done (lgkmcnt 0)
        __builtin_amdgcn_wave_barrier();
        // S^T: two key blocks, 4 K steps, 2 parts
        tf_f32x4 sc[2];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int key = 8 * (l16 >> 2) + 4 * b + (l16 & 3);
            tf_f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 4; st++) {
                const tf_h8 ka = *reinterpret_cast<const tf_h8*>(kt + key * TF_PM_KROW +
                                                                 2 * (32 * st + 8 * g));
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[st][0], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[st][1], c, 0, 0, 0);
            }
            sc[b] = c;
        }
        // lane values: keys t0 + 8g + 4b + r of query my_q
        float sv[8];
        float tmax = -1e30f;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int kp = t0 + 8 * g + 4 * b + r;
                const float v = kp <= qpos ? sc[b][r] * sscale : -1e30f;
                sv[4 * b + r] = v;
                tmax = fmaxf(tmax, v);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float m_new = fmaxf(mx, tmax);
        const float alpha = __expf(mx - m_new);
        float ls = 0.f;
        tf_h8 pa[2];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float e = sv[i] > -1e29f ? __expf(sv[i] - m_new) : 0.f;
            ls += e;
            const _Float16 hi = (_Float16)e;
            pa[0][i] = hi;
            pa[1][i] = (_Float16)(e - (float)hi);
        }
        ls += __shfl_xor(ls, 16);
        ls += __shfl_xor(ls, 32);
        l = l * alpha + ls;
        mx = m_new;
        // O rows are queries 4g .. 4g+3: their alpha from lanes 4g + r
        float al[4];
#pragma unroll
        for (int r = 0; r < 4; r++) al[r] = __shfl(alpha, 4 * g + r);
#pragma unroll
        for (int nb = 0; nb < 8; nb++) {
#pragma unroll
            for (int r = 0; r < 4; r++) o[nb][r] *= al[r];
            // V fragment: keys 8g .. 8g+7, dim 16 nb + l16
            const uint8_t* vp = vt + (8 * g) * TF_PM_VROW + 2 * (16 * nb + l16);
            tf_h8 vf;
#pragma unroll
            for (int i = 0; i < 8; i++)
                vf[i] = __builtin_bit_cast(_Float16, *reinterpret_cast<const uint16_t*>(vp + i * TF_PM_VROW));
            o[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[0], vf, o[nb], 0, 0, 0);
            o[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[1], vf, o[nb], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();  // tile reads done before the next staging
    }
    // merge the 4 waves: (m, l) per query, O through LDS
    if (g == 0) {
        ml[0][wave][l16] = mx;
        ml[1][wave][l16] = l;
    }
    __syncthreads();  // every wave's tiles consumed; ml visible
    float* ow = reinterpret_cast<float*>(lds + wave * TF_PM_WAVE_BYTES);  // [16][128]
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int qi = 4 * g + r;
        float mall = ml[0][0][qi];
        for (int w = 1; w < 4; w++) mall = fmaxf(mall, ml[0][w][qi]);
        const float sc_w = __expf(ml[0][wave][qi] - mall);
#pragma unroll
        for (int nb = 0; nb < 8; nb++) ow[qi * HD + 16 * nb + l16] = o[nb][r] * sc_w;
    }
    __syncthreads();
    {
        const int qi = tid >> 4, d0 = 8 * (tid & 15);
        if (q0 + qi < n_q) {
            float mall = ml[0][0][qi];
            for (int w = 1; w < 4; w++) mall = fmaxf(mall, ml[0][w][qi]);
            float L = 0.f;
            for (int w = 0; w < 4; w++) L += ml[1][w][qi] * __expf(ml[0][w][qi] - mall);
            const float inv = 1.f / fmaxf(L, 1e-20f);
            float acc[8];
            for (int i = 0; i < 8; i++) acc[i] = 0.f;
            for (int w = 0; w < 4; w++) {
                const float* src = reinterpret_cast<const float*>(lds + w * TF_PM_WAVE_BYTES) + qi * HD + d0;
                for (int i = 0; i < 8; i++) acc[i] += src[i];
            }
            float* dst = out + (size_t)(q0 + qi) * n_head * HD + (size_t)h * HD + d0;
            *reinterpret_cast<float4*>(dst) = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
            *reinterpret_cast<float4*>(dst + 4) = make_float4(acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv);
        }
    }
}

// ------------------------------------------------- batched prefill glue
//
// Embedding rows of a prompt (kernels/embed.cu embed_q{4,6}_k :1-50) and
// silu_mul_f32 (kernels/ops.cu:202).

template <int BB>
__global__ __launch_bounds__(256) void tf_pf_embed_kernel(const uint8_t* __restrict__ table,
                                                          const int* __restrict__ tokens,
                                                          float* __restrict__ out, int n_rows,
                                                          int col_bytes) {
    const int t = blockIdx.y;
    const uint8_t* col = table + (size_t)tokens[t] * col_bytes;
    const int nb = n_rows / 256;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nb * 256; i += gridDim.x * blockDim.x) {
        const uint8_t* blk = col + (size_t)(i >> 8) * BB;
        out[(size_t)t * n_rows + i] = BB == 144 ? tf_q4k_value(blk, i & 255) : tf_q6k_value(blk, i & 255);
    }
}

__global__ __launch_bounds__(256) void tf_pf_silu_mul_kernel(float* __restrict__ g,
                                                             const float* __restrict__ u,
                                                             long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float v = g[i];
        g[i] = (v / (1.f + __expf(-v))) * u[i];
    }
}

int tf_pf_embed(const uint8_t* table, int block_bytes, const int* tokens_dev, float* out,
                int n_rows, int col_bytes, int n_tok, tf_stream_t stream) {
    const int nb = n_rows / 256;
    TF_CHECK_ARG(table && tokens_dev && out && nb > 0 && n_tok > 0);
    TF_CHECK_ARG((block_bytes == 144 || block_bytes == 210) && col_bytes >= nb * block_bytes);
    const dim3 grid((nb * 256 + 255) / 256, n_tok);
    if (block_bytes == 144)
        hipLaunchKernelGGL(tf_pf_embed_kernel<144>, grid, dim3(256), 0, tf_stream(stream), table,
                           tokens_dev, out, n_rows, col_bytes);
    else
        hipLaunchKernelGGL(tf_pf_embed_kernel<210>, grid, dim3(256), 0, tf_stream(stream), table,
                           tokens_dev, out, n_rows, col_bytes);
    return TF_LAUNCH_RESULT();
}

int tf_pf_silu_mul(float* g, const float* u, long long n, tf_stream_t stream) {
    TF_CHECK_ARG(g && u && n > 0);
    hipLaunchKernelGGL(tf_pf_silu_mul_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       tf_stream(stream), g, u, n);
    return TF_LAUNCH_RESULT();
}

// ---------------------------------------------------------------- C ABI

int tf_attn_prefill_any(const float* q, const uint16_t* k_cache, const uint16_t* v_cache,
                               float* out, int n_head, int n_kv, int head_dim, int pos0,
                               const int* pos0_dev, int n_q, float scale, tf_stream_t stream) {
    TF_CHECK_ARG(q && k_cache && v_cache && out && n_head > 0 && n_kv > 0 && n_q > 0);
    TF_CHECK_ARG(n_head % n_kv == 0 && (pos0_dev || pos0 >= 0));
    TF_CHECK_ARG(head_dim == 64 || head_dim == 128 || head_dim == 256);
    TF_CHECK_ARG(((uintptr_t)q & 15) == 0 && ((uintptr_t)out & 15) == 0);
    TF_CHECK_ARG(((uintptr_t)k_cache & 7) == 0 && ((uintptr_t)v_cache & 7) == 0);
    const dim3 grid((n_q + TF_PA_Q - 1) / TF_PA_Q, n_head);
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, tf_stream(stream), q, k_cache, v_cache, out,
                           n_head, n_kv, pos0, pos0_dev, n_q, scale);
    };
    if (head_dim == 64) go(tf_attn_prefill_kernel<64>);
    else if (head_dim == 128) {
        const dim3 g16((n_q + 15) / 16, n_head);
        hipLaunchKernelGGL(tf_attn_prefill_mfma_kernel, g16, dim3(256), 0, tf_stream(stream), q,
                           k_cache, v_cache, out, n_head, n_kv, pos0, pos0_dev, n_q, scale);
    } else go(tf_attn_prefill_kernel<256>);
    return TF_LAUNCH_RESULT();
}

extern "C" int tf_attn_prefill(const float* q, const uint16_t* k_cache, const uint16_t* v_cache,
                               float* out, int n_head, int n_kv, int head_dim, int pos0, int n_q,
                               float scale, tf_stream_t stream) {
    return tf_attn_prefill_any(q, k_cache, v_cache, out, n_head, n_kv, head_dim, pos0, nullptr,
                               n_q, scale, stream);
}

extern "C" int tf_attn_prefill_d(const float* q, const uint16_t* k_cache,
                                 const uint16_t* v_cache, float* out, int n_head, int n_kv,
                                 int head_dim, const int* pos0_dev, int n_q, float scale,
                                 tf_stream_t stream) {
    TF_CHECK_ARG(pos0_dev != nullptr);
    return tf_attn_prefill_any(q, k_cache, v_cache, out, n_head, n_kv, head_dim, 0, pos0_dev, n_q,
                               scale, stream);
}
