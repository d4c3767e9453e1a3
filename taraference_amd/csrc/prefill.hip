// Prefill (n_tok > 1) for gfx950: causal tiled attention and the batched glue
// of the n_tok-row forward (the GEMMs are in prefill_gemm.hip).
//
// Replaces kernels/attn/fast_v2.cu attn_fast_v2 / attn_fast_v2_d (:12, :103).
#include "dequant.hpp"
#include "lds_dma.hpp"
#include "prefill.hpp"
#include "tf_common.hpp"
#include "tf_host.hpp"

typedef float tf_f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 tf_h8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------- attention
//
// Causal attention of n_q queries (positions pos0 .. pos0+n_q-1) over the
// f16 cache; head_dim 256 in fp32 vector arithmetic, 64 and 128 on the matrix
// cores (below).  A workgroup (256 threads) owns one head and 16 consecutive
// queries; K/V tiles of 16 keys (about 45 KB of LDS) are staged in LDS as f32
// and shared by the 16 queries.  Thread (query qi = tid / 16, m = tid % 16): scores of keys
// m, m+16, ... of the tile (a DPP row holds one query, so the row max and
// sum are row reductions), then output dims DPT m .. DPT m + DPT-1 with
// DPT = head_dim / 16.  Online softmax as
// the reference: m_new = max(m, tile max), alpha = e^(m - m_new),
// l = l alpha + tile sum, out = acc / max(l, 1e-20).

#define TF_PA_Q 16

__global__ __launch_bounds__(256) void tf_attn_prefill_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    float* __restrict__ out, int n_head, int n_kv, int pos0_arg, const int* __restrict__ pos0_ptr,
    int n_q, float scale) {
    constexpr int HD = 256;
    constexpr int DPT = HD / 16;      // output dims per thread
    constexpr int TF_PA_T = 16;       // keys per tile
    constexpr int NS = TF_PA_T / 16;  // scores per thread
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

// Matrix-core form for head_dim 64 and 128.  The rows of a kv head are its
// (query, head) pairs, heads fastest: row r is query r / G, head r % G of the
// group (G = n_head / n_kv).  A workgroup owns 32 rows, so each K/V byte it
// reads serves 32 rows whatever the group or the prompt length, and its eight
// waves share the 32-key tiles round-robin, each with its own LDS tile pair and
// its own (m, l, O); the eight are merged with the log-sum-exp rule at the end.
// Rows are split this finely because a prompt has few of them (512 tokens of 16
// heads over 2 kv heads: 256 workgroups, one a CU); the waves take keys, not
// rows, so that they never wait for each other while streaming.
//
// K and V move HBM / L2 -> LDS without registers (global_load_lds), one tile
// ahead: the next K tile is requested when the scores of this one are formed
// and arrives under the softmax and P V, the next V tile when P V is done and
// arrives under the next scores.  Copies complete in issue order, so vmcnt(one
// tile's copies) waits for exactly the older tile.
//
// Per tile, on v_mfma_f32_32x32x16_f16 (lane l, h = l / 32: A[l % 32][8h ..],
// B[8h ..][l % 32], C[8 (i / 4) + 4 h + i % 4][l % 32]):
//   S^T[key][row] = K q^T, q in two f16 parts after a power-of-two scale per
//       row (2^-22 relative per product; K is f16, the products are exact);
//   softmax over the lane's 16 keys and the other half's 16 (one exchange), in
//       powers of two; O is rescaled only where a row's maximum moved;
//   O^T[dim][row] += V^T P^T with 2^14 P in two f16 parts: 2^-22 of a weight, and
//       2^-39 of the row's largest where a weight is below 2^-17 of it (unscaled the
//       parts end at 2^-24: 8000 keys e^-17 below a sink lost half their share).
//       l stays unscaled; the merge takes 2^14 out again.  k index i of half h in
//       step s stands for key 16 s + 8 (i / 4) + 4 h + i % 4, which is how
//       the scores already lie, so P needs no exchange; the V operand is two
//       transposing LDS reads (ds_read_b64_tr_b16: four keys of a lane's dim).
// At head_dim 64, which fp32 vector arithmetic served before, the products of second
// parts come first in each sum, where it is still small, so that half of the additions
// round 2^-11 as much (registers for both parts' operands: head_dim 128 has none).
// Error against 64 bits for 5 tokens at 20, 40 and 300 keys 1.44, 1.62 and 2.25e-7 (part
// by part 1.86, 2.08 and 2.88; the vector ALU 1.49, 1.79 and 3.59), at the same time.
// LDS rows keep their 16-byte chunks xor-ed with the row, so that 16 K rows, or
// the 4 rows x 64 bytes of a transposing read, fall on distinct banks.
// What bounds it: long contexts, the matrix cores (two products per score and per
// P V term) and LDS bandwidth about equally, 27 us each of the 74 us that 256
// tokens of 28 heads at position 8000 take, with the softmax between them (a raised
// wave priority for either half changed nothing); short ones, the chain of copy,
// scores, P V and merge of one tile.  The form before it (16 queries of one head,
// keys staged through registers, V gathered two bytes at a time; head_dim 64 on the
// vector ALU) took 234 us there, 16.5 where this takes 11.0 for a fresh 512-token
// prompt of 16 heads, 33 against 7.7 for 400 tokens of 14 heads of 64, 5.1 and 5.1
// for 5 tokens (q split by each wave for itself instead of once: 13.4, 9.1 and 5.1
// us for these three).  Error against 64 bits 5.1e-7 at 8000 and
// 2.5e-7 at 512, before 6.7e-7 and 2.7e-7.
#define TF_PM_WAVES 8
#define TF_PM_T 32  // keys per tile, rows per workgroup
#define TF_PM_FEW 16  // keys of a workgroup that head_dim 64 takes in fp32

template <int HD>
struct TfPmLds {
    static constexpr int ROWB = 2 * HD;                // K / V row bytes
    static constexpr int TILE = TF_PM_T * ROWB;        // a K or V tile
    static constexpr int OROW = HD + 4;                // floats of a merge row
    static constexpr int WAVE = TF_PM_T * OROW * 4;    // the K + V tiles, then the wave's O
    static constexpr int ML = TF_PM_WAVES * WAVE;      // m, l: [2][waves][32]
    static constexpr int Q = ML + 2 * TF_PM_WAVES * TF_PM_T * 4;  // q fragments, two parts
    static constexpr int S2 = Q + 2 * TILE;                       // a factor per row
    static constexpr int BYTES = S2 + TF_PM_T * 4;
    static_assert(2 * TILE <= WAVE, "the tiles fit where O goes");
};

typedef float tf_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 tf_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 tf_h4 __attribute__((ext_vector_type(4)));
typedef short tf_s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t tf_lds_u8;

template <int N>
__device__ __forceinline__ void tf_wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 2^14 e = hi + lo in f16 parts, two values at a time.  hi is opaque to the compiler,
// which would otherwise convert each value a second time for lo's difference.
__device__ __forceinline__ void tf_split2(float a, float b, tf_h2& hi, tf_h2& lo) {
    a *= 0x1p14f;
    b *= 0x1p14f;
    uint32_t h = __builtin_bit_cast(uint32_t, tf_h2{(_Float16)a, (_Float16)b});
    asm("" : "+v"(h));
    hi = __builtin_bit_cast(tf_h2, h);
    lo = tf_h2{(_Float16)(a - (float)hi.x), (_Float16)(b - (float)hi.y)};
}

// v *= f, each product rounded (not fused into what uses it)
__device__ __forceinline__ void tf_scores_pow2(tf_f32x16& v, float f) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 16; i++) {
        float t = v[i] * f;
        asm("" : "+v"(t));
        v[i] = t;
    }
}

// r / d by the reciprocal m = ceil(2^32 / d) (0 for d = 1): the product is at
// most one too large
__device__ __forceinline__ uint32_t tf_div_by(uint32_t r, uint32_t d, uint32_t m) {
    if (m == 0) return r;
    const uint32_t t = __umulhi(r, m);
    return t * d > r ? t - 1 : t;
}

// A head_dim 64 row in fp32, by 16 threads of four dims each, one key after the other.
// For rows in which something is not finite: an infinity in q, K or V times one f16
// part of the other operand is NaN where the product is not.  A NaN or -inf score is
// no key, a +inf one makes the row NaN, as in the vector form.  And for workgroups of
// at most TF_PM_FEW keys, where the matrix cores' sums and P's 22 bits are what is left
// of the error (2, 5 and 12 keys: 4.5, 6.9 and 8.8e-8 against 64 bits, 3.9, 6.2 and
// 8.4 here, 4.1, 6.3 and 8.5 on the vector ALU before; from 20 keys on the matrix
// cores are the better: 1.4 against 1.5e-7).  5.0 us for 5 tokens either way.
__device__ __noinline__ float4 tf_attn_row64(const float* q, const uint8_t* kbase,
                                             const uint8_t* vbase, uint32_t row_bytes, int n_keys,
                                             float scale) {
    const int m = threadIdx.x & 15;
    const float4 a = *reinterpret_cast<const float4*>(q + 4 * m);
    auto score = [&](int t) {
        const uint2 k = *reinterpret_cast<const uint2*>(kbase + (size_t)t * row_bytes + 8 * m);
        return scale * tf_row16_sum(a.x * tf_h2f(k.x) + a.y * tf_h2f(k.x >> 16) +
                                    a.z * tf_h2f(k.y) + a.w * tf_h2f(k.y >> 16));
    };
    float mx = -1e30f, l = 0.f;
    for (int t = 0; t < n_keys; t++) mx = fmaxf(mx, score(t));
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int t = 0; t < n_keys; t++) {
        const uint2 v = *reinterpret_cast<const uint2*>(vbase + (size_t)t * row_bytes + 8 * m);
        const float s = score(t);
        const float e = s > -1e29f ? __expf(s - mx) : 0.f;
        l += e;
        acc.x += e * tf_h2f(v.x);
        acc.y += e * tf_h2f(v.x >> 16);
        acc.z += e * tf_h2f(v.y);
        acc.w += e * tf_h2f(v.y >> 16);
    }
    const float inv = 1.f / fmaxf(l, 1e-20f);
    return make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

// DW: bytes a lane copies (16; 4 where the caches are only 8-byte aligned)
template <int HD, int DW>
__global__ __launch_bounds__(64 * TF_PM_WAVES, 2) void tf_attn_prefill_mfma_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
    float* __restrict__ out, int n_head, int n_kv, int pos0_arg, const int* __restrict__ pos0_ptr,
    int n_rows, int G, uint32_t g_inv, uint32_t kv_inv, float scale) {
    using L = TfPmLds<HD>;
    constexpr int ROWB = L::ROWB, ST = HD / 16, DB = HD / 32;
    constexpr int NC = L::TILE / (64 * DW);  // copies of a tile
    constexpr int NCU = NC > 16 ? 16 : NC;   // 32 at once do not fit the registers
    extern __shared__ __align__(16) uint8_t lds[];
    const int pos0 = pos0_ptr ? pos0_ptr[0] : pos0_arg;
    // kv heads fastest (workgroups of one kv head share few XCDs' L2), the
    // rows with the most keys first
    const int rb = tf_div_by(gridDim.x - 1 - blockIdx.x, n_kv, kv_inv);
    const int kv_h = (gridDim.x - 1 - blockIdx.x) - rb * n_kv, r0 = rb * TF_PM_T;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const int rl = (r0 + TF_PM_T < n_rows ? r0 + TF_PM_T : n_rows) - 1;
    const int kv_len = pos0 + (int)tf_div_by(rl, G, g_inv) + 1;  // keys the workgroup reads
    const int first_pos = pos0 + (int)tf_div_by(r0, G, g_inv);   // every row sees keys up to here
    const int n_t = (kv_len + TF_PM_T - 1) / TF_PM_T;
    const uint32_t row_bytes = (uint32_t)n_kv * ROWB;
    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(kc) + (size_t)kv_h * ROWB;
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(vc) + (size_t)kv_h * ROWB;
    if (HD == 64 && kv_len <= TF_PM_FEW) {
        const int r = r0 + (tid >> 4), qo = tf_div_by(r, G, g_inv);
        if (r < n_rows) {
            const size_t row = ((size_t)qo * n_head + (size_t)kv_h * G + (r - qo * G)) * HD;
            *reinterpret_cast<float4*>(out + row + 4 * (tid & 15)) =
                tf_attn_row64(q + row, kbase, vbase, row_bytes, pos0 + qo + 1, scale);
        }
        return;
    }
    uint8_t* kt = lds + wave * L::WAVE;
    uint8_t* vt = kt + L::TILE;

    // the query of this lane's row
    const int qpos = pos0 + (int)tf_div_by(r0 + l32 < n_rows ? r0 + l32 : rl, G, g_inv);

    // copy i of a tile: byte p = 64 DW i + DW lane of it, row p / ROWB; rows past
    // the last key repeat it (their scores are masked)
    auto issue = [&](const uint8_t* base, uint8_t* dst, int t0, bool is_v) {
        const uint8_t* tb = base + (size_t)t0 * row_bytes;
        const uint32_t ldst = tf_lds_off(dst);
        const int rmax = kv_len - 1 - t0;
        auto off = [&](int i, int last) -> uint32_t {
            const int p = 64 * DW * i + DW * lane, r = p / ROWB;
            const int c = (p % ROWB) >> 4;
            const int sw = is_v ? (HD == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1))
                                : (HD == 128 ? r & 15 : (r >> 1) & 7);
            return (uint32_t)(r < last ? r : last) * row_bytes + 16 * (c ^ sw) + (p & 15);
        };
        if (rmax >= TF_PM_T - 1) {
#pragma unroll NCU
            for (int i = 0; i < NC; i++)
                tf_lds_dma_s<DW>(tb, off(i, TF_PM_T), ldst + 64 * DW * i);
        } else {
#pragma unroll 1
            for (int i = 0; i < NC; i++)
                tf_lds_dma_s<DW>(tb, off(i, rmax), ldst + 64 * DW * i);
        }
    };
    // q^T fragments: dims 16 st + 8 h .. +7 of a row in two f16 parts, after a
    // power of two that takes the row's largest value to [2^14, 2^15) and with the
    // sign of the scale, so that the largest score has the largest product.  Made
    // once for the workgroup: wave w copies rows 4 w .. + 3 (where its V tile will
    // go, K right behind them), a thread splits eight dims; chunk c = 2 st + h of
    // row r at 16-byte slot 32 c + (r ^ c) of a part.
    float s2;  // score in powers of two = product * s2
    tf_h8 qb[ST][2];
    {
        constexpr int QC = 4 * HD * 4 / 1024;  // copies of a wave's q rows
        const bool tiles = wave < n_t;
#pragma unroll
        for (int i = 0; i < QC; i++) {
            const int p = 1024 * i + 16 * lane, rq = r0 + 4 * wave + p / (4 * HD);
            const int r = rq < n_rows ? rq : rl;
            const int ri = tf_div_by(r, G, g_inv);
            tf_lds_dma16(reinterpret_cast<const uint8_t*>(
                             q + ((size_t)ri * n_head + (size_t)kv_h * G + (r - ri * G)) * HD) +
                             p % (4 * HD),
                         tf_lds_off(vt) + 1024 * i);
        }
        if (tiles) {
            issue(kbase, kt, wave * TF_PM_T, false);
            tf_wait_vm<NC>();
        } else {
            tf_wait_vm<0>();
        }
        const int c = lane & (HD / 8 - 1), rw = lane / (HD / 8);
        if (rw < 4) {
            const float4 a = *reinterpret_cast<const float4*>(vt + rw * 4 * HD + 32 * c);
            const float4 b = *reinterpret_cast<const float4*>(vt + rw * 4 * HD + 32 * c + 16);
            const float qv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            float amax = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(qv[i]));
#pragma unroll
            for (int x = 1; x < HD / 8; x <<= 1) amax = fmaxf(amax, __shfl_xor(amax, x));
            const int eb = (int)((__float_as_uint(amax) >> 23) & 0xff);
            int fe = amax > 0.f ? 141 - eb : 0;
            fe = fe > 126 ? 126 : fe;
            const float f = copysignf(__uint_as_float((uint32_t)(fe + 127) << 23), scale);
            tf_h8 q0, q1;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float v = qv[i] * f;
                const _Float16 hi = (_Float16)v;
                q0[i] = hi;
                q1[i] = (_Float16)(v - (float)hi);
            }
            const int r = 4 * wave + rw;
            tf_h8* slot = reinterpret_cast<tf_h8*>(lds + L::Q) + 32 * c + (r ^ c);
            slot[0] = q0;
            slot[L::TILE / 16] = q1;
            if (c == 0)
                reinterpret_cast<float*>(lds + L::S2)[r] =
                    fabsf(scale) * 1.44269504088896340736f *
                    __uint_as_float((uint32_t)(127 - fe) << 23);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // q read, fragments written
        if (tiles) issue(vbase, vt, wave * TF_PM_T, true);
        __builtin_amdgcn_s_barrier();  // the copies stay in flight over it
        asm volatile("" ::: "memory");
        s2 = reinterpret_cast<const float*>(lds + L::S2)[l32];
#pragma unroll
        for (int st = 0; st < ST; st++)
#pragma unroll
            for (int pl = 0; pl < 2; pl++)
                qb[st][pl] = reinterpret_cast<const tf_h8*>(
                    lds + L::Q)[pl * (L::TILE / 16) + 32 * (2 * st + h) + (l32 ^ (2 * st + h))];
    }

    float mx = -1e30f, l = 0.f;  // of the row; l is this half's share
    [[maybe_unused]] bool nan_row = false;
    tf_f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    const int ksw = HD == 128 ? l32 & 15 : (l32 >> 1) & 7;
    // transposing read: lane 4 a + b of 16 fetches 8 bytes of key a, dims 4 b ..,
    // and receives keys 0 .. 3 of dim 4 a + b; lanes 16 .. 31 take dims 16 ..
    const int ta = (lane & 15) >> 2, tb4 = lane & 3;
    const int vsw = HD == 128 ? ta : (ta >> 1);
    const int vrow = (4 * h + ta) * ROWB + 16 * (2 * ((lane >> 4) & 1) + (tb4 >> 1)) + 8 * (tb4 & 1);

    for (int j = wave; j < n_t; j += TF_PM_WAVES) {
        const int t0 = j * TF_PM_T;
        const bool more = j + TF_PM_WAVES < n_t;
        tf_wait_vm<NC>();  // K of tile j is there, V still on its way
        tf_f32x16 sc;
#pragma unroll
        for (int i = 0; i < 16; i++) sc[i] = 0.f;
        auto k_frag = [&](int st) {
            return *reinterpret_cast<const tf_h8*>(kt + l32 * ROWB + 16 * ((2 * st + h) ^ ksw));
        };
        if constexpr (HD == 64) {  // the second parts first, see above
            tf_h8 ka[ST];
#pragma unroll
            for (int st = 0; st < ST; st++) ka[st] = k_frag(st);
#pragma unroll
            for (int pl = 1; pl >= 0; pl--)
#pragma unroll
                for (int st = 0; st < ST; st++)
                    sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[st], qb[st][pl], sc, 0, 0, 0);
        } else {
#pragma unroll
            for (int st = 0; st < ST; st++) {
                const tf_h8 ka = k_frag(st);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qb[st][0], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qb[st][1], sc, 0, 0, 0);
            }
        }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the K tile has been read
            issue(kbase, kt, t0 + TF_PM_WAVES * TF_PM_T, false);
        }
        // the lane's keys: t0 + 8 (i / 4) + 4 h + i % 4
        const bool edge = t0 + TF_PM_T - 1 > first_pos;
        if (edge) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int kp = t0 + 8 * (i >> 2) + 4 * h + (i & 3);
                sc[i] = kp <= qpos ? sc[i] : -INFINITY;
            }
        }
        // rounded before the maximum is subtracted: a fused step would leave the
        // maximum itself above 0 by 2^-24 of a score, past f16's range for scores
        // of 2^28 and more
        tf_scores_pow2(sc, s2);
        float tmax = sc[0];
        if constexpr (HD == 64) {  // the largest of the lane's scores, or NaN if it has one
#pragma unroll
            for (int i = 1; i < 16; i++) tmax = __builtin_elementwise_maximum(tmax, sc[i]);
            nan_row |= tmax != tmax;
        }
        if (HD == 128 || __ballot(tmax != tmax)) {
            tmax = sc[0];
#pragma unroll
            for (int i = 1; i < 16; i++) tmax = fmaxf(tmax, sc[i]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float m_new = fmaxf(mx, tmax);
        if (__ballot(m_new > mx)) {
            const float alpha = __builtin_amdgcn_exp2f(mx - m_new);
            l *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
            mx = m_new;
        }
        tf_h8 pa[2][2];
        float ls = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            // a NaN score counts as no key (one instruction: med3 with 0 and 1 is the
            // exponential's own clamp)
            const float e0 = __builtin_amdgcn_fmed3f(__builtin_amdgcn_exp2f(sc[i] - mx), 0.f, 1.f);
            const float e1 =
                __builtin_amdgcn_fmed3f(__builtin_amdgcn_exp2f(sc[i + 1] - mx), 0.f, 1.f);
            ls += e0 + e1;
            tf_h2 hi, lo;
            tf_split2(e0, e1, hi, lo);
            pa[i >> 3][0][i & 7] = hi.x;
            pa[i >> 3][0][(i & 7) + 1] = hi.y;
            pa[i >> 3][1][i & 7] = lo.x;
            pa[i >> 3][1][(i & 7) + 1] = lo.y;
        }
        l += ls;
        if (more) tf_wait_vm<NC>();  // V of tile j
        else tf_wait_vm<0>();
        auto v_frag = [&](int s, int db) {
            const tf_lds_u8* vp = (const tf_lds_u8*)(vt + vrow + 16 * s * ROWB + 64 * (db ^ vsw));
            const tf_h4 v0 = __builtin_bit_cast(
                tf_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                           (__attribute__((address_space(3))) tf_s4*)vp));
            const tf_h4 v1 = __builtin_bit_cast(
                tf_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                           (__attribute__((address_space(3))) tf_s4*)(vp + 8 * ROWB)));
            return __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        if constexpr (HD == 64) {
            tf_h8 vf[2][DB];
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int db = 0; db < DB; db++) vf[s][db] = v_frag(s, db);
#pragma unroll
            for (int pl = 1; pl >= 0; pl--)
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int db = 0; db < DB; db++)
                        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[s][db], pa[s][pl], o[db],
                                                                       0, 0, 0);
        } else {
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int db = 0; db < DB; db++) {
                    const tf_h8 vf = v_frag(s, db);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pa[s][0], o[db], 0, 0, 0);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pa[s][1], o[db], 0, 0, 0);
                }
        }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the V tile has been read
            issue(vbase, vt, t0 + TF_PM_WAVES * TF_PM_T, true);
        }
    }

    // merge the waves that had tiles
    const int nw = n_t < TF_PM_WAVES ? n_t : TF_PM_WAVES;
    float* ml = reinterpret_cast<float*>(lds + L::ML);
    if (HD == 64 && nan_row) l = NAN;
    l += __shfl_xor(l, 32);
    if (h == 0) {
        ml[wave * TF_PM_T + l32] = mx;
        ml[(TF_PM_WAVES + wave) * TF_PM_T + l32] = l;
    }
    __syncthreads();
    if (wave < nw) {
        float mall = ml[l32];
        for (int w = 1; w < nw; w++) mall = fmaxf(mall, ml[w * TF_PM_T + l32]);
        const float sw = __builtin_amdgcn_exp2f(mx - mall);
        float* ow = reinterpret_cast<float*>(kt) + l32 * L::OROW + 4 * h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int b = 0; b < 4; b++)
                *reinterpret_cast<float4*>(ow + 32 * db + 8 * b) =
                    make_float4(o[db][4 * b] * sw, o[db][4 * b + 1] * sw, o[db][4 * b + 2] * sw,
                                o[db][4 * b + 3] * sw);
    }
    __syncthreads();
    // 16 threads a row, HD / 16 dims each
    const int mr = tid >> 4, r = r0 + mr;
    if (r >= n_rows) return;
    float mall = ml[mr];
    for (int w = 1; w < nw; w++) mall = fmaxf(mall, ml[w * TF_PM_T + mr]);
    float ltot = 0.f;
    for (int w = 0; w < nw; w++)
        ltot += ml[(TF_PM_WAVES + w) * TF_PM_T + mr] * __builtin_amdgcn_exp2f(ml[w * TF_PM_T + mr] - mall);
    float inv = 0x1p-14f / fmaxf(ltot, 1e-20f);  // O carries 2^14 P
    if (mall < -1.4e29f) inv = 0.f;      // no score above the mask: nothing to attend to
    if (mall == INFINITY) inv = NAN;     // an infinite score has no softmax
    const int qo = tf_div_by(r, G, g_inv);
    const size_t row = ((size_t)qo * n_head + (size_t)kv_h * G + (r - qo * G)) * HD;
    float* dst = out + row;
#pragma unroll
    for (int c = 0; c < HD / 64; c++) {
        const int d0 = 4 * (tid & 15) + 64 * c;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int w = 0; w < nw; w++) {
            const float4 v = *reinterpret_cast<const float4*>(lds + w * L::WAVE + 4 * (mr * L::OROW + d0));
            acc.x += v.x;
            acc.y += v.y;
            acc.z += v.z;
            acc.w += v.w;
        }
        acc = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
        if constexpr (HD == 64) {
            const float sum = (acc.x + acc.y) + (acc.z + acc.w);
            if (tf_row16_max(ltot != ltot || sum != sum ? 1.f : 0.f) > 0.f)
                acc = tf_attn_row64(q + row, kbase, vbase, row_bytes, pos0 + qo + 1, scale);
        }
        *reinterpret_cast<float4*>(dst + d0) = acc;
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
    if (head_dim == 256) {
        hipLaunchKernelGGL(tf_attn_prefill_kernel, dim3((n_q + TF_PA_Q - 1) / TF_PA_Q, n_head),
                           dim3(256), 0, tf_stream(stream), q, k_cache, v_cache, out, n_head, n_kv,
                           pos0, pos0_dev, n_q, scale);
        return TF_LAUNCH_RESULT();
    }
    const int G = n_head / n_kv;
    const uint32_t g_inv = G > 1 ? (uint32_t)(((1ull << 32) + G - 1) / G) : 0;
    const uint32_t kv_inv = n_kv > 1 ? (uint32_t)(((1ull << 32) + n_kv - 1) / n_kv) : 0;
    const long long tiles = ((long long)n_q * G + TF_PM_T - 1) / TF_PM_T;
    TF_CHECK_ARG(tiles * TF_PM_T <= INT32_MAX && tiles * n_kv <= UINT32_MAX / (64 * TF_PM_WAVES));
    auto go = [&](auto kern, int bytes) -> int {
        const int rc = tf_set_lds_limit((const void*)kern, bytes);
        if (rc) return rc;
        hipLaunchKernelGGL(kern, dim3((unsigned)(tiles * n_kv)), dim3(64 * TF_PM_WAVES), bytes,
                           tf_stream(stream), q, k_cache, v_cache, out, n_head, n_kv, pos0, pos0_dev,
                           n_q * G, G, g_inv, kv_inv, scale);
        return TF_LAUNCH_RESULT();
    };
    const bool a16 = (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0;
    if (head_dim == 64)
        return a16 ? go(tf_attn_prefill_mfma_kernel<64, 16>, TfPmLds<64>::BYTES)
                   : go(tf_attn_prefill_mfma_kernel<64, 4>, TfPmLds<64>::BYTES);
    return a16 ? go(tf_attn_prefill_mfma_kernel<128, 16>, TfPmLds<128>::BYTES)
               : go(tf_attn_prefill_mfma_kernel<128, 4>, TfPmLds<128>::BYTES);
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
