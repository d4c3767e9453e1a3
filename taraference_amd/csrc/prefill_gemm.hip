// Prefill GEMMs (n_tok > 1) for gfx950: Q4_K and Q6_K weights times f32
// activations on the matrix cores.
//
// Replaces kernels/gemm.cu gemm_q4_k (:6) and gemm_q6_k (:69) (matmul.rs:1269
// gemm): out[t][j] = sum_k W[k][j] x[t][k].  The reference dequantizes each
// weight to f32 and accumulates in fp32; here the products are formed exactly
// by v_mfma_f32_32x32x16_f16:
//   Q4_K  W = d sc q - dmin m (q in 0..15, 32-value sub-blocks): B = sc q, an
//         integer <= 945, exact in f16; the min term is one more MFMA per
//         super-block, sum over sub-blocks of m S with S the sub-block's sum
//         of x;
//   Q6_K  W = d sc (q - 32) (16-value sub-blocks): v = sc (q - 32) needs 13
//         bits, so B = f16(v) plus the remainder v - f16(v) (0 or +-1, only
//         for |v| > 2048).
// x = 2^-e (h0 + h1), h0 = f16(x 2^e), h1 = f16(x 2^e - h0), with e per
// (token, super-block) such that max |x 2^e| lies in [2^14, 2^15): the split
// keeps 22 bits.  A super-block therefore accumulates in the matrix cores (two
// MFMAs per 16 values for Q4_K; three for Q6_K, the remainder against h0 only,
// what is left out being below 2^-23 of the largest product), and d, dmin and
// 2^-e are applied in fp32 once per super-block (short Q6_K rows: all four
// products, and every 64 values, see FINE).
//
// What bounds it: the matrix cores and the vector ALU about equally.  Per
// super-block a wave's 32 x 64 tile is 64 MFMAs of 32 cycles (Q6_K: 96), and
// turning 64 columns of packed codes into B operands is about 300 vector
// instructions (Q6_K: 830).
//
// Work split: a wave owns 64 columns (two 32-column tiles) x 32 tokens.  A
// lane holds one column of each tile, so every per-column quantity (codes,
// scales, d, dmin) is read from memory by the lane that uses it, and only x
// passes through LDS.  A workgroup is CW column groups x KW slices of K:
// wide outputs take CW = 4, KW = 1 (the x image is shared by 256 columns);
// with few tiles the waves of a workgroup split K instead and add their sums
// at the end.  The runtime's prompts bring x already split (images made by
// the kernel that produces it), so their GEMMs only copy it into LDS.
//
// K order.  Within a super-block the lanes of half h (lane / 32) take bytes
// 16 h .. 16 h + 15 of each 32-byte run of codes, so a lane reads 16 contiguous
// bytes.  MFMA step (s, b), s = sub-block 0..7 of 32 values, b = 0, 1: lane half
// h supplies values 32 s + 16 h + 8 b + {0, 2, 1, 3, 4, 6, 5, 7} (the order in
// which nibbles come out of a dword), for x and W alike.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "lds_dma.hpp"
#include "prefill.hpp"
#include "tf_common.hpp"
#include "tf_host.hpp"

typedef _Float16 tf_pg_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 tf_pg_h8 __attribute__((ext_vector_type(8)));
typedef float tf_pg_f16v __attribute__((ext_vector_type(16)));
typedef float tf_pg_f4 __attribute__((ext_vector_type(4)));

// LDS image of x for 32 tokens of one super-block: 2 parts x 16 steps x 64
// lanes x 16 bytes, fragment (part, 2 s + b) being one 1 KB run in lane order
// with token t of half h at 16 * (32 h + (t ^ (4 (s & 1) + 2 h + b))): the xor
// spreads the stores of one token's eight chunks over the banks and permutes
// a fragment read within groups of eight lanes, so both run without
// conflicts.  Then the sums S 2^(e-5), [part][token][8] f16, and 2^-e.
#define TF_PG_IMG 32768
#define TF_PG_SUMS (2 * 32 * 8 * 2)
#define TF_PG_SLOT (34 * 1024)  // a whole number of 1 KB copies

__device__ __forceinline__ uint32_t tf_pg_pk(float a, float b) {
    const tf_pg_h2 h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
}
// (v & mask) | 0x64006400 in one instruction: the mask in a VGPR, the
// constant in an SGPR (VOP3 takes no literal).
__device__ __forceinline__ uint32_t tf_pg_and_or(uint32_t v, uint32_t mask) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(mask), "s"(0x64006400u));
    return r;
}
__device__ __forceinline__ uint32_t tf_pg_and_or3(uint32_t v, uint32_t mask, uint32_t o) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(o));
    return r;
}
__device__ __forceinline__ tf_pg_h2 tf_pg_fma2(tf_pg_h2 a, tf_pg_h2 b, tf_pg_h2 c) {
    return __builtin_elementwise_fma(a, b, c);
}

// Weight formats: Q4_K, raw 210-byte Q6_K blocks in memory that starts at a
// multiple of 4 bytes (W6), or of 2 (W6U), and 212-byte compact Q6_K blocks.
enum { TF_PG_W4, TF_PG_W6, TF_PG_W6U, TF_PG_W6C };

struct TfPgQkv {
    const uint8_t* w[3];
    int n_cols[3], col_bytes[3], fmt[3];
    int ct[3];   // column tiles of 256 up to and including this matrix
    int col[3];  // first output column
};

// What a lane holds of one column for one super-block.
template <bool Q6>
struct TfPgCol;
template <>
struct TfPgCol<false> {
    tf_u32x4 hd;    // d | dmin, 12 scale bytes
    tf_u32x4 q[4];  // bytes 32 c + 16 h .. + 15 of the codes
};
template <>
struct TfPgCol<true> {
    tf_u32x4 q[6];   // bytes 32 r + 16 h .. + 15 of the block: ql in r = 2 n + o, qh in 4 + n
    tf_u32x4 sc;     // 16 int8 scales
    uint32_t st, d;  // W6: the last two scales; d
};

// 16 bytes at a uniform base plus a lane's offset.
__device__ __forceinline__ tf_u32x4 tf_pg_ld16(const uint8_t* base, uint32_t off) {
    return ((const TF_GAS tf_a4x4*)(base + off))->v;
}
struct __attribute__((packed, aligned(2))) tf_a2x4 { tf_u32x4 v; };
__device__ __forceinline__ tf_u32x4 tf_pg_ld16u(const uint8_t* base, uint32_t off) {
    return ((const TF_GAS tf_a2x4*)(base + off))->v;
}
__device__ __forceinline__ uint32_t tf_pg_ld2(const uint8_t* base, uint32_t off) {
    return *(const TF_GAS uint16_t*)(base + off);
}

// Raw Q6_K blocks are 210 bytes, so every other one starts at 2 mod 4, and a
// 16-byte load from there costs four times an aligned one (3992 cache accesses
// a super-block against 1024 on the wave's 64 columns).  W6 therefore loads
// the aligned 16 bytes that begin 2 bytes earlier, `odd` lanes shift them by
// 16 bits, and the two bytes missing at the end are the first ones of the next
// run of 16, which the lane of the other half holds.  The bytes read before a
// block are the end of the block before it: the memory starts aligned.
template <int FMT>
__device__ __forceinline__ void tf_pg_load_run(const uint8_t* base, uint32_t off, uint32_t odd,
                                               int h, int r, TfPgCol<true>& c) {
    const uint32_t o = off + 32 * r + 16 * h;
    if constexpr (FMT == TF_PG_W6U) c.q[r] = tf_pg_ld16u(base, o);
    else if constexpr (FMT == TF_PG_W6) c.q[r] = tf_pg_ld16(base - 2, o + 2 - odd);
    else c.q[r] = tf_pg_ld16(base, o);
}
template <int FMT>
__device__ __forceinline__ void tf_pg_load_hdr(const uint8_t* base, uint32_t off, uint32_t odd,
                                               TfPgCol<true>& c) {
    if constexpr (FMT == TF_PG_W6U) c.sc = tf_pg_ld16u(base, off + 192);
    else c.sc = tf_pg_ld16(base, off + 192 - (FMT == TF_PG_W6 ? odd : 0));
    if constexpr (FMT == TF_PG_W6) c.st = tf_pg_ld2(base, off + 206);
    c.d = tf_pg_ld2(base, off + 208);
}
__device__ __forceinline__ tf_u32x4 tf_pg_shift(tf_u32x4 v, uint32_t next, uint32_t sh) {
    return tf_u32x4{__builtin_amdgcn_alignbit(v.y, v.x, sh), __builtin_amdgcn_alignbit(v.z, v.y, sh),
                    __builtin_amdgcn_alignbit(v.w, v.z, sh),
                    __builtin_amdgcn_alignbit(next, v.w, sh)};
}
// First dword of the run after this lane's: half 0 finds it in its partner's
// `cur`, half 1 in its partner's `nxt`.
__device__ __forceinline__ uint32_t tf_pg_next(uint32_t cur, uint32_t nxt, int h) {
    const auto s = __builtin_amdgcn_permlane32_swap(cur, nxt, false, false);
    return h ? s[0] : s[1];
}

// The scheduler moves nothing over this point: the loads of the next
// super-block are issued where their registers become free, most of a
// super-block ahead of their use.
#define TF_PG_FENCE() __builtin_amdgcn_sched_barrier(0)

// x of tokens t0 + tl (tl = st + RP j) of one super-block into its image.
// Thread (st, ci) holds the 8 values 8 ci .. 8 ci + 7 of its tokens; the 32
// threads of a token are half a wave.
template <int RP, int NP, bool SUMS>
__device__ __forceinline__ void tf_pg_store_x(const tf_pg_f4 (&xr)[NP][2], uint8_t* slot, int st,
                                              int ci) {
    const int sw = ci & 7, off = (ci >> 1 & 1) * 512 + (2 * (ci >> 2) + (ci & 1)) * 1024;
    // token st + RP j sits at ((st + RP (j mod 8/RP)) ^ sw) + 8 (RP j / 8)
    constexpr int NB = RP < 8 ? 8 / RP : 1;
    uint8_t* dst[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) dst[i] = slot + off + (((st + RP * i) ^ sw) << 4);
    _Float16* const sums = reinterpret_cast<_Float16*>(slot + TF_PG_IMG) +
                           ((ci & 1) * 32 + st) * 8 + (ci >> 2);
    uint32_t* const xinv = reinterpret_cast<uint32_t*>(slot + TF_PG_IMG + TF_PG_SUMS) + st;
#pragma unroll
    for (int j = 0; j < NP; j++) {
        const tf_pg_f4 a = xr[j][0], b = xr[j][1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i += 2)
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(amax) : "v"(v[i]), "v"(v[i + 1]));
        amax = tf_row16_max_nonneg(amax);
        // f = 2^fe, fe = 14 - floor(log2 amax), at most 126 so that 2^-fe is a
        // normal float (amax below 2^-112 then scales to below 2^14): with eb
        // the biased exponent of amax, fe + 127 = 268 - eb, eb >= 15
        uint32_t eb = max(__float_as_uint(amax), __float_as_uint(tf_swap16(amax))) & 0x7f800000u;
        eb = max(eb, 15u << 23);
        const float f = __uint_as_float((268u << 23) - eb);
        constexpr int perm[8] = {0, 2, 1, 3, 4, 6, 5, 7};
        uint32_t h0[4], h1[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float p = v[perm[2 * i]] * f, q = v[perm[2 * i + 1]] * f;
            const tf_pg_h2 hi2 = {(_Float16)p, (_Float16)q};
            h0[i] = __builtin_bit_cast(uint32_t, hi2);
            h1[i] = tf_pg_pk(p - (float)hi2[0], q - (float)hi2[1]);
        }
        uint8_t* const o = dst[j % NB] + (RP * j / 8) * 128;
        *reinterpret_cast<tf_u32x4*>(o) = tf_u32x4{h0[0], h0[1], h0[2], h0[3]};
        *reinterpret_cast<tf_u32x4*>(o + 16384) = tf_u32x4{h1[0], h1[1], h1[2], h1[3]};
        if constexpr (SUMS) {
            float gs = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            gs += tf_dpp<TF_DPP_QUAD_1032>(gs);
            gs += tf_dpp<TF_DPP_QUAD_2301>(gs);
            const float sv = gs * __uint_as_float((263u << 23) - eb);  // 2^(fe - 5): |sv| <= 2^15
            const _Float16 s0 = (_Float16)sv;
            const _Float16 s1 = (_Float16)(sv - (float)s0);
            sums[RP * j * 8] = ci & 1 ? s1 : s0;
        }
        xinv[RP * j] = eb - (14u << 23);  // 2^-fe
    }
}

// One workgroup's tile: CW x KW waves, KW slices of K of CW column groups of 64
// (DUAL: 32 of w and 32 of w2), times the 32 tokens from t0; slice z of n_split.
// PRE: x is already in images (ximg, [token tile of 32][super-block], TF_PG_SLOT
// bytes each) and is copied into LDS; otherwise the workgroup converts x itself,
// into one image a slice or, NBUF 2, two in turn.  out has rows of ldo floats.
// FINE (Q6_K): the products of h0 and the weights' f16 values are scaled and added to
// the sum after every 64 values; all smaller ones, those of h1 and the remainders
// among them, have accumulators of their own.
template <int FMT, int CW, int KW, bool PRE, int NBUF, bool DUAL, bool FINE>
__device__ __forceinline__ void tf_pg_body(uint8_t* __restrict__ lds, const uint8_t* __restrict__ w,
                                           const uint8_t* __restrict__ w2,
                                           const float* __restrict__ x,
                                           const uint8_t* __restrict__ ximg,
                                           float* __restrict__ out, int ldo, int n_rows, int n_cols,
                                           int col_bytes, int n_tok, int n_split,
                                           int t0, int ctile) {
    static_assert(!PRE || NBUF == 1, "one image a slice is copied");
    constexpr int CPW = DUAL ? 32 : 64;  // output columns of a wave
    constexpr bool Q6 = FMT != TF_PG_W4;
    constexpr int BLK = FMT == TF_PG_W4 ? 144 : FMT == TF_PG_W6C ? 212 : 210;
    constexpr int RP = 2 * CW, NP = 32 / RP;  // tokens staged per pass, passes
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wave % CW, kw = wave / CW;
    const int h = lane >> 5, l32 = lane & 31;
    uint8_t* const img0 = lds + kw * NBUF * TF_PG_SLOT;

    const int c0 = ctile * (CPW * CW) + CPW * cw;
    const int nb = n_rows / 256;
    // slice z of nz takes super-blocks [lo, hi); every slice runs n_it rounds
    // (all waves meet all barriers), those past hi with scales of 0
    const int nz = n_split * KW, z = blockIdx.z * KW + kw;
    const int lo = (int)((long long)z * nb / nz), hi = (int)((long long)(z + 1) * nb / nz);
    const int n_it = KW > 1 ? (nb + nz - 1) / nz : hi - lo;
    const int last = hi > lo ? hi - 1 : (lo < nb ? lo : nb - 1);

    // this wave's columns: a uniform base and a lane's offset
    const int cb = c0 < n_cols ? c0 : n_cols - 1;
    const uint8_t* const wbase[2] = {w + (size_t)cb * col_bytes,
                                     (DUAL ? w2 : w) + (size_t)cb * col_bytes};
    uint32_t woff[2];
    bool wodd[2];  // W6: column c starts at 2 mod 4 (then the odd super-blocks do not)
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        const int c = c0 + (DUAL ? 0 : 32 * ct) + l32;
        woff[ct] = (uint32_t)((c < n_cols ? c : n_cols - 1) - cb) * (uint32_t)col_bytes;
        wodd[ct] = ((c < n_cols ? c : n_cols - 1) & 1) && (col_bytes & 2);
    }
    // staging (rows past n_tok hold row t0's values: their outputs are not
    // written): 8-value chunk ci of the super-block, tokens st + RP j
    const int gtid = tid - 64 * CW * kw;
    const int ci = gtid & 31, st = gtid >> 5;
    tf_pg_f4 xr[PRE ? 1 : NP][2];
    auto load_x = [&](int sb) {
        if constexpr (!PRE) {
            const uint8_t* xb = reinterpret_cast<const uint8_t*>(x + (size_t)t0 * n_rows + sb * 256);
#pragma unroll
            for (int j = 0; j < NP; j++) {
                const int t = t0 + st + RP * j < n_tok ? st + RP * j : 0;
                const uint32_t o = (uint32_t)t * (uint32_t)(4 * n_rows) + 32 * ci;
                xr[j][0] = *(const TF_GAS tf_pg_f4*)(xb + o);
                xr[j][1] = *(const TF_GAS tf_pg_f4*)(xb + o + 16);
            }
        }
    };
    auto store_x = [&](uint8_t* slot) {
        if constexpr (!PRE) tf_pg_store_x<RP, NP, !Q6>(xr, slot, st, ci);
    };
    auto dma_x = [&](int sb, uint8_t* slot) {
        if constexpr (PRE) {
            const uint32_t l0 = tf_lds_off(slot);
            const uint8_t* src = ximg + ((size_t)(t0 >> 5) * nb + sb) * TF_PG_SLOT + 16 * lane;
            for (int i = cw; i < TF_PG_SLOT / 1024; i += CW)
                tf_lds_dma16(src + 1024 * i, l0 + 1024 * i);
        }
    };

    tf_pg_f16v acc[2];
#pragma unroll
    for (int ct = 0; ct < 2; ct++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[ct][i] = 0.f;

    uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u;
    asm("" : "+v"(m_lo), "+v"(m_hi));  // the masks in VGPRs (see tf_pg_and_or)

    TfPgCol<Q6> wc[2];
    auto round_sb = [&](int it) { return lo + it < hi ? lo + it : last; };
    // column ct of super-block sb: the base, and whether it starts at 2 mod 4
    auto sb_base = [&](int ct, int sb) { return wbase[ct] + (size_t)sb * BLK; };
    auto odd_of = [&](int ct, int sb) -> uint32_t {
        return FMT == TF_PG_W6 ? ((sb & 1) != (int)wodd[ct] ? 2u : 0u) : 0u;
    };
    {
        load_x(round_sb(0));
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const uint8_t* const wb = sb_base(ct, round_sb(0));
            if constexpr (!Q6) {
                wc[ct].hd = tf_pg_ld16(wb, woff[ct]);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    wc[ct].q[i] = tf_pg_ld16(wb, woff[ct] + 16 + 32 * i + 16 * h);
            } else {
                const uint32_t odd = odd_of(ct, round_sb(0));
                tf_pg_load_hdr<FMT>(wb, woff[ct], odd, wc[ct]);
#pragma unroll
                for (int r = 0; r < 6; r++) tf_pg_load_run<FMT>(wb, woff[ct], odd, h, r, wc[ct]);
            }
        }
    }
    if (NBUF == 2) {
        store_x(img0);
        load_x(round_sb(1));
    }
    for (int it = 0; it < n_it; it++) {
        const int n1 = round_sb(it + 1);
        const bool live = KW == 1 || lo + it < hi;
        uint8_t* slot = img0 + (NBUF == 2 ? (it & 1) * TF_PG_SLOT : 0);
        __syncthreads();
        if (NBUF == 2) {
            // the other image: its readers passed the barrier above
            store_x(img0 + ((it + 1) & 1) * TF_PG_SLOT);
            load_x(round_sb(it + 2));
        } else {
            store_x(slot);
            dma_x(round_sb(it), slot);
            if (PRE) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the copies landed
            __syncthreads();
            load_x(n1);
        }
        const uint8_t* const wn[2] = {sb_base(0, n1), sb_base(1, n1)};  // the next super-block
        TF_PG_FENCE();

        const uint8_t* xo[4];  // this lane's place in a fragment, by 4 (s & 1) + b
#pragma unroll
        for (int e = 0; e < 4; e++)
            xo[e] = slot + 512 * h + ((l32 ^ (2 * h + (e & 1) + 4 * (e >> 1))) << 4);
        auto xfrag = [&](int pl, int s, int b) {
            return *reinterpret_cast<const tf_pg_h8*>(xo[2 * (s & 1) + b] + 16384 * pl +
                                                      1024 * (2 * s + b));
        };
        tf_pg_f16v P[2];
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int i = 0; i < 16; i++) P[ct][i] = 0.f;

        if constexpr (!Q6) {
            float dv[2], dm[2];
            uint32_t scb[2][2];
            tf_pg_h8 mv[2];
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                const tf_u32x4 hd = wc[ct].hd;
                dv[ct] = live ? tf_h2f(hd.x) : 0.f;
                dm[ct] = live ? 32.f * tf_h2f(hd.x >> 16) : 0.f;
                scb[ct][0] = hd.y & 0x3f3f3f3fu;
                scb[ct][1] = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
                const uint32_t mn0 = hd.z & 0x3f3f3f3fu;
                const uint32_t mn1 = ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    mv[ct][i] = (_Float16)(float)((mn0 >> (8 * i)) & 255u);
                    mv[ct][4 + i] = (_Float16)(float)((mn1 >> (8 * i)) & 255u);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                uint32_t q[2][4], q8[2][4];
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    const tf_u32x4 v = wc[ct].q[c];
                    q[ct][0] = v.x; q[ct][1] = v.y; q[ct][2] = v.z; q[ct][3] = v.w;
#pragma unroll
                    for (int i = 0; i < 4; i++) q8[ct][i] = q[ct][i] >> 8;
                }
#pragma unroll
                for (int o = 0; o < 2; o++) {  // low, high nibbles: sub-block 2c + o
                    const int s = 2 * c + o;
                    tf_pg_h2 sc2[2], n2v[2];
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) {
                        // the high nibbles come out as 16 q: scale / 16
                        const float sf = (float)((scb[ct][s >> 2] >> (8 * (s & 3))) & 255u) *
                                         (o ? 0.0625f : 1.f);
                        sc2[ct] = tf_pg_h2{(_Float16)sf, (_Float16)sf};
                        n2v[ct] = sc2[ct] * tf_pg_h2{(_Float16)-1024.f, (_Float16)-1024.f};
                    }
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        tf_pg_h8 xf[2];
#pragma unroll
                        for (int pl = 0; pl < 2; pl++) xf[pl] = xfrag(pl, s, b);
                        tf_pg_h8 bw[2];
#pragma unroll
                        for (int ct = 0; ct < 2; ct++) {
                            const uint32_t mk = o ? m_hi : m_lo;
                            const uint32_t t[4] = {tf_pg_and_or(q[ct][2 * b], mk),
                                                   tf_pg_and_or(q8[ct][2 * b], mk),
                                                   tf_pg_and_or(q[ct][2 * b + 1], mk),
                                                   tf_pg_and_or(q8[ct][2 * b + 1], mk)};
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                // (1024 + q) sc - 1024 sc: one fused step, exact
                                const tf_pg_h2 r = tf_pg_fma2(__builtin_bit_cast(tf_pg_h2, t[i]),
                                                              sc2[ct], n2v[ct]);
                                bw[ct][2 * i] = r[0];
                                bw[ct][2 * i + 1] = r[1];
                            }
                        }
#pragma unroll
                        for (int pl = 0; pl < 2; pl++)
#pragma unroll
                            for (int ct = 0; ct < 2; ct++)
                                P[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[pl], bw[ct],
                                                                               P[ct], 0, 0, 0);
                    }
                }
                TF_PG_FENCE();
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
                    wc[ct].q[c] = tf_pg_ld16(wn[ct], woff[ct] + 16 + 32 * c + 16 * h);
            }
#pragma unroll
            for (int ct = 0; ct < 2; ct++) wc[ct].hd = tf_pg_ld16(wn[ct], woff[ct]);
            // acc += 2^-e (d P - 32 dmin M); C rows 8 k + 4 h + r = tokens
            const uint8_t* aux = slot + TF_PG_IMG;
            // M: K = part (half h) x 8 sub-blocks
            const tf_pg_h8 xs = *reinterpret_cast<const tf_pg_h8*>(aux + (32 * h + l32) * 16);
            tf_pg_f16v M[2];
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
#pragma unroll
                for (int i = 0; i < 16; i++) M[ct][i] = 0.f;
                M[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs, mv[ct], M[ct], 0, 0, 0);
            }
            const float* xinv = reinterpret_cast<const float*>(aux + TF_PG_SUMS);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 fi = *reinterpret_cast<const float4*>(xinv + 8 * k + 4 * h);
                const float fv[4] = {fi.x, fi.y, fi.z, fi.w};
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float t = dv[ct] * P[ct][4 * k + r] - dm[ct] * M[ct][4 * k + r];
                        acc[ct][4 * k + r] = fmaf(fv[r], t, acc[ct][4 * k + r]);
                    }
            }
        } else {
            float dv[2];
            uint32_t scw[2][4];  // bytes 0 and 2 of [k]: scales of sub-blocks 4k + h, 4k + 2 + h
            uint32_t sh[2];      // W6: bits to shift this super-block's runs by
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                dv[ct] = live ? tf_h2f(wc[ct].d) : 0.f;
                tf_u32x4 v = wc[ct].sc;
                sh[ct] = 0;
                if constexpr (FMT == TF_PG_W6) {
                    sh[ct] = odd_of(ct, round_sb(it)) * 8;
                    v = tf_pg_shift(v, wc[ct].st, sh[ct]);
                    // every run's tail, before its registers take the next super-block
                    uint32_t nx[6];
#pragma unroll
                    for (int r = 0; r < 6; r++)
                        nx[r] = tf_pg_next(wc[ct].q[r].x, r < 5 ? wc[ct].q[r + 1].x : wc[ct].sc.x, h);
#pragma unroll
                    for (int r = 0; r < 6; r++) wc[ct].q[r] = tf_pg_shift(wc[ct].q[r], nx[r], sh[ct]);
                }
                scw[ct][0] = v.x >> (8 * h);
                scw[ct][1] = v.y >> (8 * h);
                scw[ct][2] = v.z >> (8 * h);
                scw[ct][3] = v.w >> (8 * h);
            }
            TF_PG_FENCE();
#pragma unroll
            for (int ct = 0; ct < 2; ct++) tf_pg_load_hdr<FMT>(wn[ct], woff[ct], odd_of(ct, n1), wc[ct]);
            auto fold = [&](tf_pg_f16v (&p)[2]) {  // acc += 2^-e d p, p = 0
                const float* xinv = reinterpret_cast<const float*>(slot + TF_PG_IMG + TF_PG_SUMS);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float4 fi = *reinterpret_cast<const float4*>(xinv + 8 * k + 4 * h);
                    const float fv[4] = {fi.x, fi.y, fi.z, fi.w};
#pragma unroll
                    for (int ct = 0; ct < 2; ct++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int i = 4 * k + r;
                            acc[ct][i] = fmaf(fv[r], dv[ct] * p[ct][i], acc[ct][i]);
                            p[ct][i] = 0.f;
                        }
                }
            };
            [[maybe_unused]] tf_pg_f16v lo[2];
            if constexpr (FINE) {
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
#pragma unroll
                    for (int i = 0; i < 16; i++) lo[ct][i] = 0.f;
            }
#pragma unroll
            for (int n = 0; n < 2; n++) {
                uint32_t qh[2][4], qh8[2][4];
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    const tf_u32x4 v = wc[ct].q[4 + n];
                    qh[ct][0] = v.x; qh[ct][1] = v.y; qh[ct][2] = v.z; qh[ct][3] = v.w;
#pragma unroll
                    for (int i = 0; i < 4; i++) qh8[ct][i] = qh[ct][i] >> 8;
                }
#pragma unroll
                for (int o = 0; o < 2; o++) {
                    uint32_t ql[2][4], ql8[2][4];
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) {
                        const tf_u32x4 v = wc[ct].q[2 * n + o];
                        ql[ct][0] = v.x; ql[ct][1] = v.y; ql[ct][2] = v.z; ql[ct][3] = v.w;
#pragma unroll
                        for (int i = 0; i < 4; i++) ql8[ct][i] = ql[ct][i] >> 8;
                    }
#pragma unroll
                    for (int g = 0; g < 2; g++) {  // low, high nibbles
                        const int qd = 2 * g + o, s = 4 * n + qd;
                        tf_pg_h2 sc2[2];
#pragma unroll
                        for (int ct = 0; ct < 2; ct++) {
                            const float sf = (float)(int8_t)(scw[ct][s >> 1] >> (16 * (s & 1))) *
                                             (g ? 0.0625f : 1.f);
                            sc2[ct] = tf_pg_h2{(_Float16)sf, (_Float16)sf};
                        }
                        const float off = g ? -1536.f : -1056.f;  // -(1024 + 32), 32 x 16
                        const tf_pg_h2 off2 = {(_Float16)off, (_Float16)off};
                        const uint32_t mk = g ? m_hi : m_lo;
#pragma unroll
                        for (int b = 0; b < 2; b++) {
                            tf_pg_h8 xf[2];
#pragma unroll
                            for (int pl = 0; pl < 2; pl++) xf[pl] = xfrag(pl, s, b);
                            tf_pg_h8 bh[2], bl[2];
#pragma unroll
                            for (int ct = 0; ct < 2; ct++) {
#pragma unroll
                                for (int i = 0; i < 4; i++) {
                                    const int dw = 2 * b + (i >> 1);
                                    const uint32_t l = i & 1 ? ql8[ct][dw] : ql[ct][dw];
                                    const uint32_t u = i & 1 ? qh8[ct][dw] : qh[ct][dw];
                                    // the two high bits to their place above the nibble
                                    const uint32_t up = o ? u << 2 : u << 4;
                                    const uint32_t t = tf_pg_and_or3(
                                        up, g ? 0x03000300u : 0x00300030u, tf_pg_and_or(l, mk));
                                    const tf_pg_h2 q = __builtin_bit_cast(tf_pg_h2, t) + off2;
                                    const tf_pg_h2 vh = q * sc2[ct];
                                    const tf_pg_h2 vl = tf_pg_fma2(q, sc2[ct], -vh);
                                    bh[ct][2 * i] = vh[0];
                                    bh[ct][2 * i + 1] = vh[1];
                                    bl[ct][2 * i] = vl[0];
                                    bl[ct][2 * i + 1] = vl[1];
                                }
                            }
#pragma unroll
                            for (int m = 0; m < (FINE ? 4 : 3); m++)
#pragma unroll
                                for (int ct = 0; ct < 2; ct++) {
                                    tf_pg_f16v& p = FINE && m > 0 ? lo[ct] : P[ct];
                                    p = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                        xf[m & 1], m >= 2 ? bl[ct] : bh[ct], p, 0, 0, 0);
                                }
                        }
                    }
                    if constexpr (FINE) fold(P);
                    TF_PG_FENCE();
#pragma unroll
                    for (int ct = 0; ct < 2; ct++)
                        tf_pg_load_run<FMT>(wn[ct], woff[ct], odd_of(ct, n1), h, 2 * n + o, wc[ct]);
                }
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
                    tf_pg_load_run<FMT>(wn[ct], woff[ct], odd_of(ct, n1), h, 4 + n, wc[ct]);
            }
            if constexpr (FINE) fold(lo);
            else fold(P);
        }
    }
    if constexpr (KW > 1) {  // slices 1.. hand their sums to slice 0, added in slice order
        __syncthreads();  // the images are read
        float* part = reinterpret_cast<float*>(lds);
        if (kw > 0) {
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    part[(((kw - 1) * CW + cw) * 32 + 16 * ct + i) * 64 + lane] = acc[ct][i];
        }
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int q = 0; q < KW - 1; q++)
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    acc[ct][i] += part[((q * CW + cw) * 32 + 16 * ct + i) * 64 + lane];
    }
    if constexpr (DUAL) {  // silu(gate) * up
        const int c = c0 + l32;
        if (c >= n_cols) return;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = t0 + 8 * (i >> 2) + 4 * h + (i & 3);
            const float g = acc[0][i];
            if (t < n_tok) out[(size_t)t * ldo + c] = (g / (1.f + __expf(-g))) * acc[1][i];
        }
        return;
    }
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        const int c = c0 + 32 * ct + l32;
        if (c >= n_cols) continue;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = t0 + 8 * (i >> 2) + 4 * h + (i & 3);
            if (t < n_tok) out[(size_t)t * ldo + c] = acc[ct][i];
        }
    }
}

// XCD-aware tile order: workgroups go round-robin to the 8 XCDs, so XCD
// k = blockIdx.x % 8 takes the contiguous tile range [k per, (k+1) per) (token
// tiles fastest): a column tile's weights are fetched into one XCD's L2 and
// reused there by all its token tiles.  false: a workgroup of the grid's padding.
__device__ __forceinline__ bool tf_pg_tile(int ntx, int n_ct, int& tx, int& ct) {
    const int n_tiles = ntx * n_ct;
    const int per = (n_tiles + 7) >> 3;
    const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    tx = tile % ntx;
    ct = tile / ntx;
    return tile < n_tiles;
}

// Waves per SIMD: 3 where the registers allow it (Q4_K without conversion
// registers), else 2, or what four images of LDS (136 KB) leave room for.
template <int FMT, int CW, int KW, bool PRE, int NBUF, bool DUAL = false, bool FINE = false>
__global__ __launch_bounds__(64 * CW * KW, KW * NBUF >= 4            ? CW * KW / 4
                                           : PRE && FMT == TF_PG_W4 ? 3
                                           : FINE                   ? 1
                                                                    : 2) void
tf_gemm_kq_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2,
                  const float* __restrict__ x, const uint8_t* __restrict__ ximg,
                  float* __restrict__ out, int n_rows, int n_cols, int col_bytes, int n_tok,
                  int n_split, int ldo, long long split_stride) {
    __shared__ __align__(16) uint8_t lds[KW * NBUF * TF_PG_SLOT];
    constexpr int COLS = (DUAL ? 32 : 64) * CW;
    int tx, ct;
    if (!tf_pg_tile((n_tok + 31) / 32, (n_cols + COLS - 1) / COLS, tx, ct)) return;
    tf_pg_body<FMT, CW, KW, PRE, NBUF, DUAL, FINE>(
        lds, w, w2, x, ximg, out + (size_t)blockIdx.z * (size_t)split_stride, ldo, n_rows, n_cols,
        col_bytes, n_tok, n_split, tx * 32, ct);
}

// q, k and v of a prompt in one launch (their outputs side by side in rows of
// ldo floats): the column tiles of the three matrices one after the other.
template <bool FINE>
__global__ __launch_bounds__(256, FINE ? 1 : 2) void tf_pg_qkv_kernel(TfPgQkv m, const uint8_t* __restrict__ ximg,
                                                           float* __restrict__ out, int ldo,
                                                           int n_rows, int n_tok, int n_split,
                                                           long long split_stride) {
    __shared__ __align__(16) uint8_t lds[TF_PG_SLOT];
    int tx, ct;
    if (!tf_pg_tile((n_tok + 31) >> 5, m.ct[2], tx, ct)) return;
    const int i = ct < m.ct[0] ? 0 : ct < m.ct[1] ? 1 : 2;
    if (i) ct -= m.ct[i - 1];
    float* o = out + (size_t)blockIdx.z * (size_t)split_stride + m.col[i];
    auto go = [&](auto fmt) {
        tf_pg_body<decltype(fmt)::value, 4, 1, true, 1, false, FINE>(
            lds, m.w[i], nullptr, nullptr, ximg, o, ldo, n_rows, m.n_cols[i], m.col_bytes[i], n_tok,
            n_split, tx * 32, ct);
    };
    if (m.fmt[i] == TF_PG_W4) go(std::integral_constant<int, TF_PG_W4>{});
    else if (m.fmt[i] == TF_PG_W6) go(std::integral_constant<int, TF_PG_W6>{});
    else go(std::integral_constant<int, TF_PG_W6U>{});
}

// x[n_tok][n_rows] into images, [token tile of 32][super-block].
__global__ __launch_bounds__(256) void tf_pg_image_kernel(const float* __restrict__ x,
                                                          uint8_t* __restrict__ img, int n_rows,
                                                          int n_tok) {
    const int ci = threadIdx.x & 31, st = threadIdx.x >> 5;
    const int sb = blockIdx.x, t0 = 32 * blockIdx.y;
    tf_pg_f4 xr[4][2];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int t = t0 + st + 8 * j;
        const float* p = x + (size_t)(t < n_tok ? t : 0) * n_rows + sb * 256 + 8 * ci;
        xr[j][0] = *reinterpret_cast<const tf_pg_f4*>(p);
        xr[j][1] = *reinterpret_cast<const tf_pg_f4*>(p + 4);
    }
    tf_pg_store_x<8, 4, true>(xr, img + ((size_t)blockIdx.y * gridDim.x + sb) * TF_PG_SLOT, st, ci);
}

// x += the n_split slices of `part` (in order), then RMSNorm of the row and its
// image: a workgroup per token, the row kept in LDS.  The sum of squares keeps
// the reference's order (kernels/ops.cu:4-34: 256 strided fused sums, halving
// tree).  Latency bound: a thread's loads are n / 1024 times 16 bytes of every
// slice, all independent (a wave per token instead, four times the loads a
// thread: 17 us at 20 tokens and 8 slices).  At 700 tokens of 2048 and four
// slices 11.2 us, 15.2 with 4-byte loads and the parts of an image line written
// from eight XCDs.
// Rows wider than TF_PG_NORM_MAX values do not fit the LDS (ROW false): the sums go
// to x as ever and the row is read back from there.
#define TF_PG_NORM_MAX 40448  // 158 KB of row
template <bool ROW>
__global__ __launch_bounds__(256) void tf_pg_norm_image_kernel(
    float* __restrict__ x, const float* __restrict__ part, int n_split, long long split_stride,
    const float* __restrict__ w, float eps, uint8_t* __restrict__ img, int n) {
    extern __shared__ __align__(16) float row_lds[];
    __shared__ float red[1];
    const int tid = threadIdx.x;
    // Workgroup b runs on XCD b mod 8; eight consecutive tokens share the
    // image's 128-byte lines (16 bytes each), so within a whole group of 64 they
    // go to one XCD, whose L2 then holds whole lines to write back.
    int t = blockIdx.x;
    if ((t | 63) < (int)gridDim.x) t = (t & ~63) | ((t & 7) << 3) | ((t >> 3) & 7);
    float* xr = x + (size_t)t * n;
    float* const row = ROW ? row_lds : xr;
    const float* pr = part + (size_t)t * n;
#pragma unroll 2
    for (int i = 4 * tid; i < n; i += 1024) {
        tf_pg_f4 v = *reinterpret_cast<const tf_pg_f4*>(xr + i);
        if (n_split) {
            tf_pg_f4 a = *reinterpret_cast<const tf_pg_f4*>(pr + i);
#pragma unroll 4
            for (int z = 1; z < n_split; z++)
                a += *reinterpret_cast<const tf_pg_f4*>(pr + (size_t)z * (size_t)split_stride + i);
            v += a;
            *reinterpret_cast<tf_pg_f4*>(xr + i) = v;
        }
        if constexpr (ROW) *reinterpret_cast<tf_pg_f4*>(row + i) = v;
    }
    __syncthreads();
    float local = 0.f;
    for (int i = tid; i < n; i += 256) local = fmaf(row[i], row[i], local);
    // the halving tree over 256: 128 and 64 across the waves, the rest within one
    __shared__ float buf[256];
    buf[tid] = local;
    __syncthreads();
    if (tid < 64) {
        float ss = (buf[tid] + buf[tid + 128]) + (buf[tid + 64] + buf[tid + 192]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_down(ss, o);
        if (tid == 0) red[0] = 1.0f / sqrtf(ss / (float)n + eps);
    }
    __syncthreads();
    const float scale = red[0];
    const int ci = tid & 31, nb = n / 256;
    for (int sb = tid >> 5; sb < nb; sb += 8) {  // uniform per half wave
        const int k = 256 * sb + 8 * ci;
        tf_pg_f4 v[1][2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const tf_pg_f4 a = *reinterpret_cast<const tf_pg_f4*>(row + k + 4 * i);
            // the caller's vector, at any multiple of 4 bytes
            const tf_pg_f4 g = __builtin_bit_cast(
                tf_pg_f4, tf_pg_ld16(reinterpret_cast<const uint8_t*>(w), 4 * (k + 4 * i)));
#pragma unroll
            for (int q = 0; q < 4; q++) v[0][i][q] = a[q] * scale * g[q];
        }
        tf_pg_store_x<8, 1, true>(v, img + ((size_t)(t >> 5) * nb + sb) * TF_PG_SLOT, t & 31, ci);
    }
}

// x[i] += sum over z of part[z][i], z in order.
__global__ __launch_bounds__(256) void tf_pg_add_kernel(float* __restrict__ x,
                                                        const float* __restrict__ part, int n4,
                                                        int n_split, long long split_stride) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 v = reinterpret_cast<const float4*>(part)[i];
#pragma unroll 4
    for (int z = 1; z < n_split; z++) {
        const float4 q = reinterpret_cast<const float4*>(part + (size_t)z * (size_t)split_stride)[i];
        v = make_float4(v.x + q.x, v.y + q.y, v.z + q.z, v.w + q.w);
    }
    float4* o = reinterpret_cast<float4*>(x) + i;
    const float4 r = *o;
    *o = make_float4(r.x + v.x, r.y + v.y, r.z + v.z, r.w + v.w);
}

// q/k/v rows of token t (position pos0 + t) from the n_split slices of their
// GEMM (columns q | k | v): the slices' sum and the bias, q and k rotated
// (NeoX pairs (i, i + hd/2) by (pos0+t) theta^(-2i/hd)), q to q_out, k and v
// to the f16 cache.  A workgroup per token and 512 / hd heads (hd / 2 divides
// 256), one round of loads a thread; the angles of the hd / 2 pairs are formed
// once for all of its heads while the loads arrive.  Bound by its bytes: 700
// tokens of 20 heads and three slices are 30 MB, 6.3 us at the rate of a large
// copy, and take 8.6 us (9.1 with powf and sincosf in every thread, 9.8 with all
// heads of a token in one workgroup, a round after the other).
__global__ __launch_bounds__(256) void tf_pg_qkv_post_kernel(
    const float* __restrict__ part, int n_split, long long split_stride,
    const float* __restrict__ bq, const float* __restrict__ bk, const float* __restrict__ bv,
    float* __restrict__ q_out, uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, int n_head,
    int n_kv, int hd, int pos0, float theta) {
    const int t = blockIdx.x, pos = pos0 + t, half = hd / 2;
    const int nq = n_head * hd, kvd = n_kv * hd, ld = nq + 2 * kvd;
    const float* row = part + (size_t)t * ld;
    const int i = threadIdx.x % half;
    __shared__ float2 rot[256];  // cos, sin of pair i
    const int hb = blockIdx.y * (256 / half) + threadIdx.x / half;
    const int c0 = hb * hd + i, c1 = c0 + half;
    float x0 = 0.f, x1 = 0.f;
    if (hb < n_head + 2 * n_kv) {
        x0 = row[c0];
        x1 = row[c1];
#pragma unroll 4
        for (int z = 1; z < n_split; z++) {
            x0 += row[(size_t)z * (size_t)split_stride + c0];
            x1 += row[(size_t)z * (size_t)split_stride + c1];
        }
    }
    if ((int)threadIdx.x < half) {
        const float freq = powf(theta, -2.f * (float)i / (float)hd);
        const float ang = (float)pos * freq;
        float sn, cs;
        sincosf(ang, &sn, &cs);
        rot[i] = make_float2(cs, sn);
    }
    __syncthreads();
    if (hb < n_head + 2 * n_kv) {
        const float* b = hb < n_head ? bq : hb < n_head + n_kv ? bk : bv;
        const int o = hb < n_head ? c0 : hb < n_head + n_kv ? c0 - nq : c0 - nq - kvd;
        if (b) {
            x0 += b[o];
            x1 += b[o + half];
        }
        if (hb < n_head + n_kv) {
            const float cs = rot[i].x, sn = rot[i].y;
            const float r0 = x0 * cs - x1 * sn, r1 = x0 * sn + x1 * cs;
            x0 = r0;
            x1 = r1;
        }
        if (hb < n_head) {
            q_out[(size_t)t * nq + o] = x0;
            q_out[(size_t)t * nq + o + half] = x1;
        } else {
            uint16_t* c = (hb < n_head + n_kv ? kc : vc) + (size_t)pos * kvd + o;
            c[0] = tf_f2h_halfup(x0);
            c[half] = tf_f2h_halfup(x1);
        }
    }
}

// ------------------------------------------------------------------ launches

namespace {

struct TfPgJob {
    const uint8_t *w, *w2;
    const float* x;
    const uint8_t* img;
    float* out;
    int n_rows, n_cols, col_bytes, n_tok, n_split, ldo;  // ldo: floats of an output row
    hipStream_t stream;
};

template <int FMT, int CW, int KW, bool PRE, int NBUF, bool DUAL = false, bool FINE = false>
void tf_pg_go(const TfPgJob& j) {
    const int cols = (DUAL ? 32 : 64) * CW;
    const size_t tiles = (size_t)((j.n_tok + 31) / 32) *
                         (size_t)((j.n_cols + cols - 1) / cols);
    // 8 x ceil(tiles / 8) workgroups (the kernel maps them XCD by XCD; the
    // padding exits at once)
    const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)), 1, j.n_split);
    hipLaunchKernelGGL((tf_gemm_kq_kernel<FMT, CW, KW, PRE, NBUF, DUAL, FINE>), grid,
                       dim3(64 * CW * KW), 0, j.stream, j.w, j.w2, j.x, j.img, j.out, j.n_rows,
                       j.n_cols, j.col_bytes, j.n_tok, j.n_split, j.ldo,
                       (long long)j.n_tok * j.n_cols);
}

// tf_pg_go for Q6_K weights, FINE where K is short.  A super-block is 48 additions to
// one fp32 sum in the matrix cores, 1.7e-7 of the result whatever K.  The form before
// them scaled and added every 16 values, an error that grows with K but begins lower:
// against 64 bits 0.91, 1.14, 1.50, 1.70 and 2.11e-7 at K = 256, 512, 1024, 1280 and
// 2048.  FINE has 0.90, 0.93, 0.98 and 1.01e-7 at the first four.  It costs 8.9
// against 7.8 us for 256 -> 2000 at 64 tokens and 25.2 against 20.8 for 1024 -> 4096 at
// 300 (9.6 and 43.1 before); sums of 128 or 32 values in one accumulator gave 1.3 and
// 1.04e-7 at K = 256 and 22.9 and 29.2 us at K = 1024.
bool tf_pg_fine(int n_rows) { return n_rows / 256 <= 5; }
template <int FMT, int CW, int KW, bool PRE, int NBUF>
void tf_pg_go6(const TfPgJob& j) {
    if (tf_pg_fine(j.n_rows)) tf_pg_go<FMT, CW, KW, PRE, NBUF, false, true>(j);
    else tf_pg_go<FMT, CW, KW, PRE, NBUF>(j);
}

size_t tiles_of(int n_tok, int n_cols, int toks, int cols) {
    return (size_t)((n_tok + toks - 1) / toks) * (size_t)((n_cols + cols - 1) / cols);
}

int tf_pg_check(bool q6, const uint8_t* w, const float* out, int n_rows, int n_cols, int col_bytes,
                int n_tok, int blk) {
    const int nb = n_rows / 256;
    TF_CHECK_ARG(w && out && nb > 0 && n_cols > 0 && n_tok > 0);
    // nb = n_rows / 256 floors a partial last super-block away, as the
    // reference's gemm_q4_k / gemm_q6_k do (kernels/gemm.cu:28, :89); the
    // GPU tests pin that case (K = 896 -> three super-blocks)
    TF_CHECK_ARG(col_bytes >= nb * blk && (n_rows & 3) == 0);
    const int align = q6 && blk == 210 ? 2 : 4;
    TF_CHECK_ARG(((uintptr_t)w & (align - 1)) == 0 && (col_bytes & (align - 1)) == 0);
    TF_CHECK_ARG(((uintptr_t)out & 15) == 0);
    TF_CHECK_ARG(tiles_of(n_tok, n_cols, 32, 64) <= (size_t)1 << 29);
    // a lane's offset from its tile's first column or token is 32 bits: 4 GB
    // for 64 columns of weights, or for 32 rows of x
    TF_CHECK_ARG((long long)std::min(n_cols, 64) * col_bytes < (1ll << 32));
    TF_CHECK_ARG((long long)std::min(n_tok, 32) * n_rows < (1ll << 30));
    return 0;
}

// The GEMM on f32 rows.  There is no memory besides the operands, so K is
// split only inside a workgroup: 256 columns a workgroup and K whole, or fewer
// columns and K over two or four slices of its waves.  The first converts x
// once for 256 columns and needs a third of a CU's LDS, the others (four
// images) all of it.  A launch takes rounds x (a + b x super-blocks of a
// slice), the rounds being the tiles over the CUs; a and b in us, fitted to
// 256 CUs over 1..43 super-blocks, 77..11008 columns and 1..512 tokens:
//                           Q4_K           Q6_K
//   256 columns, K whole    2.8 + 3.0 n    4.4 + 3.7 n
//   128 columns, K / 4      2.0 + 8.6 n    -
//   128 columns, K / 2      -              6.5 + 4.9 n
//   64 columns, K / 4       -              6.0 + 7.0 n
// Measured at 300 tokens, 11008 -> 2048 (10 token tiles), Q6_K: 162, 113 and
// 166 us in the order above; Q4_K 2048 -> 11008 at 512: 71 and 125; 1024 ->
// 2048 at 100: 15.7 and 12.3.
void tf_pg_f32(bool q6, const TfPgJob& j) {
    const size_t cus = (size_t)tf_device_cus();
    const int nb = j.n_rows / 256;
    auto cost = [&](int cols, int kw, float a, float b) {
        const size_t rounds = (tiles_of(j.n_tok, j.n_cols, 32, cols) + cus - 1) / cus;
        return (float)rounds * (a + b * (float)((nb + kw - 1) / kw));
    };
    if (!q6) {
        if (cost(256, 1, 2.8f, 3.0f) <= cost(128, 4, 2.0f, 8.6f))
            tf_pg_go<TF_PG_W4, 4, 1, false, 1>(j);
        else
            tf_pg_go<TF_PG_W4, 2, 4, false, 1>(j);
        return;
    }
    const float whole = cost(256, 1, 4.4f, 3.7f), half = cost(128, 2, 6.5f, 4.9f),
                quarter = cost(64, 4, 6.0f, 7.0f);
    if ((uintptr_t)j.w & 2) {  // unaligned loads: the same order
        if (whole <= half) tf_pg_go6<TF_PG_W6U, 4, 1, false, 1>(j);
        else tf_pg_go6<TF_PG_W6U, 2, 2, false, 2>(j);
    } else if (whole <= half && whole <= quarter) {
        tf_pg_go6<TF_PG_W6, 4, 1, false, 1>(j);
    } else if (half <= quarter) {
        tf_pg_go6<TF_PG_W6, 2, 2, false, 2>(j);
    } else {
        tf_pg_go6<TF_PG_W6, 1, 4, false, 1>(j);
    }
}

}  // namespace

size_t tf_pg_image_bytes(int n_rows, int n_tok) {
    return (size_t)((n_tok + 31) / 32) * (size_t)(n_rows / 256) * TF_PG_SLOT;
}

int tf_pg_image(const float* x, uint8_t* img, int n_rows, int n_tok, tf_stream_t stream) {
    TF_CHECK_ARG(x && img && n_rows >= 256 && n_rows % 4 == 0 && n_tok > 0);
    TF_CHECK_ARG((((uintptr_t)x | (uintptr_t)img) & 15) == 0);
    hipLaunchKernelGGL(tf_pg_image_kernel, dim3(n_rows / 256, (n_tok + 31) / 32), dim3(256), 0,
                       tf_stream(stream), x, img, n_rows, n_tok);
    return TF_LAUNCH_RESULT();
}

int tf_pg_norm_image(float* x, const TfPgPart* part, const float* w, float eps, uint8_t* img, int n,
                     int n_tok, tf_stream_t stream) {
    TF_CHECK_ARG(x && w && img && n >= 256 && n % 256 == 0 && n_tok > 0);
    TF_CHECK_ARG((((uintptr_t)x | (uintptr_t)img) & 15) == 0);
    TF_CHECK_ARG(!part || (((uintptr_t)part->p & 15) == 0 && part->stride % 4 == 0));
    auto go = [&](auto kern, int lds) -> int {
        const int rc = tf_set_lds_limit((const void*)kern, lds);
        if (rc) return rc;
        hipLaunchKernelGGL(kern, dim3(n_tok), dim3(256), lds, tf_stream(stream), x,
                           part ? part->p : nullptr, part ? part->n_split : 0,
                           part ? part->stride : 0, w, eps, img, n);
        return TF_LAUNCH_RESULT();
    };
    if (n <= TF_PG_NORM_MAX) return go(tf_pg_norm_image_kernel<true>, n * (int)sizeof(float));
    return go(tf_pg_norm_image_kernel<false>, 0);
}

int tf_pg_add_row(float* x, const TfPgPart& part, int row, int n, tf_stream_t stream) {
    TF_CHECK_ARG(x && part.p && part.n_split > 0 && n % 4 == 0 && part.stride % 4 == 0);
    TF_CHECK_ARG((((uintptr_t)x | (uintptr_t)part.p) & 15) == 0);
    hipLaunchKernelGGL(tf_pg_add_kernel, dim3((n / 4 + 255) / 256), dim3(256), 0, tf_stream(stream),
                       x + (size_t)row * n, part.p + (size_t)row * n, n / 4, part.n_split,
                       part.stride);
    return TF_LAUNCH_RESULT();
}

// Slices of K for `tiles` output tiles: about 2.5 workgroups a CU in all, as many as
// fit ws.  Two 3B layers and the head at 1, 1.5, 2, 2.5 and 3 a CU: 1065, 981, 1010,
// 962 and 966 us for 700 tokens, 1327, 1292, 1285, 1285 and 1291 for 1024, 580, 568,
// 575, 583 and 598 for 300, no more than 2 % apart for 20 to 180.  More slices shorten
// the GEMM and lengthen the kernel that adds them.
static int tf_pg_splits(size_t tiles, int nb, size_t slice, size_t ws_floats) {
    const size_t target = 5 * (size_t)tf_device_cus() / 2;
    int n = tiles >= target ? 1 : (int)((target + tiles / 2) / tiles);
    n = std::max(1, std::min(n, std::min(nb, 16)));  // 16: what the adding kernel can hide
    while (n > 1 && (size_t)n * slice > ws_floats) n--;
    return n;
}

int tf_pg_gemm(const uint8_t* w, int block_bytes, const uint8_t* img, int n_rows, int n_cols,
               int col_bytes, int n_tok, float* ws, size_t ws_floats, TfPgPart* part,
               tf_stream_t stream) {
    const bool q6 = block_bytes != 144;
    const int rc = tf_pg_check(q6, w, ws, n_rows, n_cols, col_bytes, n_tok, block_bytes);
    if (rc) return rc;
    const size_t slice = (size_t)n_tok * n_cols;
    TF_CHECK_ARG(img && slice <= ws_floats);
    const int n_split = tf_pg_splits(tiles_of(n_tok, n_cols, 32, 256), n_rows / 256, slice, ws_floats);
    *part = TfPgPart{ws, n_split, (long long)slice};
    TfPgJob j{w, nullptr, nullptr, img, ws, n_rows, n_cols, col_bytes, n_tok, n_split, n_cols,
              tf_stream(stream)};
    if (!q6) tf_pg_go<TF_PG_W4, 4, 1, true, 1>(j);
    else if (block_bytes == 212) tf_pg_go6<TF_PG_W6C, 4, 1, true, 1>(j);
    else if ((uintptr_t)w & 2) tf_pg_go6<TF_PG_W6U, 4, 1, true, 1>(j);
    else tf_pg_go6<TF_PG_W6, 4, 1, true, 1>(j);
    return TF_LAUNCH_RESULT();
}

int tf_pg_qkv(const uint8_t* const w[3], const int block_bytes[3], const int n_cols[3],
              const int col_bytes[3], const uint8_t* img, int n_rows, int n_tok, float* ws,
              size_t ws_floats, TfPgPart* part, tf_stream_t stream) {
    TfPgQkv m{};
    int ct = 0, col = 0;
    for (int i = 0; i < 3; i++) {
        TF_CHECK_ARG(block_bytes[i] == 144 || block_bytes[i] == 210);  // no compact form
        const bool q6 = block_bytes[i] != 144;
        const int rc = tf_pg_check(q6, w[i], ws, n_rows, n_cols[i], col_bytes[i], n_tok, block_bytes[i]);
        if (rc) return rc;
        m.w[i] = w[i];
        m.n_cols[i] = n_cols[i];
        m.col_bytes[i] = col_bytes[i];
        m.fmt[i] = !q6 ? TF_PG_W4 : (uintptr_t)w[i] & 2 ? TF_PG_W6U : TF_PG_W6;
        m.col[i] = col;
        col += n_cols[i];
        m.ct[i] = ct += (n_cols[i] + 255) / 256;
    }
    const size_t slice = (size_t)n_tok * col, tiles = (size_t)((n_tok + 31) / 32) * ct;
    TF_CHECK_ARG(img && slice <= ws_floats);
    const int n_split = tf_pg_splits(tiles, n_rows / 256, slice, ws_floats);
    *part = TfPgPart{ws, n_split, (long long)slice};
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(8 * ((tiles + 7) / 8)), 1, n_split), dim3(256), 0,
                           tf_stream(stream), m, img, ws, col, n_rows, n_tok, n_split,
                           (long long)slice);
    };
    if (tf_pg_fine(n_rows)) go(tf_pg_qkv_kernel<true>);
    else go(tf_pg_qkv_kernel<false>);
    return TF_LAUNCH_RESULT();
}

int tf_pg_qkv_post(const TfPgPart& part, const float* bq, const float* bk, const float* bv,
                   float* q_out, uint16_t* k_cache, uint16_t* v_cache, int n_head, int n_kv,
                   int head_dim, int pos0, int n_tok, float theta, tf_stream_t stream) {
    TF_CHECK_ARG(part.p && q_out && k_cache && v_cache && n_head > 0 && n_kv > 0 && n_tok > 0);
    TF_CHECK_ARG(head_dim > 0 && head_dim % 2 == 0 && 256 % (head_dim / 2) == 0 && pos0 >= 0);
    const int per = 512 / head_dim;  // heads of a workgroup
    const dim3 grid(n_tok, (n_head + 2 * n_kv + per - 1) / per);
    hipLaunchKernelGGL(tf_pg_qkv_post_kernel, grid, dim3(256), 0, tf_stream(stream), part.p,
                       part.n_split, part.stride, bq, bk, bv, q_out, k_cache, v_cache, n_head, n_kv,
                       head_dim, pos0, theta);
    return TF_LAUNCH_RESULT();
}

int tf_pg_gate_up(const uint8_t* gate, const uint8_t* up, const uint8_t* img, float* out,
                  int n_rows, int n_cols, int col_bytes, int n_tok, tf_stream_t stream) {
    int rc = tf_pg_check(false, gate, out, n_rows, n_cols, col_bytes, n_tok, 144);
    if (!rc) rc = tf_pg_check(false, up, out, n_rows, n_cols, col_bytes, n_tok, 144);
    if (rc) return rc;
    TF_CHECK_ARG(img);
    const TfPgJob j{gate, up, nullptr, img, out, n_rows, n_cols, col_bytes, n_tok, 1, n_cols,
                    tf_stream(stream)};
    // a short prompt: half the columns a workgroup and K split over its waves
    // (2048 -> 2 x 11008 at 20 tokens, 86 workgroups: 31 us)
    if (tiles_of(n_tok, n_cols, 32, 128) < (size_t)tf_device_cus() * 3 / 4)
        tf_pg_go<TF_PG_W4, 2, 4, true, 1, true>(j);
    else
        tf_pg_go<TF_PG_W4, 4, 1, true, 1, true>(j);
    return TF_LAUNCH_RESULT();
}

// ---------------------------------------------------------------- C ABI

// Columns and rows so long that a launch's 32-bit offsets cannot take 64 and 32 of
// them (above 2^26 bytes and 2^25 values) go in groups that they can.
static int tf_gemm_f32(bool q6, const uint8_t* w, const float* x, float* out, int n_rows,
                       int n_cols, int col_bytes, int n_tok, tf_stream_t stream) {
    const int blk = q6 ? 210 : 144;
    TF_CHECK_ARG(x && ((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0);
    const int max_c = col_bytes < (1 << 26) ? n_cols : (int)(((1ll << 32) - 1) / col_bytes);
    const int max_t = n_rows < (1 << 25) ? n_tok : (int)(((1ll << 30) - 1) / n_rows);
    for (int t0 = 0; t0 == 0 || t0 < n_tok; t0 += max_t)
        for (int c0 = 0; c0 == 0 || c0 < n_cols; c0 += max_c) {
            const int nt = std::min(n_tok - t0, max_t), nc = std::min(n_cols - c0, max_c);
            const uint8_t* wc = w + (size_t)c0 * col_bytes;
            const int rc = tf_pg_check(q6, wc, out, n_rows, nc, col_bytes, nt, blk);
            if (rc) return rc;
            tf_pg_f32(q6, TfPgJob{wc, nullptr, x + (size_t)t0 * n_rows, nullptr,
                                  out + (size_t)t0 * n_cols + c0, n_rows, nc, col_bytes, nt, 1,
                                  n_cols, tf_stream(stream)});
        }
    return TF_LAUNCH_RESULT();
}

extern "C" int tf_gemm_q4k_f32(const uint8_t* w, const float* x, float* out, int n_rows,
                               int n_cols, int col_bytes, int n_tok, tf_stream_t stream) {
    return tf_gemm_f32(false, w, x, out, n_rows, n_cols, col_bytes, n_tok, stream);
}

extern "C" int tf_gemm_q6k_f32(const uint8_t* w, const float* x, float* out, int n_rows,
                               int n_cols, int col_bytes, int n_tok, tf_stream_t stream) {
    return tf_gemm_f32(true, w, x, out, n_rows, n_cols, col_bytes, n_tok, stream);
}
