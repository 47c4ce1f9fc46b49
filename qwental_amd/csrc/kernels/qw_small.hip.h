// The dense product for matrices that the device takes in one go (the projections of a decode step): one workgroup per tile
// of 16 rows, one wave per 256 values of K. Such a launch is bound by latency, not by bytes (4096 x 2048 in IQ3_S is 14 KB a
// compute unit), so everything a wave needs is asked for at its entry and in one round trip: its block of the sixteen rows,
// its 256 values of every token, and for IQ3_S its share of a 4 KB table. Nothing is staged for the whole workgroup: a wave
// puts its tokens into LDS for itself (coalesced loads, 512 bytes a token; read back in fragment order). The partial sums
// of the waves meet in LDS and are added in the order of K.
// The persistent kernels copy 64 KB of pre-signed table and all tokens' activations into every compute unit first
// (2 to 3 us, behind it the weights' round trip). One launch of a chain of them, one token, 2048 values, us there -> here:
// 2000 rows IQ3_S 6.0 -> 4.0, Q8_0 8.0 -> 4.9, Q4_K 8.2 -> 4.2, Q6_K 9.7 -> 5.1; 8192 rows 6.5 -> 5.8, 8.4 -> 6.5, 8.7 ->
// 5.7, 10.2 -> 6.6; 4096 x 4096 9.6 -> 6.1, 20.2 -> 6.6, 12.4 -> 5.9, 16.6 -> 7.0 (16 tokens: 16.9 -> 7.5, 22 -> 8.1).
#pragma once
#include "qw_kquants.hip.h"

// A wave's 256 values of up to 16 tokens in LDS: chunk c (8 values) of token m at (c << sh) + (m ^ (c & (2^sh - 1))), units of 16
// bytes, 2^sh >= tokens: neither the writes (a token's chunks by 32 lanes) nor the reads (16 tokens of a chunk) meet in a bank.
struct qw_afrag_small {
    const u4 *x;
    uint32_t m, sh; // m: lane & 15, taken modulo 2^sh (lanes without a token read another's; their results are not stored)
    static constexpr bool has_lo = false;
    __device__ __forceinline__ uint32_t unit(uint32_t c) const { return (c << sh) + (m ^ (c & ((1u << sh) - 1))); }
    __device__ __forceinline__ h8 at8(uint32_t k) const { return __builtin_bit_cast(h8, x[unit(k >> 3)]); }
    __device__ __forceinline__ h4 at4(uint32_t k) const { return __builtin_bit_cast(h4, ((const u2 *)x)[unit(k >> 3) * 2 + ((k >> 2) & 1)]); }
    __device__ __forceinline__ h8 hi(uint32_t k) const { return at8(k); }
    __device__ __forceinline__ h8 lo(uint32_t) const { return h8{}; }
    __device__ __forceinline__ h4 hi4(uint32_t k) const { return at4(k); }
    __device__ __forceinline__ h4 lo4(uint32_t) const { return h4{}; }
};

// The sign masks behind the table: nibble s (bit j = the sign of value j)
__device__ __forceinline__ void qw_small_signs(u2 *tab, uint32_t s) { tab[512 + s] = u2{(s & 1) << 15 | (s & 2) << 30, (s & 4) << 13 | (s & 8) << 28}; }
// Eight values of step J of an IQ3_S block from the 4 KB table: the magnitudes of two codebook entries, their signs put in by
// masks (bit j of a nibble is the sign of value j), then the sub-block factor, as in qw_iq3_step.
template <int J> __device__ __forceinline__ h8 qw_small_iq3(const qw_iq3_slice &s, const u2 *tab) {
    constexpr int t = J / 4, j = J % 4;
    const uint32_t q = s.qs[J / 2] >> (16 * (J % 2)), h = s.qh >> (8 * t + 2 * j), n = s.sg[t] >> (8 * j);
    const u2 m0 = tab[(q & 255) | (h & 1) << 8], m1 = tab[((q >> 8) & 255) | (h & 2) << 7], s0 = tab[512 + (n & 15)], s1 = tab[512 + ((n >> 4) & 15)];
    const h2 ff = qw_iq3_factor(s, t);
    u4 raw = {m0.x ^ s0.x, m0.y ^ s0.y, m1.x ^ s1.x, m1.y ^ s1.y};
#pragma unroll
    for (int i = 0; i < 4; i++) raw[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (uint32_t)raw[i]) * ff);
    return __builtin_bit_cast(h8, raw);
}
template <int J> __device__ __forceinline__ void qw_small_iq3_steps(const qw_iq3_slice &s, const u2 *tab, const qw_afrag_small &af, uint32_t kg, f4 (&sub)[2]) {
    if constexpr (J < 8) {
        sub[J & 1] = qw_mfma(af.at8(64 * kg + 8 * J), qw_small_iq3<J>(s, tab), sub[J & 1]);
        qw_small_iq3_steps<J + 1>(s, tab, af, kg, sub);
    }
}

// A block of Q4_K or Q5_K with the factors as integers, as in qw_chunk<QW_F_PACKED_Q4K>: d (q - C) sc + (C d sc - dmin m), C half of
// the range of q, (q - C) sc exact in binary16. The sums of 32 activations are made by the lane that brings them to the binary32
// matrix instruction. (Scale and minimum applied to each step's binary32 result, the sums by a matrix instruction a step, take twice
// the vector instructions. Errors to float64, 2-norm, 1024 to 4096 values, one to sixteen tokens, that form -> this one with two
// steps an accumulator: Q4_K 8.2e-8 to 1.04e-7 -> 8.1e-8 to 1.04e-7, Q5_K 8.4e-8 to 1.16e-7 -> 8.0e-8 to 1.11e-7. All eight steps in one
// accumulator lose: at 2048 values Q4_K 1.14e-7, Q5_K 1.05e-7, where both forms are at 0.8e-7 to 0.97e-7.)
template <int F, int S> __device__ __forceinline__ void qw_small_k45_steps(const qw_kq<F> &b, const qw_afrag_small &af, uint32_t kg, const uint32_t (&sc)[2], f4 (&sub)[4]) {
    if constexpr (S < 8) {
        constexpr int sh = 4 * (S & 1), q0 = F == 13 ? 6 : 4;
        uint32_t lo = (b.r[q0 + 2 * (S >> 1)] >> sh) & 0x0f0f0f0fu, hi = (b.r[q0 + 1 + 2 * (S >> 1)] >> sh) & 0x0f0f0f0fu;
        if constexpr (F == 13) lo |= ((b.r[4] >> S) & 0x01010101u) << 4, hi |= ((b.r[5] >> S) & 0x01010101u) << 4;
        const h2 f = qw_byte_h2<(S & 3)>(sc[S >> 2]);
        const h8 q = qw_bytes_h8(lo, hi, F == 13 ? 16.0f : 8.0f);
        u4 w = __builtin_bit_cast(u4, q);
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (uint32_t)w[i]) * f);
        sub[S & 3] = qw_mfma(af.at8(32 * S + 8 * kg), __builtin_bit_cast(h8, w), sub[S & 3]);
        qw_small_k45_steps<F, S + 1>(b, af, kg, sc, sub);
    }
}
template <int F> __device__ __forceinline__ void qw_small_k45(const qw_kq<F> &b, const qw_afrag_small &af, uint32_t kg, f4 &acc) {
    uint32_t sc[2], mn[2];
    qw_k4_scales(b.r + 1, sc, mn);
    f4 sub[4] = {};
    qw_small_k45_steps<F, 0>(b, af, kg, sc, sub);
    const float d = qw_h2f((uint16_t)b.r[0]), dm = qw_h2f((uint16_t)(b.r[0] >> 16));
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(d, (sub[0][i] + sub[1][i]) + (sub[2][i] + sub[3][i]), acc[i]);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        float xs = 0;
        const h2 one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int f = 0; f < 4; f++) {
            const u4 v = __builtin_bit_cast(u4, af.at8(32 * (4 * j + kg) + 8 * f));
#pragma unroll
            for (int i = 0; i < 4; i++) xs = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, (uint32_t)v[i]), one, xs, false);
        }
        const float c = __builtin_fmaf((F == 13 ? 16.0f : 8.0f) * d, (float)((sc[j] >> (8 * kg)) & 255), -dm * (float)((mn[j] >> (8 * kg)) & 255));
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xs, c, acc, 0, 0, 0);
    }
}

// 256 values of K of one tile as the wave loads and multiplies them.
template <int F> struct qw_small_blk { // Q4_K, Q5_K, Q6_K, IQ4_XS; eight blocks of IQ4_NL, binary16, bfloat16
    static constexpr int NB = qw_kq<F>::BLK_K == 256 ? 1 : 8;
    typedef qw_chunk_kq<F, NB> C;
    static constexpr uint32_t BYTES = NB * qw_kq<F>::BLK_B;
    static __device__ __forceinline__ f4 mac(const C &c, const u2 *tab, const qw_afrag_small &af, uint32_t kg) {
        f4 acc = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if constexpr (qw_kq<F>::HAS_MIN) qw_small_k45<F>(c.b[i], af, kg, acc);
            else qw_kq_block<F>(c.b[i], (const uint32_t *)tab, af, qw_kq<F>::BLK_K * i, kg, acc);
        }
        return acc;
    }
};
template <> struct qw_small_blk<8> {
    typedef qw_chunk<8, 8> C;
    static constexpr uint32_t BYTES = 8 * 34;
    static __device__ __forceinline__ f4 mac(const C &c, const u2 *, const qw_afrag_small &af, uint32_t kg) {
        f4 acc = {0, 0, 0, 0};
        c.mac(nullptr, af, 0, kg, acc);
        return acc;
    }
};
template <> struct qw_small_blk<21> {
    typedef qw_chunk<21, 1> C;
    static constexpr uint32_t BYTES = 110;
    static __device__ __forceinline__ f4 mac(const C &c, const u2 *tab, const qw_afrag_small &af, uint32_t kg) {
        f4 sub[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        qw_small_iq3_steps<0>(c.s[0], tab, af, kg, sub);
        return c.s[0].d * (sub[0] + sub[1]);
    }
};
template <> struct qw_small_blk<QW_F_PACKED> {
    typedef qw_chunk<QW_F_PACKED, 1> C;
    static constexpr uint32_t BYTES = QW_SLAB_BYTES;
    static __device__ __forceinline__ f4 mac(const C &c, const u2 *tab, const qw_afrag_small &af, uint32_t kg) { return qw_small_blk<21>::mac(c, tab, af, kg); }
};

// The workgroup's matrix, chosen by value from arguments that all come in one read. (Chosen by index they were read one after the
// other, the tile counts up to the workgroup's own, then the format, then the rest: three and more scalar round trips in front of the weights.)
struct qmvs_mat {
    const uint8_t *W;
    void *y;
    float *yh;
    uint32_t N, fmt, rowbytes, ystride;
};
template <class T> __device__ __forceinline__ T qw_pick4(uint32_t j, T a, T b, T c, T d) { return j == 0 ? a : j == 1 ? b : j == 2 ? c : d; }
__device__ __forceinline__ qmvs_mat qmvs_pick(const qwk_qmvm_args &a, uint32_t &t) { // t: tile among all of them -> of the matrix
    const uint32_t e0 = a.ntiles[0], e1 = e0 + a.ntiles[1], e2 = e1 + a.ntiles[2], n = a.nmat - 1;
    uint32_t j = (t >= e0) + (t >= e1) + (t >= e2);
    j = j < n ? j : n; // (what lies behind the last matrix in the record is not looked at)
    t -= qw_pick4(j, 0u, e0, e1, e2);
#define QW_P(v) qw_pick4(j, a.v[0], a.v[1], a.v[2], a.v[3])
    return {QW_P(W), QW_P(y), QW_P(yh), QW_P(N), QW_P(fmt), QW_P(rowbytes), QW_P(ystride)};
#undef QW_P
}
// The wave's part of tile t of a matrix: block `wave` of the rows. x: the wave's own LDS. XN: loads of two tokens, 2 XN >= nb.
template <int F, int XN> __device__ __forceinline__ f4 qmvs_part(const qwk_qmvm_args &a, const qmvs_mat &M, uint32_t t, u2 *tab, u4 *x) {
    typedef qw_small_blk<F> B;
    constexpr bool iq3 = F == 21 || F == QW_F_PACKED, iq4 = F == 20 || F == 23;
    const uint32_t lane = qw_lane(), wave = qw_wave(), n = lane & 15, kg = lane >> 4, row = 16 * t + (lane >> 2);
    // the part of the 256 units of table that this thread puts into LDS: one from 256 threads on, else four (some by several threads)
    u4 te[4];
    const bool many = a.K < 1024; // (K / 4 threads)
    if constexpr (iq3) {
        te[0] = ((const u4 *)a.ctab)[threadIdx.x & 255];
        if (many)
#pragma unroll
            for (uint32_t i = 1; i < 4; i++) te[i] = ((const u4 *)a.ctab)[(threadIdx.x + i * 64) & 255];
    }
    u4 xv[XN];
    const uint16_t *xs = a.x + wave * 256 + 8 * (lane & 31);
#pragma unroll
    for (uint32_t i = 0; i < XN; i++) {
        const uint32_t m = 2 * i + (lane >> 5);
        xv[i] = *(const u4 *)(xs + (size_t)(m < a.nb ? m : a.nb - 1) * a.xstride);
    }
    typename B::C c;
    if constexpr (F == QW_F_PACKED) c.load(M.W + (size_t)t * M.rowbytes + wave * B::BYTES, lane);
    else c.load(M.W + (size_t)(row < M.N ? row : M.N - 1) * M.rowbytes + wave * B::BYTES, lane & 3);
    if constexpr (iq3) {
        ((u4 *)tab)[threadIdx.x & 255] = te[0];
        if (many)
#pragma unroll
            for (uint32_t i = 1; i < 4; i++) ((u4 *)tab)[(threadIdx.x + i * 64) & 255] = te[i];
        if (threadIdx.x < 16) qw_small_signs(tab, threadIdx.x);
    }
    if constexpr (iq4) qw_kq_tab_build((uint32_t *)tab);
#pragma unroll
    for (uint32_t i = 0; i < XN; i++) {
        const uint32_t m = 2 * i + (lane >> 5), cc = lane & 31;
        if (m < (1u << a.sh)) x[(cc << a.sh) + (m ^ (cc & ((1u << a.sh) - 1)))] = xv[i];
    }
    if constexpr (iq3 || iq4) __syncthreads();
    else __builtin_amdgcn_wave_barrier(); // (a wave's LDS operations complete in order)
    c.transpose();
    const qw_afrag_small af = {x, n & ((1u << a.sh) - 1), a.sh};
    return B::mac(c, tab, af, kg);
}
