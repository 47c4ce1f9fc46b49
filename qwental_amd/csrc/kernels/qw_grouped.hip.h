// The grouped product for steps of many rows: Y[m] = X[m] . W[expert]^T over tile-major weights (IQ3_S, IQ4_NL), blocked
// so that what a weight costs (its bytes, its decoding) is paid once for up to 64 packed rows and what a row costs (its
// trip through LDS) once for sixteen weight tiles.
//
// A task is (up to 64 consecutive rows of one expert, 16 weight tiles); a workgroup of eight waves gives every wave two
// tiles. K runs in steps of one block (256 values of IQ3_S, 320 of IQ4_NL): the rows' activations of a step lie in LDS for
// all waves, double buffered, copied there by direct loads while the step before is multiplied; a wave's two slabs of
// weights come through registers, one step ahead too. In a step every weight fragment is decoded once and multiplied
// into one to four groups of 16 rows. The steps of a workgroup's tasks form one sequence, so the loads of a task's first
// step are under way during the last step of the task before.
//
// Rows in LDS: units of 16 bytes (8 values); a wave's direct load of 64 of them takes 16 rows x 64 contiguous bytes (whole
// sectors of memory; eight bytes a row and lane, the layout of the decode kernels, makes 64 requests of one load). The
// loads place lane l's unit at 16 l, so the permutation that keeps operand reads free of bank conflicts is made in the
// source: row r's unit q of a group of four lies at 4 r + (q ^ (r >> 2 & 3)), and the sixteen rows of an operand read then
// touch sixteen different bank groups.
//
// Results go through LDS once more so that they leave as rows of 16-byte stores; for a gate / up pair SwiGLU is made there.
//
// Measured (Zipf(1.1) routing over 512 experts, top-10, D = 2048, I = 512; gate / up and down product, us), against the
// kernel before, in which a wave took 16 weight rows and up to 64 packed rows and read the activations from memory:
// 2048 rows 1102 + 522 -> 255 + 140 (219 + 127 with the groups listed by size), 1000 rows 573 + 273 -> 195 + 101; reference model's layer, 1082 rows 840 + 627 ->
// 268 + 212 (1000 rows, down product: 213 -> 198 with operand reads that are not paired). What bounds it: at 2048 rows the loads alone (640 MB of slabs, 335 MB of rows that every block of tiles asks
// for again) take 168 us, the arithmetic alone (vector ALU busy half of the time, LDS 53 %, matrix cores 21 %, at 1.75 GHz)
// 209. Sixteen waves of one tile each, a barrier every step instead of every four, activations a step ahead or not, all
// table values of a block at once: within 3 %.
#pragma once
#include "qw_kquants.hip.h"

#define QW_PFG_TW 2u            /* weight tiles of a wave */
#define QW_PFG_WAVES (QW_WG_PFG / 64)
#define QW_PFG_TB (QW_PFG_TW * QW_PFG_WAVES) /* tiles of a task */
#define QW_PFG_ROWS 64u
#define QW_PFG_OS 264u          /* halves between rows of the result tile in LDS (256 + 8: rows start at different banks) */

// K-steps of which the rows lie in LDS at once: a buffer holds 64 rows of one step, 32 of two or 16 of four.
__device__ __forceinline__ constexpr uint32_t qw_pfg_subs(uint32_t rows) { return rows <= 16 ? 4 : rows <= 32 ? 2 : 1; }
// Fragments of operand A from a step's rows in LDS. buf: the step's first unit; NG groups of rows.
template <uint32_t KS, int NG> struct qw_pfg_rows {
    const u4 *buf;
    uint32_t n, kg;
    static constexpr uint32_t GU = qw_pfg_subs(16 * NG) * KS / 32 * 64; // units of a group of rows in the buffer
    __device__ __forceinline__ uint32_t unit(uint32_t g, uint32_t c) const { return g * GU + (c >> 2) * 64 + 4 * n + ((c & 3) ^ ((n >> 2) & 3)); } // c: which 8 values of the step
    __device__ __forceinline__ h8 at8(uint32_t g, uint32_t c) const { return __builtin_bit_cast(h8, buf[unit(g, c)]); }
    __device__ __forceinline__ h4 at4(uint32_t g, uint32_t c4) const { return __builtin_bit_cast(h4, qw_half_read(buf, unit(g, c4 >> 1) * 16 + (c4 & 1) * 8)); } // c4: which 4 values
};

// A barrier of the workgroup behind its LDS operations only (__syncthreads also waits for every load and store in flight)
__device__ __forceinline__ void qw_wg_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}
// The same once all but the wave's last N vector memory operations have completed. One piece, so that no load is moved
// between the wait and the barrier.
template <int N> __device__ __forceinline__ void qw_wg_barrier_but() {
    static_assert(N > 0 && N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}
// Written as fused multiply-adds: left to the compiler, the first group of rows was multiplied and added in two roundings
// (its addition merged over the four row counts) and the others in one, and a row's bits depended on where it lay.
__device__ __forceinline__ void pfg_fma(f4 &acc, float d, const f4 s) {
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(d, s[i], acc[i]);
}
// LOADS: the fewest loads that bring a lane its part of one slab. The loop counts on no more than these behind the rows'
// loads (more only make its wait stricter); qwental_amd/build.py counts them in the code object, on every path.
template <int F> struct qw_pfg;
template <> struct qw_pfg<QW_F_PACKED> {
    static constexpr uint32_t KS = 256, BYTES = QW_SLAB_BYTES, LOADS = 3;
    static_assert(BYTES == 64 * (16 + 8 + 4), "a lane's bytes lie in three places");
    typedef qw_chunk<QW_F_PACKED, 1> C;
    template <int J> static __device__ __forceinline__ void look(const C (&c)[QW_PFG_TW], const qw_iq3_keys (&k)[QW_PFG_TW], const u2 *lut, u2 (&w)[QW_PFG_TW][2]) {
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) {
            uint32_t a0, a1;
            qw_iq3_addr<J>(c[t].s[0], k[t], a0, a1);
            w[t][0] = qw_lut_at(lut, a0), w[t][1] = qw_lut_at(lut, a1);
        }
    }
    // Steps J .. 7 of both tiles, NG groups of rows; v: step J's table values, read while the step before was multiplied.
    // (The barriers keep the scheduler from reading the whole block's values at once: with them in registers the kernel
    // spilled 67.)
    template <int NG, int J> static __device__ __forceinline__ void steps(const C (&c)[QW_PFG_TW], const qw_iq3_keys (&k)[QW_PFG_TW], const u2 *lut, const qw_pfg_rows<KS, NG> &x, u2 (&v)[QW_PFG_TW][2], h8 (&a)[NG], f4 (&sub)[QW_PFG_TW][NG]) {
        u2 vn[QW_PFG_TW][2];
        h8 an[NG], w[QW_PFG_TW];
        if constexpr (J < 7) {
            look<J + 1>(c, k, lut, vn);
#pragma unroll
            for (int g = 0; g < NG; g++) an[g] = x.at8(g, 8 * x.kg + J + 1);
        }
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) {
            const h2 ff = qw_iq3_factor(c[t].s[0], J / 4);
            u4 raw = {v[t][0].x, v[t][0].y, v[t][1].x, v[t][1].y};
#pragma unroll
            for (int i = 0; i < 4; i++) raw[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, (uint32_t)raw[i]) * ff);
            w[t] = __builtin_bit_cast(h8, raw);
        }
#pragma unroll
        for (int g = 0; g < NG; g++)
#pragma unroll
            for (uint32_t t = 0; t < QW_PFG_TW; t++) sub[t][g] = qw_mfma(a[g], w[t], sub[t][g]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (J < 7) steps<NG, J + 1>(c, k, lut, x, vn, an, sub);
    }
    template <int NG> static __device__ __forceinline__ void mac(const C (&c)[QW_PFG_TW], const u2 *lut, const qw_pfg_rows<KS, NG> &x, f4 (&acc)[QW_PFG_TW][4]) {
        qw_iq3_keys k[QW_PFG_TW];
        f4 sub[QW_PFG_TW][NG];
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) {
            k[t] = qw_iq3_prep(c[t].s[0]);
#pragma unroll
            for (int g = 0; g < NG; g++) sub[t][g] = f4{0, 0, 0, 0};
        }
        u2 v[QW_PFG_TW][2];
        look<0>(c, k, lut, v);
        h8 a[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) a[g] = x.at8(g, 8 * x.kg);
        steps<NG, 0>(c, k, lut, x, v, a, sub);
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++)
#pragma unroll
            for (int g = 0; g < NG; g++) pfg_fma(acc[t][g], c[t].s[0].d, sub[t][g]);
    }
};
template <> struct qw_pfg<QW_F_PACKED_NL> {
    static constexpr uint32_t KS = 320, BYTES = QW_NL_CHUNK_BYTES, LOADS = 5;
    static_assert(BYTES == 64 * (16 + 16 + 8) + 16 * 20, "a lane's bytes lie in four places, of which one is longer than the longest load");
    typedef qw_chunk<QW_F_PACKED_NL, 10> C;
    template <int NG> static __device__ __forceinline__ void mac(const C (&c)[QW_PFG_TW], const u2 *lut, const qw_pfg_rows<KS, NG> &x, f4 (&acc)[QW_PFG_TW][4]) {
#pragma unroll
        for (int b = 0; b < 10; b++) {
            h8 w[QW_PFG_TW];
#pragma unroll
            for (uint32_t t = 0; t < QW_PFG_TW; t++) w[t] = qw_iq4_pairs((const uint32_t *)lut, c[t].q[b]);
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const h8 a = qw_chunk<20, 1>::join(x.at4(g, 8 * b + x.kg), x.at4(g, 8 * b + 4 + x.kg));
#pragma unroll
                for (uint32_t t = 0; t < QW_PFG_TW; t++) {
                    f4 sub = {0, 0, 0, 0};
                    sub = qw_mfma(a, w[t], sub);
                    pfg_fma(acc[t][g], c[t].scale(b), sub);
                }
            }
        }
    }
};

template <int F> struct qw_pfg_lds {
    u2 lut[F == QW_F_PACKED ? QW_LUT_ENTRIES : QW_KQ_TAB / 2];
    u4 x[2][QW_PFG_ROWS * qw_pfg<F>::KS / 8 > QW_PFG_ROWS * QW_PFG_OS / 8 ? QW_PFG_ROWS * qw_pfg<F>::KS / 8 : QW_PFG_ROWS * QW_PFG_OS / 8];
    uint32_t m0[2048];   // the groups of rows: the first row,
    uint16_t er[2048];   // expert | rows - 1 << 10
    uint32_t last[QW_PFG_WAVES], sum[2][QW_PFG_WAVES];
};

// Entry f carries on where entry e of the table ends: the same expert, the next rows, and e is full.
__device__ __forceinline__ bool pfg_follows(const u4 e, const u4 f, uint32_t tm) { return f.z > f.y && f.x == e.x && f.y == e.z && e.z - e.y == tm; }
// The table's entries (tm rows each, an expert's one after the other) taken together to groups of up to 64 rows, listed by size:
// those of more than 48 rows first, then of more than 32, of more than 16, the others (in the table's order within each). Four
// entries a thread, two scans (first entry of each run, groups of each size before). Why by size: a task takes 6 to 12 us
// (64 rows cost almost twice what 16 do) and a workgroup has one in 256 of the list. In the table's order some
// workgroups had many long ones and the launch waited for them: 2048 rows 406.7 -> 379.4 us for the whole path, 1000 rows 286.5 ->
// 268.7, 400 rows 233.5 -> 219.9, the reference model's layer at 1000 rows 487 -> 430. Dealt there and back instead of in rounds
// from the same end (where two rounds are not full, whoever had the longest task got a second one): 386.8 -> 380.4, 275.4 -> 269.3,
// 227.0 -> 224.7, 436 -> 427; 272 rows of a layer of 256 experts of 256 x 1024 68.5 -> 62.0.
template <class L> __device__ __forceinline__ uint32_t pfg_groups(const qwk_pf_args &a, L &S, uint32_t per) {
    const uint32_t lane = qw_lane(), wave = threadIdx.x >> 6, i0 = 4 * threadIdx.x; // (threads past entry 2047 have none)
    u4 e[5]; // e[0]: the entry before the thread's first
    uint32_t used = 0;
#pragma unroll
    for (uint32_t j = 0; j < 5; j++) {
        const uint32_t i = i0 + j - 1;
        e[j] = i < a.max_tiles ? *(const u4 *)(a.tiles + 4 * i) : u4{0, 0, 0, 0};
        if (j && e[j].z > e[j].y) used |= 1u << (j - 1);
    }
    uint32_t first[4], run = 0; // index + 1 of the latest entry at or before this one that begins a run
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        if ((used >> j & 1) && !pfg_follows(e[j], e[j + 1], a.tm)) run = i0 + j + 1;
        first[j] = run;
    }
    uint32_t m = run;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(m, o);
        if (lane >= (uint32_t)o && u > m) m = u;
    }
    if (lane == 63) S.last[wave] = m;
    uint32_t before = __shfl_up(m, 1);
    if (lane == 0) before = 0;
    __syncthreads();
    for (uint32_t w = 0; w < wave; w++) before = S.last[w] > before ? S.last[w] : before;
    uint32_t rows[4], cnt[2] = {0, 0}; // rows: of the group that begins here, or 0; cnt: groups of one and two, of three and four times sixteen rows (16 bits each)
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t f = first[j] > before ? first[j] : before;
        rows[j] = 0;
        if ((used >> j & 1) && (i0 + j + 1 - f) % per == 0) {
            u4 l = e[j + 1]; // the group's last entry
            for (uint32_t i = 1; i < per && i0 + j + i < a.max_tiles; i++) {
                const u4 g = *(const u4 *)(a.tiles + 4 * (i0 + j + i));
                if (!pfg_follows(l, g, a.tm)) break;
                l = g;
            }
            rows[j] = l.z - e[j + 1].y < QW_PFG_ROWS ? l.z - e[j + 1].y : QW_PFG_ROWS;
            const uint32_t c = (rows[j] - 1) / 16, one = 1u << (c & 1) * 16;
            if (c < 2) cnt[0] += one;
            else cnt[1] += one;
        }
    }
    uint32_t at[2] = {cnt[0], cnt[1]}, total[2] = {0, 0};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u0 = __shfl_up(at[0], o), u1 = __shfl_up(at[1], o);
        if (lane >= (uint32_t)o) at[0] += u0, at[1] += u1;
    }
    if (lane == 63) S.sum[0][wave] = at[0], S.sum[1][wave] = at[1];
    __syncthreads();
    for (uint32_t h = 0; h < 2; h++) {
        at[h] -= cnt[h];
        for (uint32_t w = 0; w < QW_PFG_WAVES; w++) {
            if (w < wave) at[h] += S.sum[h][w];
            total[h] += S.sum[h][w];
        }
    }
    // the largest class first, the table's order within a class
    const uint32_t n4 = total[1] >> 16, n3 = total[1] & 0xffff, n2 = total[0] >> 16, n1 = total[0] & 0xffff;
    at[1] += n4, at[0] += (n4 + n3) << 16, at[0] += n4 + n3 + n2;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++)
        if (rows[j]) {
            const uint32_t c = (rows[j] - 1) / 16, sh = (c & 1) * 16, i = (c < 2 ? at[0] : at[1]) >> sh & 0xffff;
            if (c < 2) at[0] += 1u << sh;
            else at[1] += 1u << sh;
            S.m0[i] = e[j + 1].y;
            S.er[i] = (uint16_t)(e[j + 1].x | (rows[j] - 1) << 10);
        }
    __syncthreads();
    return n4 + n3 + n2 + n1;
}

// Where a workgroup is in its sequence of steps: task (group of rows, block of tiles) and step of K.
struct qw_pfg_cursor {
    uint32_t task, k, expert, m0, rows, tile0, step; // step: to the next task; the list goes to the workgroups in turn, there and back (who had the longest of a round has the shortest of the next)
    template <class L> __device__ __forceinline__ void look(const L &S, uint32_t nblocks) {
        const uint32_t g = task / nblocks, er = (uint32_t)__builtin_amdgcn_readfirstlane(S.er[g]);
        m0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)S.m0[g]);
        expert = er & 1023, rows = (er >> 10) + 1, tile0 = task % nblocks * QW_PFG_TB;
    }
    // n steps on. False: there is no further one (the cursor stays, so that what it points at can still be read)
    template <class L> __device__ __forceinline__ bool next(const L &S, uint32_t n, uint32_t nsteps, uint32_t nblocks, uint32_t ntasks) {
        if (k + n < nsteps) return k += n, true;
        if (task + step >= ntasks) return false;
        task += step, step = 2 * gridDim.x - step, k = 0;
        look(S, nblocks);
        return true;
    }
};
// The rows' direct loads and the result stores are written out as assembly: the compiler then counts the weight loads
// alone and waits for those of a step while the next step's stay in flight (it takes loads into LDS, loads into
// registers and stores to complete in any order, and would empty the queue at every turn). What it does not see makes
// the hardware's count larger, so its own waits stay safe; the wait for the rows is the loop's.
__device__ __forceinline__ void pfg_load_lds(const void *src_lane, uint32_t lds_wave) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src_lane), "s"(lds_wave) : "memory", "m0");
}
__device__ __forceinline__ void pfg_store16(void *p, u4 v) { asm volatile("global_store_dwordx4 %0, %1, off" : : "v"(p), "v"(v) : "memory"); }

template <int F> __device__ __forceinline__ void pfg_body(const qwk_pf_args &a, qw_pfg_lds<F> &S) {
    typedef qw_pfg<F> P;
    typedef typename P::C C;
    constexpr uint32_t KS = P::KS;
    const uint32_t lane = qw_lane(), wave = qw_wave(), n = lane & 15, kg = lane >> 4;
    if (F == QW_F_PACKED) qw_lut_copy_issue(S.lut, (const u2 *)a.glut);
    else qw_kq_tab_build((uint32_t *)S.lut);
    const uint32_t per = a.tm < QW_PFG_ROWS ? QW_PFG_ROWS / a.tm : 1;
    const uint32_t ngroups = pfg_groups(a, S, per), nblocks = (a.ntn + QW_PFG_TB - 1) / QW_PFG_TB, ntasks = ngroups * nblocks, nsteps = a.K / KS;
    qw_pfg_cursor cur; // the step being multiplied; lx, lw: the ones whose rows (one ahead) and weights (two ahead) are asked for
    cur.task = blockIdx.x, cur.k = 0, cur.step = 2 * (gridDim.x - blockIdx.x) - 1;
    qw_lds_arrive();
    __syncthreads(); // the table
    if (cur.task >= ntasks) return;
    cur.look(S, nblocks);
    auto load_rows = [&](const qw_pfg_cursor &T, u4 *dst) { // of as many steps as the buffer holds
        const uint32_t subs = qw_pfg_subs(T.rows), left = nsteps - T.k, cbs = subs * (KS / 32), use = (left < subs ? left : subs) * (KS / 32), groups = (T.rows + 15) / 16;
        const uint32_t to = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) u4 *)dst, r = lane >> 2;
        // a wave takes units (16 rows x 32 values) of one group: with four, two or one group every wave has the same number
        const uint32_t wpg = groups == 1 ? 1 : groups == 2 ? 2 : 4, g = wave % wpg;
        if (g >= groups) return;
        const uint32_t m = 16 * g + r;
        const uint16_t *src = a.X + (size_t)(T.m0 + (m < T.rows ? m : T.rows - 1)) * a.K + T.k * KS + 8 * ((lane & 3) ^ ((r >> 2) & 3)); // rows past the end repeat the last one; never stored
        for (uint32_t cb = wave / wpg; cb < use; cb += QW_PFG_WAVES / wpg) pfg_load_lds(src + 32 * cb, to + (g * cbs + cb) * 1024);
    };
    auto load_w = [&](const qw_pfg_cursor &T, C (&c)[QW_PFG_TW]) {
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) {
            uint32_t tile = T.tile0 + wave * QW_PFG_TW + t;
            tile = tile < a.ntn ? tile : a.ntn - 1; // (past the end: the last tile again, never stored)
            c[t].load(a.W + ((size_t)T.expert * a.ntn + tile) * a.rowbytes + (size_t)T.k * P::BYTES, lane);
        }
    };
    qw_pfg_cursor lx = cur, lw = cur;
    C w[2][QW_PFG_TW];
    load_w(lw, w[0]);
    load_rows(lx, S.x[0]);
    lw.next(S, 1, nsteps, nblocks, ntasks);
    load_w(lw, w[1]);
    f4 acc[QW_PFG_TW][4];
#pragma unroll
    for (uint32_t t = 0; t < QW_PFG_TW; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) acc[t][g] = f4{0, 0, 0, 0};
    uint32_t xb = 1, xk = 0, todo = 0; // the buffer with the present rows, the step it starts at, steps still in it
    bool more = true;                  // there are rows after the present ones
    auto phase = [&](auto B) -> bool {
        constexpr int b = decltype(B)::value;
        if (todo == 0) { // on to the rows that were asked for while the ones before were multiplied
            // everybody's rows (the weights of the step after this one stay in flight: they were asked for behind the rows); and everybody is done with the other buffer
            qw_wg_barrier_but<(int)(QW_PFG_TW * P::LOADS)>();
            const uint32_t subs = qw_pfg_subs(cur.rows);
            xb ^= 1, xk = cur.k, todo = nsteps - cur.k < subs ? nsteps - cur.k : subs;
            more = lx.next(S, subs, nsteps, nblocks, ntasks);
            if (more) load_rows(lx, S.x[xb ^ 1]);
        }
        todo--;
        C c[QW_PFG_TW];
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) c[t] = w[b][t];
        // (past the last step the loads go on, to where the last one pointed: their number has to be the same in every step)
        lw.next(S, 1, nsteps, nblocks, ntasks);
        load_w(lw, w[b]);
#pragma unroll
        for (uint32_t t = 0; t < QW_PFG_TW; t++) c[t].transpose();
        const u4 *x = S.x[xb] + (cur.k - xk) * (KS / 32 * 64);
        if (cur.rows <= 16) P::template mac<1>(c, S.lut, qw_pfg_rows<KS, 1>{x, n, kg}, acc);
        else if (cur.rows <= 32) P::template mac<2>(c, S.lut, qw_pfg_rows<KS, 2>{x, n, kg}, acc);
        else if (cur.rows <= 48) P::template mac<3>(c, S.lut, qw_pfg_rows<KS, 3>{x, n, kg}, acc);
        else P::template mac<4>(c, S.lut, qw_pfg_rows<KS, 4>{x, n, kg}, acc);
        if (cur.k + 1 == nsteps) {
            uint32_t here = 0; // keeps the addresses below from being made ahead of the loop and spilled
            asm volatile("" : "+v"(here));
            uint16_t *o = (uint16_t *)S.x[xb] + here;
            qw_wg_barrier(); // everybody is done with this step's rows
            const uint32_t tb = wave * QW_PFG_TW;
#pragma unroll
            for (uint32_t t = 0; t < QW_PFG_TW; t++) {
                // a tile of two matrices: rows 0..7 are matrix A's (columns 0 .. 127 of the result tile), rows 8..15 matrix B's
                const uint32_t col = a.split == 8 ? 8 * (tb + t) + (n & 7) + (n & 8) * (QW_PFG_TB) : 16 * (tb + t) + n;
#pragma unroll
                for (uint32_t g = 0; g < 4; g++) {
                    if (16 * g < cur.rows)
#pragma unroll
                        for (uint32_t j = 0; j < 4; j++) o[(16 * g + 4 * kg + j) * QW_PFG_OS + col] = qw_f2h(acc[t][g][j]);
                    acc[t][g] = f4{0, 0, 0, 0};
                }
            }
            qw_wg_barrier();
            if (a.split == 8) {
                for (uint32_t i = threadIdx.x; i < cur.rows * QW_PFG_TB; i += 64 * QW_PFG_WAVES) {
                    const uint32_t r = i / QW_PFG_TB, t = i % QW_PFG_TB, col = 8 * (cur.tile0 + t);
                    if (cur.tile0 + t >= a.ntn) continue;
                    const u4 g = *(const u4 *)(o + r * QW_PFG_OS + 8 * t), u = *(const u4 *)(o + r * QW_PFG_OS + 8 * QW_PFG_TB + 8 * t);
                    const size_t at = (size_t)(cur.m0 + r) * a.N + col;
                    pfg_store16(a.Y + at, g);
                    pfg_store16(a.Y1 + at, u);
                    if (a.H) { // from the rounded values, the product rounded once, as qwk_moe_act leaves it
                        u4 h;
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const float g0 = qw_h2f((uint16_t)g[q]), g1 = qw_h2f((uint16_t)(g[q] >> 16)), u0 = qw_h2f((uint16_t)u[q]), u1 = qw_h2f((uint16_t)(u[q] >> 16));
                            h[q] = (uint32_t)qw_f2h(g0 / (1.0f + __expf(-g0)) * u0) | (uint32_t)qw_f2h(g1 / (1.0f + __expf(-g1)) * u1) << 16;
                        }
                        pfg_store16(a.H + at, h);
                    }
                }
            } else {
                for (uint32_t i = threadIdx.x; i < cur.rows * (2 * QW_PFG_TB); i += 64 * QW_PFG_WAVES) {
                    const uint32_t r = i / (2 * QW_PFG_TB), c8 = i % (2 * QW_PFG_TB);
                    if (cur.tile0 + c8 / 2 >= a.ntn) continue;
                    pfg_store16(a.Y + (size_t)(cur.m0 + r) * a.N + 16 * cur.tile0 + 8 * c8, *(const u4 *)(o + r * QW_PFG_OS + 8 * c8));
                }
            }
        }
        if (todo) {
            cur.k++;
            return true;
        }
        cur = lx;
        return more;
    };
    for (;;) {
        if (!phase(std::integral_constant<int, 0>{})) break;
        if (!phase(std::integral_constant<int, 1>{})) break;
    }
    qw_lds_arrive(); // (nothing of this workgroup's LDS may be written after it is given away)
}
