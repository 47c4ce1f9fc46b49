// Several groups of a ragged step in one launch: the entry points qwk_*_j, a code object of their own. In the one object with all the others
// they made launches that they have nothing to do with slower, through where those kernels come to lie (5.3 -> 6.2 MB; eight Q4_K / Q6_K layers
// at four tokens 315 -> 321 us, 24 IQ3_S layers at one token 524 -> 534, with the same instructions).
//
// Every group has its own rows of x, H, record, Pg and out, so nothing orders them, and one after the other each pays its own start: the launch, the
// selection, the first round trips, the last tiles. z picks the record, of which a workgroup reads what it needs by scalar loads, as from a
// record of its own (through the kernel's argument segment: a copy of it, indexed by z, went to scratch memory where its arrays are walked).
#pragma once
#define QW_JOINED(T) (*(const qwk_##T##_join *)(const void *)__builtin_amdgcn_kernarg_segment_ptr())
#define QW_JOIN(T)                                                                                         \
    const qwk_##T##_args &a = QW_JOINED(T).g[blockIdx.z];                                                   \
    const bool idle = blockIdx.x >= QW_JOINED(T).gx[blockIdx.z]
// The same where the workgroups of all launches lie behind one another: wg, this one's number among the nwg of its launch
#define QW_JOIN_DEALT(T)                                                                                   \
    uint32_t z = 0, wg = blockIdx.x;                                                                        \
    for (; z < QW_JOIN_MAX - 1 && wg >= QW_JOINED(T).gx[z]; z++) wg -= QW_JOINED(T).gx[z];                  \
    const qwk_##T##_args &a = QW_JOINED(T).g[z];                                                            \
    const uint32_t nwg = QW_JOINED(T).gx[z]

// The experts of the selection in the order of their numbers instead of that of the record, which has gone to memory as it is (all
// threads; sc is complete before and after; results go by token and slot, so their places and bits do not depend on it). Groups that run beside
// each other then come by an expert that several of them picked at about the same time, and all but the first find it in the last-level cache.
__device__ __forceinline__ void qw_sel_by_expert(qw_sel_cache &sc, uint32_t gnb) {
    const uint32_t U = sc.U, i = threadIdx.x, ns = gnb / 4; // (U <= 256 < threads; gnb is 8 or 16)
    uint32_t e = 0, m = 0, at = 0, sl[4] = {};
    if (i < U) {
        e = sc.ue[i], m = sc.mask[i];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (j < ns) sl[j] = ((const uint32_t *)sc.slot)[i * ns + j];
#pragma unroll 8
        for (uint32_t v = 0; v < U; v++) at += sc.ue[v] < e || (sc.ue[v] == e && v < i);
    }
    __syncthreads();
    if (i < U) {
        sc.ue[at] = e, sc.mask[at] = m;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (j < ns) ((uint32_t *)sc.slot)[at * ns + j] = sl[j];
    }
    __syncthreads();
}
// Several groups' gate/up: the compute units are shared out among the groups by their work (share_units on the host), so that one start and one
// end serve all of them. Three groups of 15 tokens (512 experts of 2048 x 512, IQ3_S): 3 x 32.4 us one after the other, 76.6 like this, 73.7 with the
// experts in order (350 MB); groups of 15 and 3 52.8 in even shares, 39.9 by work. What bounds it is the stream of a compute unit's twelve waves.
struct qw_h_joined : qw_h_global {
    uint32_t wg, nwg;
    static constexpr bool shared_grid = true;
    __device__ __forceinline__ uint32_t workgroup() const { return wg; }
    __device__ __forceinline__ uint32_t workgroups() const { return nwg; }
};
#define QW_GU_J(FGU, CHGU, NAME)                                                                            \
    extern "C" __global__ __launch_bounds__(QW_WG_GU) void NAME(qwk_gu_join a) { QW_THREADS(QW_WG_GU); \
        __shared__ struct { u2 lut[(qw_has_lut(FGU) ? QW_LUT_ENTRIES : 0) + (FGU == QW_F_RT ? QW_KQ_TAB / 2 : 1)]; u4 xf[QW_XF_MAXK * 2]; qw_sel_cache sc; qw_sel_scratch ss; } L; \
        { QW_JOIN_DEALT(gu);                                                                                 \
        qw_h_joined hs = {{a.H, a.hplane}, wg, nwg};                                                          \
        gu_body<FGU, CHGU, 0, 1>(a, L.lut, L.xf, (float *)&L.ss, &L.sc, &L.ss, hs, false, [&] { qw_sel_by_expert(L.sc, a.gnb); }); \
    } }
QW_GU_J(121, 2, qwk_gu_f121_c2_j) QW_GU_J(8, 16, qwk_gu_f8_c16_j) QW_GU_J(108, 2, qwk_gu_f108_c2_j) QW_GU_J(112, 2, qwk_gu_f112_c2_j) QW_GU_J(QW_F_RT, 1, qwk_gu_rt_j)

#define QW_PRE_J(WF, SH, NAME)                                                                           \
    extern "C" __global__ __launch_bounds__(64 * QW_PRE_WAVES) void NAME(qwk_pre_join a) {               \
        __shared__ qw_pre_lds L;                                                                         \
        { QW_JOIN(pre);                                                                                  \
        if (idle) return;                                                                                \
        qw_started(a.t_start);                                                                           \
        if (blockIdx.x < a.nrouter) pre_router_any<WF>(a, L);                                            \
        else pre_shared_any<SH>(a, blockIdx.x - a.nrouter, L);                                           \
    } }
QW_PRE_J(1, QW_F_PACKED, qwk_pre_w1_s121_j) QW_PRE_J(1, 8, qwk_pre_w1_s8_j) QW_PRE_J(1, QW_F_RT, qwk_pre_w1_kq_j)
QW_PRE_J(30, QW_F_PACKED, qwk_pre_w30_s121_j) QW_PRE_J(30, 8, qwk_pre_w30_s8_j) QW_PRE_J(30, QW_F_RT, qwk_pre_w30_kq_j)

// Down by ranges: a workgroup takes at most one expert's tiles a round, and there are more experts than a group has workgroups. In rounds that are
// filled evenly (QW_RANGE_PER): full ones, and 132 experts on 128 workgroups took two rounds of which the second was all but empty. Two groups
// of 16 tokens (512 experts of 2560 x 640, IQ4_NL): 2 x 34.8 us one after the other, 107.1 in full rounds, 67.5 like this; three of 15 3 x 33.1, 106.8, 92.6.
extern "C" __global__ __launch_bounds__(QW_WG_DN) void qwk_dnr_f120_c10_s120_c10_j(qwk_dn_join a) { QW_THREADS(QW_WG_DN);
    __shared__ struct { u2 lut[QW_KQ_TAB / 2]; uint16_t arows[2 * 16 * 2 * 640]; qw_sel_cache sc; } L;
    {
        QW_JOIN_DEALT(dn);
        dn_range_body<QW_F_PACKED_NL, 10, QW_F_PACKED_NL, 10, true>(a, L.lut, L.arows, &L.sc, wg, nwg);
    }
}

constexpr uint32_t QW_DNQ_NW = QW_WG_DN / 64, QW_DNQ_RPER = (2 * 6 * 8 + QW_DNQ_NW - 1) / QW_DNQ_NW; // 2 planes x 6 row blocks x 8 column blocks at most
struct qw_dnq_asked {
    u4 rowv[QW_DNQ_RPER];
    uint32_t at[QW_DNQ_RPER], ue, mk, U, sl[4];
    float w;
};
// (as dnq_body asks for it)
__device__ __forceinline__ void dnq_ask(const qwk_dn_args &a, const qw_dnq_work &k, qw_dnq_asked &r) {
    const uint32_t K = a.topk, gnb = a.gnb, tid = threadIdx.x, lane = qw_lane(), t0 = k.t0, nt = k.nt, GU = k.GU;
    const uint32_t *ue = (const uint32_t *)(a.sel + QW_SEL_OFF_UE(gnb, K)), *mk = (const uint32_t *)(a.sel + QW_SEL_OFF_MASK(gnb, K));
    const uint8_t *sl = a.sel + QW_SEL_OFF_SLOT(gnb, K);
    const float *wg = (const float *)(a.sel + QW_SEL_OFF_W(gnb, K)) + t0 * (K + 1);
    // (GU <= 160 and nt * (K + 1) <= 44: one element a thread; a thread without one reads element 0)
    const bool rec = tid < GU, hasw = tid < nt * (K + 1);
    const uint32_t ri = rec ? tid : 0;
    r.ue = ue[ri], r.mk = mk[ri], r.U = *(const uint32_t *)a.sel;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) r.sl[j] = sl[ri * gnb + t0 + (j < nt ? j : 0)];
    r.w = wg[hasw ? tid : 0];
    const uint32_t upr = a.I / 8, cbs = upr / 8, used = nt * (K + 1), nrb = (used + 7) / 8, nunits = 2 * nrb * cbs, wv = qw_wave();
    // (I is 256 or 512, so cbs 4 or 8; a unit in use has rest < 2 nrb. A unit's part of the addresses is scalar, a lane's the same in all of
    // them, and an offset of 32 bits goes with the load: thirty instructions and a branch a load otherwise, before the table is asked for.)
    const uint32_t lr = (lane >> 2) & 7, lc = 4 * (lane >> 5) + (lane & 3), loff = 2 * (lr * a.I + 8 * lc), lat = lc * QW_DNQ_ROWS + lr;
#pragma unroll
    for (uint32_t it = 0; it < QW_DNQ_RPER; it++) {
        const uint32_t unit = wv + it * QW_DNQ_NW, cb = unit & (cbs - 1), rest = unit >> __builtin_ctz(cbs), pl = rest >= nrb, rb = rest - (pl ? nrb : 0);
        const uint32_t off = lr < (unit < nunits ? used - 8 * rb : 0) ? 0 : ~0u;
        const uint32_t sat = (pl * upr + 8 * cb) * QW_DNQ_ROWS + 8 * rb, soff = 2 * ((pl ? a.hplane : 0) + (t0 * (K + 1) + 8 * rb) * a.I + 64 * cb);
        r.at[it] = ((uint32_t)__builtin_amdgcn_readfirstlane((int)sat) + lat) | off; // (masks: a choice became a branch)
        // (a unit that is off reads the first bytes of H: a load under a condition made the compiler keep the whole array in scratch memory)
        r.rowv[it] = *(const u4 *)((const char *)a.H + (((uint32_t)__builtin_amdgcn_readfirstlane((int)soff) + loff) & ~off));
    }
}
// Down + combine by token shares (dnq_body), several launches one after the other in a workgroup: the table is in LDS once and for all, and what
// it needs for the next one is asked for behind this one's first weights. gx: their grids. Three groups of 15 tokens (512 experts, 2048 x 512 IQ3_S
// down rows): 3 x 26.9 us as launches of their own, 80.7 with the workgroups of the three behind one another in one grid, 72.3 like this.
template <int F, int CH, int FSD, int CHSD> __device__ __forceinline__ void dnq_walk(const qwk_dn_args *as, const uint32_t *gx, u2 *lut, qw_dnq_lds &L) {
    const uint32_t tid = threadIdx.x, lane = qw_lane();
    constexpr bool TAB = qw_has_lut(F) || qw_has_lut(FSD);
    constexpr bool AHEAD = F == QW_F_PACKED && FSD == F; // (the other decoders leave no registers for it: they ask when their turn comes)
    qw_dnq_asked r;
    auto from = [&](uint32_t z) { // the next launch that this workgroup has a part in
        while (z < QW_JOIN_MAX && blockIdx.x >= gx[z]) z++;
        return z;
    };
    uint32_t z = from(0);
    bool tabled = false;
    if (AHEAD && z < QW_JOIN_MAX) dnq_ask(as[z], dnq_work(as[z]), r);
    if (TAB) qw_lut_copy_issue(lut, (const u2 *)as[0].glut); // (in registers it would hold them through the whole loop, which then spills)
    while (z < QW_JOIN_MAX) {
        const qwk_dn_args &a = as[z];
        const uint32_t K = a.topk, tpw = a.tpw, rw = 16 * tpw;
        const qw_dnq_work k = dnq_work(a);
        const uint32_t g = k.g, t0 = k.t0, nt = k.nt, GU = k.GU, next = from(z + 1);
        if (!AHEAD) dnq_ask(a, k, r);
        const bool rec = tid < GU, hasw = tid < nt * (K + 1);
        if (rec) {
            uint32_t s4 = 0;
#pragma unroll
            for (uint32_t j = 0; j < 4; j++)
                if (j < nt) s4 |= r.sl[j] << (8 * j);
            L.ue[tid] = r.ue, L.mask[tid] = (uint16_t)r.mk, L.slot4[tid] = s4;
        }
        if (hasw) L.wl[tid] = r.w;
        if (tid == 0) L.U = r.U, L.q[0] = qw_threads() >> 6, L.q[1] = 0;
        __syncthreads();
        uint32_t nv = 0;
        {
            uint32_t U = L.U;
            if (U > GU) U = GU;
            const uint32_t want = (1u << nt) - 1;
            for (uint32_t u0 = 0; u0 < U; u0 += 64) {
                const uint32_t u = u0 + lane;
                const bool on = u < U && (((uint32_t)L.mask[u] >> t0) & want);
                const unsigned long long bal = __ballot(on);
                const uint32_t at = nv + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
                if (on && at < 48) L.vlist[at] = (uint16_t)u;
                nv += (uint32_t)__popcll(bal);
            }
            if (nv > 48) nv = 48; // (four tokens of ten experts: 40 at most)
        }
        const uint32_t nsh = (FSD != 0 && a.Wsd) ? 1 : 0;
        bool staged = false;
        auto ready = [&] { // called by every wave once it has asked for its first tile
            if (staged) return;
            staged = true;
#pragma unroll
            for (uint32_t it = 0; it < QW_DNQ_RPER; it++)
                if (r.at[it] != ~0u) L.hrows[r.at[it]] = r.rowv[it];
            if (TAB && !tabled) qw_lds_arrive();
            tabled = true;
            __syncthreads();
            if (AHEAD) dnq_ask(as[next < QW_JOIN_MAX ? next : z], dnq_work(as[next < QW_JOIN_MAX ? next : z]), r); // (without a next one this one's again: a load under a condition would have the arrays in scratch memory)
        };
        const qw_dnq_view V = {L.hrows, L.part, L.ue, L.slot4, L.mask, L.vlist, L.q};
        dnq_run<F, CH, false, QW_DNQ_ROWS>(a, lut, V, g, t0, nt, nv, ready);
        if (FSD != 0) {
            if (nsh) dnq_run<FSD == 0 ? F : FSD, CHSD, true, QW_DNQ_ROWS>(a, lut, V, g, t0, nt, 1, ready);
        }
        __syncthreads();
        for (uint32_t j = tid; j < nt * rw; j += qw_threads()) { // rank order, then the shared expert (qwk_cmb's arithmetic)
            const uint32_t t = j >> (4 + __builtin_ctz(tpw)), i = j & (rw - 1), r = g * rw + i;
            const float *w = L.wl + t * (K + 1), *p = L.part + t * (K + 1) * rw + i;
            float o = 0;
            for (uint32_t s = 0; s < K; s++) o = __builtin_fmaf(w[s], p[s * rw], o);
            float sh;
            if (nsh) sh = p[K * rw];
            else sh = a.Psh[(size_t)(t0 + t) * a.D + r]; // the caller's own shared product
            o = __builtin_fmaf(w[K], sh, o);
            a.out[(size_t)(t0 + t) * a.D + r] = qw_f2h(o);
            if (a.outh) qw_store_host(a.outh + (size_t)(t0 + t) * a.D + r, qw_f2h(o));
        }
        z = next;
        __syncthreads(); // (the places that the next one fills have been read)
    }
    qw_back_fin(as[0].back, as[0].fin);
}
#define QW_DNQ_J(F, CH, FSD, CHSD, NAME)                                                            \
    extern "C" __global__ __launch_bounds__(QW_WG_DN) void NAME(qwk_dn_join a) { QW_THREADS(QW_WG_DN); \
        __shared__ struct { u2 lut[qw_has_lut(F) || qw_has_lut(FSD) ? QW_LUT_ENTRIES : 1]; qw_dnq_lds d; } L; \
        dnq_walk<F, CH, FSD, CHSD>(QW_JOINED(dn).g, QW_JOINED(dn).gx, L.lut, L.d);                  \
    }
QW_DNQ_J(121, 2, 121, 2, qwk_dnq_f121_c2_s121_c2_j) QW_DNQ_J(121, 2, 8, 4, qwk_dnq_f121_c2_s8_c4_j) QW_DNQ_J(121, 1, 121, 1, qwk_dnq_f121_c1_s121_c1_j) QW_DNQ_J(121, 1, 8, 4, qwk_dnq_f121_c1_s8_c4_j)
QW_DNQ_J(108, 1, 108, 1, qwk_dnq_f108_c1_s108_c1_j) QW_DNQ_J(114, 1, 114, 1, qwk_dnq_f114_c1_s114_c1_j)

// (qwk_cmb, line by line: one body for both, and the compiler makes another qwk_cmb)
extern "C" __global__ __launch_bounds__(QW_WG_CMB) void qwk_cmb_j(qwk_cmb_join a) {
    QW_THREADS(QW_WG_CMB);
    {
        QW_JOIN(cmb);
        if (idle || blockIdx.y >= a.nbr) return;
        const uint32_t t = blockIdx.y, row = blockIdx.x * QW_WG_CMB + threadIdx.x, K = a.topk;
        if (row >= a.D) return;
        const float *w = (const float *)(a.sel + QW_SEL_OFF_W(a.gnb, K)) + t * (K + 1);
        float pg[16], wv[16];
        const float wk = w[K], ps = a.Psh[(size_t)t * a.D + row];
#pragma unroll
        for (uint32_t s = 0; s < 16; s++) {
            const uint32_t c = s < K ? s : K - 1;
            pg[s] = a.Pg[((size_t)t * K + c) * a.D + row], wv[s] = w[c];
        }
        qw_asked();
        float o = 0;
#pragma unroll
        for (uint32_t s = 0; s < 16; s++)
            if (s < K) o = __builtin_fmaf(wv[s], pg[s], o);
        o = __builtin_fmaf(wk, ps, o);
        a.out[(size_t)t * a.D + row] = qw_f2h(o);
    }
}
