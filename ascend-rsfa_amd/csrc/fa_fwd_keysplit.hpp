// FlashAttention-2 forward with a task's keys split over the waves of its
// workgroup, for launches whose query blocks are too few, or causal ones too
// unequal, to fill the chip (the rule stands in rsfa_api.hip).
//
// What bounds such a launch is its longest task's chain of key tiles.  KG groups
// of 8 / KG waves share a task of 256 / KG query rows: in step s group g runs
// key tile s*KG + g with its own online softmax, and the groups merge (m, l, O)
// through LDS at the task's end, in fp32.  No workspace, no second launch and no
// traffic between workgroups; K and V are loaded once per 256 / KG rows instead
// of once per 256, which is why the groups do not pay where blocks fill the
// chip.  Schedule, operand layouts and number of waves per SIMD are the
// ping-pong kernel's (fa_fwd_kernel.hpp), with two K and two V buffers per group
// instead of three, filled by the group's own waves: with 64-key tiles at
// D = 128 two groups take 128 KB.  Q comes in through the V buffers 1, free
// until a task's second step.  Only a task's last step holds masked keys.
// Kernel times, before (best of the tiles without a split) and with it:
//   B=2 H=8 S=1024 D=128 causal      26.2 -> 15.6 us (64 rows, four groups)
//   B=1 H=8 S=4096 D=128 causal      79.0 -> 47.4
//   B=1 H=8 S=8192 D=128 causal     173.9 -> 132.7 (128 rows, two groups)
//   B=1 H=32 S=2048 D=128 causal     53.4 -> 43.1
//   B=5 H=4 S=832 D=64 causal        16.3 -> 12.5 (four)
//   B=1 H=16 S=4096 D=64 causal      57.9 -> 47.8 (two; the rule keeps whole blocks there)
//   B=2 H=8 S=2048 D=32 causal       26.5 -> 18.7 (four)
// A two-group step of 128 keys takes the cycles of two 64-key steps of the
// 256-row kernel on half the rows, about 3.0k; a task's start, merge and store
// about 13k.
#pragma once

#include "fa_fwd_kernel.hpp"

namespace rsfa {

// LDS bytes of the key-split kernel: two K and two V buffers per key group,
// or the accumulators and row states the groups exchange at a task's end.
constexpr int keysplit_lds(int d, int bn, int kg) {
    const int buffers = 4 * kg * bn * d * 2;
    const int exchange = (kg - 1) * 8 * (d / 2 / kg) * 256 + 8 * 64 * 8;
    return buffers > exchange ? buffers : exchange;
}

template <class T, int D, int BN, int KG, bool CAUSAL>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
fa_fwd_keysplit_kernel(FwdParams p) {
    typedef typename T::elem elem;
    typedef typename T::x8 x8;
    typedef typename T::x4 x4;
    typedef typename T::x2 x2;

    constexpr int NW = 8;
    constexpr int RW = NW / KG;           // waves of a key group, 32 query rows each
    constexpr int BM = 32 * RW;
    constexpr int KST = D / 16;           // 16-wide k-steps of QK^T
    constexpr int DT = D / 32;            // 32-row tiles of O^T
    constexpr int CPR = D / 8;            // 16-byte chunks per LDS row
    constexpr int NKT = BN / 32;          // 32-key sub-tiles of a key tile
    constexpr int BLK = 32 * D;           // bytes of a 16-row block
    constexpr int TILE = BN * D * 2;      // bytes of one K or V tile
    constexpr int NINST = TILE / 1024;    // 1-KB direct loads per tile
    constexpr int NSL = NINST / RW;       // ... per wave
    constexpr int QINST = BM * D * 2 / 1024;
    static_assert(D % 32 == 0 && BN % 32 == 0 && NINST % RW == 0, "whole load slices per wave");
    // only a task's last step may hold masked keys
    static_assert(BM % BN == 0 && KG * BN % BM == 0, "a block's diagonal lies in one step");

    __shared__ __attribute__((aligned(1024))) char smem_raw[keysplit_lds(D, BN, KG)];
    __shared__ int s_ticket;
    RSFA_LDS char* const smem = (RSFA_LDS char*)smem_raw;
    const uint32_t smem_addr = (uint32_t)(uintptr_t)smem;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kgi = wave / RW;  // key group
    const int rw = wave % RW;   // which 32 query rows
    const int lag = wave >> 2;  // waves 4-7 run one phase behind waves 0-3
    const int lane = tid & 63;
    const int hh = lane >> 5;
    const int l32 = lane & 31;
    const int l16 = lane & 15;

    // LDS read offsets inside a tile, as in fa_fwd_kernel
    uint32_t koff[2], voff[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) koff[e] = (l32 >> 4) * BLK + l16 * 64 + ((2 * e + hh) ^ row_swz(l16)) * 16;
    auto vrow = [&](int u) { return 8 * u + 4 * hh + (l16 >> 2); };
    const int vcc = 2 * ((lane >> 4) & 1) + ((l16 >> 1) & 1);
#pragma unroll
    for (int u = 0; u < 2; ++u)
        voff[u] = vrow(u) * 64 + (vcc ^ row_swz(vrow(u))) * 16 + 8 * (l16 & 1);
    // direct loads: lane i fills column i%4 of row i/4 of a 16-row plane
    const int ld_rib = lane >> 2;
    const int ld_chl = (lane & 3) ^ row_swz(ld_rib);
    auto slice_blk = [](int w) { return (w * 64) / (16 * CPR); };
    auto slice_cg = [](int w) { return ((w * 64) % (16 * CPR)) / 64; };
    // byte offsets of this wave's slices from a tile's first row, whose rows
    // past `last` re-read row `last`
    uint32_t kgo[NSL], vgo[NSL];
    auto set_offsets = [&](uint32_t(&go)[NSL], int64_t sn, int last) {
#pragma unroll
        for (int sl = 0; sl < NSL; ++sl) {
            const int w = sl * RW + rw;
            go[sl] = (uint32_t)((min(16 * slice_blk(w) + ld_rib, last) * sn + slice_cg(w) * 32 + ld_chl * 8) * 2);
        }
    };
    // buffers b = 0, 1 of this wave's key group
    auto kbuf = [&](int b) { return smem_addr + (b * KG + kgi) * TILE; };
    auto vbuf = [&](int b) { return smem_addr + ((2 + b) * KG + kgi) * TILE; };
    const uint32_t qbuf = smem_addr + 3 * KG * TILE;  // the V buffers 1, free until a task's second step

    const float c = p.c;
    const elem* const qg = (const elem*)p.q;
    const elem* const kg = (const elem*)p.k;
    const elem* const vg = (const elem*)p.v;
    elem* const og = (elem*)p.o;
    const int n = p.n_ctx;

    const Queue qu = make_queue<CAUSAL>(p);
    uint32_t* const ctr = p.ticket ? p.ticket + 16 * qu.x : nullptr;
    int t = task_of_ticket(qu, qu.rank);  // the counter hands out the tickets from nwg on

    while (t < qu.ntask) {
        int bh, mb;
        decode_task<CAUSAL>(p, qu, t, bh, mb);
        const int b = bh / p.H;
        const int h = bh - b * p.H;
        const int m0 = mb * BM;
        const int row0 = m0 + 32 * rw;  // this wave's first query row
        const elem* qb = qg + b * p.q_sz + h * p.q_sh;
        const elem* kh = kg + b * p.k_sz + h * p.k_sh;
        const elem* vh = vg + b * p.v_sz + h * p.v_sh;
        elem* ob = og + b * p.o_sz + h * p.o_sh;

        // Key tiles 0 .. ntile - 1; step s of key group g is tile s*KG + g.
        const int ntile = ((CAUSAL ? min(n, m0 + BM) : n) + BN - 1) / BN;
        const int nstep = (ntile + KG - 1) / KG;
        int lim = CAUSAL ? min(row0 + l32, n - 1) : n - 1;  // last key this lane sees
        const int vis_lo = CAUSAL ? min(row0, n - 1) : n - 1;       // last key every lane of the wave sees
        const int vis_hi = CAUSAL ? min(row0 + 31, n - 1) : n - 1;  // last key any lane of the wave sees
        const int64_t kstep = (int64_t)KG * BN * p.k_sn, vstep = (int64_t)KG * BN * p.v_sn;
        // the last step's tile of this group, and its last row inside the sequence
        const int jlast = (nstep - 1) * KG + kgi;
        const bool has_last = jlast < ntile;
        const int rlast = min(BN - 1, n - 1 - jlast * BN);

        const elem* kld = kh + (int64_t)kgi * BN * p.k_sn;
        const elem* vld = vh + (int64_t)kgi * BN * p.v_sn;
        auto load = [&](const elem* tp, const uint32_t(&go)[NSL], uint32_t dst, int sl) {
            dma16(tp, go[sl], dst + (sl * RW + rw) * 1024);
        };
        const bool one = nstep == 1;
        const bool ld0 = !one || has_last;
        set_offsets(kgo, p.k_sn, one ? rlast : BN - 1);
        set_offsets(vgo, p.v_sn, one ? rlast : BN - 1);
        if (ld0)
#pragma unroll
            for (int sl = 0; sl < NSL; ++sl) load(kld, kgo, kbuf(0), sl);
        // Q: the block's BM rows in the K tile layout, shared by the key groups
#pragma unroll
        for (int i = 0; i < (QINST + NW - 1) / NW; ++i) {
            const int w = i * NW + wave;
            if (QINST % NW == 0 || w < QINST) {
                const int r0 = min(m0 + 16 * slice_blk(w), n - 1);
                const int rr = min(m0 + 16 * slice_blk(w) + ld_rib, n - 1) - r0;
                const uint64_t a = (uint64_t)(uintptr_t)(qb + (int64_t)r0 * p.q_sm + slice_cg(w) * 32);
                const uint64_t ua = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                                    (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
                dma16((const void*)(uintptr_t)ua, (uint32_t)((rr * p.q_sm + ld_chl * 8) * 2), qbuf + w * 1024);
            }
        }
        // K_0 and Q first: V_0 and K_1, read two phases later, and the next ticket
        // go out once those have arrived (all at once they queue up in the CU's
        // vector-memory path: 8.2k cycles to here, 6.4k)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        phase_barrier();
        // Q^T fragments, read here by the compiler's own loads (they are in flight
        // while the direct loads below go out)
        x8 qf[KST];
        const RSFA_LDS char* const qa = smem + 3 * KG * TILE + rw * 2 * BLK;
#pragma unroll
        for (int s = 0; s < KST; ++s) qf[s] = *(const RSFA_LDS x8*)(qa + koff[s & 1] + (s >> 1) * 1024);
        if (ld0)
#pragma unroll
            for (int sl = 0; sl < NSL; ++sl) load(vld, vgo, vbuf(0), sl);
        kld += kstep;
        vld += vstep;
        if (nstep == 2) set_offsets(kgo, p.k_sn, rlast);
        if (nstep > 2 || (nstep == 2 && has_last))
#pragma unroll
            for (int sl = 0; sl < NSL; ++sl) load(kld, kgo, kbuf(1), sl);
        kld += kstep;
        int nxt = 0;
        if (ctr && tid == 0 && !pair_continues(p, qu, t)) nxt = (int)atomicAdd(ctr, 1u);
        const int qs = p.neg ? (int)0x80008000u : 0;
#pragma unroll
        for (int s = 0; s < KST; ++s) qf[s] = __builtin_bit_cast(x8, __builtin_bit_cast(i32x4, qf[s]) ^ qs);

        f32x16 o[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
        float m_use = -INFINITY;
        float l_sum = 0.0f;

        // Row max and P of one tile, as in fa_fwd_kernel; but any tile may leave
        // a row without a finite score yet: a group's first one, whose scores may
        // all be -inf while other groups' keys are not, or a masked one.
        auto softmax = [&](f32x16(&sacc)[NKT], x8(&pk)[NKT][2]) {
            float mx = sacc[0][0];
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (kt + r > 0) mx = __builtin_elementwise_maximum(mx, sacc[kt][r]);
            mx = swap_max(mx);
            const float m_tile = mx * c;
            const bool need = m_tile > m_use + RESCALE_SLACK;
            if (__builtin_amdgcn_ballot_w64(need)) {
                const float m_new = need ? m_tile : m_use;
                const float alpha = need ? __builtin_amdgcn_exp2f(m_use - m_new) : 1.0f;
                l_sum *= alpha;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
                m_use = m_new;
            }
            const float msub = m_use == -INFINITY ? 0.0f : m_use;
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kt][2 * i], c, -msub));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kt][2 * i + 1], c, -msub));
                    const x2 pr = T::cvt2(p0, p1);
                    l_sum = T::dot2(pr, T::ones2(), l_sum);
                    pk[kt][i >> 2][2 * (i & 3)] = pr[0];
                    pk[kt][i >> 2][2 * (i & 3) + 1] = pr[1];
                }
            asm volatile("" : "+v"(l_sum));
        };

        // MFMA phase: ops [from, to) of P.V of the tile in V buffer va, then S^T of
        // the tile in K buffer ka, operands read ahead as in fa_fwd_kernel; the
        // direct loads (ldk, ldv) of a whole phase go out from op D0 on.
        constexpr int NPV = DT * NKT * 2;
        constexpr int NQK = KST * NKT;
        constexpr int XPF = PV_PREFETCH;
        constexpr int XNB = XPF + 1;
        constexpr int NDMA = 2 * NSL;
        constexpr int DSTEP = (NPV + NQK) / 2 / NDMA > 0 ? (NPV + NQK) / 2 / NDMA : 1;
        constexpr int D0 = NPV + NQK - NDMA * DSTEP;
        static_assert(D0 >= 0, "operand stream shorter than its loads");
        auto x_phase = [&](auto from, auto to, uint32_t ka, uint32_t va, uint32_t kdst, uint32_t vdst, bool ldk, bool ldv,
                           const x8(&pk)[NKT][2], f32x16(&sacc)[NKT]) {
            constexpr int M0 = decltype(from)::value, M = decltype(to)::value;
            const uint32_t xa0 = va + voff[0], xa1 = va + voff[1], xk0 = ka + koff[0], xk1 = ka + koff[1];
            i32x2 rlo[XNB], rhi[XNB];
            i32x4 kr[XNB];
            auto issue = [&](auto mc) {
                constexpr int m = decltype(mc)::value;
                if constexpr (m < NPV) {
                    constexpr int d = m / (2 * NKT), kt = (m / 2) % NKT, h2 = m % 2;
                    constexpr int off = (2 * kt + h2) * BLK + d * 1024;
                    rlo[m % XNB] = lds_read_tr16<off>(xa0);
                    rhi[m % XNB] = lds_read_tr16<off>(xa1);
                } else {
                    constexpr int i = m - NPV, ss = i / NKT, kt = i % NKT;
                    kr[i % XNB] = lds_read_b128<kt * 2 * BLK + (ss >> 1) * 1024>((ss & 1) ? xk1 : xk0);
                }
            };
            static_for<XPF < M - M0 ? XPF : M - M0>([&](auto xc) { issue(std::integral_constant<int, M0 + decltype(xc)::value>()); });
            const f32x16 zero = {};
            static_for<M - M0>([&](auto mc) {
                constexpr int m = M0 + decltype(mc)::value;
                // reads issued after op m's: those of ops m + 1 .. m + XPF - 1
                constexpr int last = m + XPF - 1 < M - 1 ? m + XPF - 1 : M - 1;
                constexpr int pv_after = (last < NPV ? last : NPV - 1) - m > 0 ? (last < NPV ? last : NPV - 1) - m : 0;
                constexpr int N = (last - m) + pv_after;  // a P.V op has two
                if constexpr (m < NPV) {
                    constexpr int d = m / (2 * NKT), kt = (m / 2) % NKT, h2 = m % 2;
                    lgkm_wait2<N>(rlo[m % XNB], rhi[m % XNB]);
                    const i32x2 lo = rlo[m % XNB], hi = rhi[m % XNB];
                    o[d] = T::mfma(__builtin_bit_cast(x8, (i32x4){lo[0], lo[1], hi[0], hi[1]}), pk[kt][h2], o[d]);
                } else {
                    constexpr int i = m - NPV, ss = i / NKT, kt = i % NKT;
                    lgkm_wait<N>(kr[i % XNB]);
                    sacc[kt] = T::mfma(__builtin_bit_cast(x8, kr[i % XNB]), qf[ss], ss == 0 ? zero : sacc[kt]);
                }
                if constexpr (m + XPF < M) issue(std::integral_constant<int, m + XPF>());
                if constexpr (M0 == 0 && M > NPV && m >= D0 && (m - D0) % DSTEP == 0 && (m - D0) / DSTEP < NDMA) {
                    constexpr int q = (m - D0) / DSTEP;
                    if constexpr (q < NSL) {
                        if (ldk) load(kld, kgo, kdst, q);
                    } else {
                        if (ldv) load(vld, vgo, vdst, q - NSL);
                    }
                }
            });
        };

        const std::integral_constant<int, 0> op_0;
        const std::integral_constant<int, NPV> op_pv_end;
        const std::integral_constant<int, NPV + NQK> op_end;

        // Phases, cut by workgroup barriers: X_s = P.V of step s - 1, then S^T
        // of step s; Y_s = its softmax.  Waves 4-7 run one phase behind waves
        // 0-3 (the two waves of each SIMD).  A key group loads its own tiles:
        // X_s loads K_{s+1} and V_s into the buffers of K_{s-1} and V_{s-2},
        // last read in X_{s-1}; they are waited for at the end of Y_s.
        if (lag) phase_barrier();
        __builtin_amdgcn_s_setprio(1);
        f32x16 sacc[NKT];
        x8 pk[NKT][2];
        x_phase(op_pv_end, op_end, kbuf(0), 0, 0, 0, false, false, pk, sacc);
        int s = 0;
        uint32_t k_cur = kbuf(0), k_nxt = kbuf(1), v_cur = vbuf(0), v_nxt = vbuf(1);
        for (; s + 1 < nstep; ++s) {
            phase_barrier();  // Y_s
            __builtin_amdgcn_s_setprio(0);
            softmax(sacc, pk);
            if (s + 3 == nstep) set_offsets(kgo, p.k_sn, rlast);
            if (s + 2 == nstep) set_offsets(vgo, p.v_sn, rlast);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // V_s, K_{s+1}
            phase_barrier();  // X_{s+1}
            __builtin_amdgcn_s_setprio(1);
            x_phase(op_0, op_end, k_nxt, v_cur, k_cur, v_nxt, s + 3 < nstep || (s + 3 == nstep && has_last),
                    s + 2 < nstep || has_last, pk, sacc);
            kld += kstep;
            vld += vstep;
            const uint32_t k_old = k_cur, v_old = v_cur;
            k_cur = k_nxt;
            k_nxt = k_old;
            v_cur = v_nxt;
            v_nxt = v_old;
        }
        phase_barrier();  // Y of the last step, masked
        __builtin_amdgcn_s_setprio(0);
        const int kbase = jlast * BN;
        if (kbase + BN - 1 > vis_lo) {
            asm volatile("" : "+v"(lim));  // one comparison per score here, not masks kept in SGPRs
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kbase + 32 * kt + 8 * (i >> 2) + 4 * hh + (i & 3) > lim) sacc[kt][i] = -INFINITY;
        }
        softmax(sacc, pk);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        phase_barrier();  // its P.V
        __builtin_amdgcn_s_setprio(1);
        if (kbase + BN - 32 <= vis_hi) {
            x_phase(op_0, op_pv_end, 0, v_cur, 0, 0, false, false, pk, sacc);
        } else {
            // without the 32-key sub-tiles no row of the wave sees
            const RSFA_LDS char* const vt = smem + (v_cur - smem_addr);
#pragma unroll
            for (int kt = 0; kt + 1 < NKT; ++kt)
                if (kbase + 32 * kt <= vis_hi) {
#pragma unroll
                    for (int d = 0; d < DT; ++d)
#pragma unroll
                        for (int h2 = 0; h2 < 2; ++h2) {
                            const RSFA_LDS char* vp = vt + (2 * kt + h2) * BLK + d * 1024;
                            const i32x2 lo = __builtin_bit_cast(i32x2, T::tr_read(vp + voff[0]));
                            const i32x2 hi = __builtin_bit_cast(i32x2, T::tr_read(vp + voff[1]));
                            o[d] = T::mfma(__builtin_bit_cast(x8, (i32x4){lo[0], lo[1], hi[0], hi[1]}), pk[kt][h2], o[d]);
                        }
                }
        }
        __builtin_amdgcn_s_setprio(0);
        if (!lag) phase_barrier();
        __syncthreads();  // realigned; the tiles are done with

        // Merge of the key groups through LDS: every group finalises D / KG
        // head dims of the block.  A wave hands the other groups' shares of
        // its accumulators over as they are, with its row states (m, l).
        constexpr int OWN = DT * 16 / KG;  // accumulator registers a group finalises
        constexpr int XREG = OWN * 256;    // bytes one wave hands to another
        auto xreg = [&](int dst, int src) { return ((dst * (KG - 1) + src - (src > dst ? 1 : 0)) * RW + rw) * XREG; };
        RSFA_LDS char* const xml = smem + KG * (KG - 1) * RW * XREG;
        const float lt = swap_sum(l_sum);
        *(RSFA_LDS f32x2*)(xml + ((kgi * RW + rw) * 64 + lane) * 8) = (f32x2){m_use, lt};
        static_for<KG>([&](auto dc) {
            constexpr int dst = decltype(dc)::value;
            if (dst != kgi) {
                RSFA_LDS char* const xo = smem + xreg(dst, kgi) + lane * 16;
                static_for<OWN / 4>([&](auto qc) {
                    constexpr int r = dst * OWN + 4 * decltype(qc)::value;
                    typedef float f32x4 __attribute__((ext_vector_type(4)));
                    *(RSFA_LDS f32x4*)(xo + decltype(qc)::value * 1024) =
                        (f32x4){o[r / 16][r % 16], o[r / 16][r % 16 + 1], o[r / 16][r % 16 + 2], o[r / 16][r % 16 + 3]};
                });
            }
        });
        __syncthreads();
        float m_g[KG], l_g[KG], m_all = -INFINITY;
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            const f32x2 ml = *(const RSFA_LDS f32x2*)(xml + ((g * RW + rw) * 64 + lane) * 8);
            m_g[g] = ml[0];
            l_g[g] = ml[1];
            m_all = fmaxf(m_all, m_g[g]);
        }
        const float m_sub = m_all == -INFINITY ? 0.0f : m_all;
        float l_all = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            m_g[g] = __builtin_amdgcn_exp2f(m_g[g] - m_sub);  // the group's factor
            l_all = __builtin_fmaf(l_g[g], m_g[g], l_all);
        }
        const float inv = 1.0f / l_all;
        constexpr int OC = D / KG;         // head dims a group finalises
        constexpr int OROW = 2 * OC + 16;  // bytes per staged row
        constexpr int CH = OC / 8;         // 16-byte chunks per row
        constexpr int RPI = 64 / CH;       // rows per store instruction
        static_assert(32 * OROW <= XREG, "a staged share fits the region it was read from");
        RSFA_LDS char* const ow = smem + xreg(kgi, kgi == 0 ? 1 : 0);
        static_for<KG>([&](auto gc) {
            constexpr int g = decltype(gc)::value;
            if (g == kgi) {
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                x4 out[OWN / 4];
#pragma unroll
                for (int q = 0; q < OWN / 4; ++q) {
                    const int r = g * OWN + 4 * q;
                    f32x4 a;
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[e] = o[r / 16][r % 16 + e] * m_g[g];
#pragma unroll
                    for (int src = 0; src < KG; ++src)
                        if (src != g) {
                            const f32x4 xv = *(const RSFA_LDS f32x4*)(smem + xreg(g, src) + lane * 16 + q * 1024);
#pragma unroll
                            for (int e = 0; e < 4; ++e) a[e] = __builtin_fmaf(xv[e], m_g[src], a[e]);
                        }
#pragma unroll
                    for (int e = 0; e < 4; ++e) out[q][e] = (elem)(a[e] * inv);
                }
                // out through this wave's region of the exchange, as whole row chunks
#pragma unroll
                for (int q = 0; q < OWN / 4; ++q) *(RSFA_LDS x4*)(ow + l32 * OROW + (8 * q + 4 * hh) * 2) = out[q];
            }
        });
        {
            const int rr = lane / CH, cc = (lane % CH) * 8;
#pragma unroll
            for (int it = 0; it < (32 + RPI - 1) / RPI; ++it) {
                const int r = it * RPI + rr;
                if ((RPI <= 32 || r < 32) && row0 + r < n) {
                    const x8 v = *(const RSFA_LDS x8*)(ow + r * OROW + cc * 2);
                    *(x8*)(ob + (int64_t)(row0 + r) * p.o_sm + kgi * OC + cc) = v;
                }
            }
        }
        if (p.lse && kgi == 0 && hh == 0 && row0 + l32 < n)
            p.lse[(int64_t)bh * n + row0 + l32] = (m_sub + __log2f(l_all)) * 0.69314718055994530942f;

        __syncthreads();
        if (ctr) {
            if (pair_continues(p, qu, t)) {
                t = t + 1;
            } else {
                if (tid == 0) s_ticket = nxt;
                __syncthreads();
                t = task_of_ticket(qu, qu.nwg + __builtin_amdgcn_readfirstlane(s_ticket));
            }
        } else {
            t = pair_continues(p, qu, t) ? t + 1 : task_of_ticket(qu, ticket_of_task(qu, t) + qu.nwg);
        }
    }
    // the counter returns to zero as in fa_fwd_kernel
    if (ctr && tid == 0 && ticket_of_task(qu, t) == ticket_of_task(qu, qu.ntask) + qu.nwg - 1) atomicExch(ctr, 0u);
}

}  // namespace rsfa
