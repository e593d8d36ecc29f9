// Fast-block H*v (hv_fb_*) and the slab pass that takes its degree-three slow
// terms (hv_slab_kernel).
#include "nv_hvcore.hpp"

namespace nv {

// ------------------------------------------------------------------------
// Fast-block H*v (tables in NvFbDev).  A wave owns one block of P <= 64
// consecutive rows, lane p = row row0 + p: the trailing ("fast") modes vary
// across the lanes and the slow digits are the same for the whole wave.
//   1. every distinct slow monomial S: w_S[p] = sum f_S(Delta_s) x[row0 +
//      Delta_s + p] (wave-uniform factors from a per-wave LDS table, offsets
//      in the scalar offset field of the buffer loads), mixed into the
//      channels V_F += C_t w_S of the fast monomials it pairs with (V_1 = y);
//   2. every channel F > 1: y[p] += sum h_F(p, Delta_f) V_F[p + Delta_f]
//      through a wave-private LDS row with zero margins;
//   3. the remaining terms without slow steps, one by one from x[row0 + p].
// An out-of-basis slow step has factor 0 and reads the first rows of the
// zero margin that the interleaved copy of x carries, which all such steps
// share; out-of-block fast neighbours carry factor 0.
// ------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ const T *fbtab_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *fbtab_of<double>(const NvOpDev &op) { return op.fb.tab64; }
template <> __device__ __forceinline__ const float *fbtab_of<float>(const NvOpDev &op) { return op.fb.tab32; }

// The four factors h(p, n, -s + 2i) of a slow slot at the wave's digit.
template <typename T> struct Fb4 { T v[4]; };

template <typename T> __device__ __forceinline__ const T *fbc_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *fbc_of<double>(const NvOpDev &op) { return op.fb.c64; }
template <> __device__ __forceinline__ const float *fbc_of<float>(const NvOpDev &op) { return op.fb.c32; }

// Element (s, s2) of a symmetric state matrix stored as its lower triangle.
__host__ __device__ constexpr int sym_at(int s, int s2) { return s >= s2 ? s * (s + 1) / 2 + s2 : s2 * (s2 + 1) / 2 + s; }
constexpr int sym_size(int ns) { return ns * (ns + 1) / 2; }

// V_c += C_c w for the channels C0 <= c < C1 that the slow monomial d feeds
// (channel 0 without the middle step when d.excl0).  C holds the lower
// triangles of the monomial's C1 - C0 matrices one after the other, so their
// addresses depend on no load, and the whole list of a cubic four-state
// operator stays within the 16 KB scalar cache in FP32 (with full matrices it
// did not, and every product waited on the L2).
template <int NS, typename TAcc, int C0, int C1, bool ODD>
__device__ __forceinline__ void fb_mix(const TAcc *__restrict__ C, const NvFbS &d, const TAcc (&w)[NS],
                                       const TAcc (&wf)[NS], TAcc (&V)[C1 - C0][NS]) {
    constexpr int Q = sym_size(NS);
#pragma unroll
    for (int c = C0; c < C1; ++c) {
        if (C1 > 1 && !(d.cmask >> c & 1)) continue;
        const bool ex = c == 0 && ODD && d.excl0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            TAcc a = V[c - C0][s];
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2) a += C[(c - C0) * Q + sym_at(s, s2)] * (ex ? w[s2] : wf[s2]);
            V[c - C0][s] = a;
        }
    }
}

// The slow monomials [t0, t1) of shape (K0, K1, K2), gathered and mixed into
// the channels V; vl is the lane's byte offset in its block, rb the byte
// offset of the block's first row in the padded buffer, fw/fwm the wave's
// factor rows and their masks of slots inside the basis.  The loop is
// software-pipelined: monomial t+1's rows are loaded while monomial t's are
// summed and mixed, each load reusing the registers of the row just summed,
// so a wave keeps one monomial's loads in flight through the mixing.
template <int NS, typename TIn, typename TAcc, int C0, int C1, int K0, int K1, int K2>
__device__ __forceinline__ void fb_slow(const NvOpDev &op, const XRes<NS, TIn> &xs, unsigned vl, unsigned rb,
                                        const TAcc *fw, const int *fwm, int t0, int t1,
                                        TAcc (&V)[C1 - C0][NS]) {
    using X = XRes<NS, TIn>;
    constexpr unsigned kEl = X::kEl;
    constexpr int J0 = K0 ? K0 : 1, J1 = K1 ? K1 : 1, J2 = K2 ? K2 : 1, J = J0 * J1 * J2;
    // all stepping slots odd: the middle step is Delta_s = 0
    constexpr bool odd = K0 > 0 && (K0 & 1) && (K1 == 0 || (K1 & 1)) && (K2 == 0 || (K2 & 1));
    if (t0 >= t1) return;
    // this phase's matrices: phase 1 starts at the monomials of phase 0, whose channels 0..3 it has
    constexpr int PH = C0 > 0 ? 0 : C1 == 4 ? 1 : 2;
    const TAcc *__restrict__ cm = fbc_of<TAcc>(op) + op.fb.cbase[PH];
    constexpr int CB = PH == 0 ? 4 : 0, NC = PH == 0 ? NV_FB_NCH - 4 : PH == 1 ? 4 : 1;
    const int tfirst = op.fb.sgrp[PH == 2 ? 2 : 0][0];
    // scalar byte offsets of monomial t's steps, in (i0, i1, i2) order; a step
    // outside the basis reads the zero margin at offset 0
    auto offsets = [&](int t, unsigned (&so)[J]) {
        const NvFbS &d = op.fb.S[t];
        // slot i of slow slot j is inside the basis when bit i of m_j is set
        int m0 = 1, m1 = 1, m2 = 1;
        if constexpr (K0 > 0) m0 = __builtin_amdgcn_readfirstlane(fwm[d.tab[0]]);
        if constexpr (K1 > 0) m1 = __builtin_amdgcn_readfirstlane(fwm[d.tab[1]]);
        if constexpr (K2 > 0) m2 = __builtin_amdgcn_readfirstlane(fwm[d.tab[2]]);
        const unsigned b0 = rb + (unsigned)d.base * kEl;
        const unsigned ib0 = (unsigned)d.inc[0] * kEl, ib1 = (unsigned)d.inc[1] * kEl,
                       ib2 = (unsigned)d.inc[2] * kEl;
#pragma unroll
        for (int i0 = 0; i0 < J0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < J1; ++i1)
#pragma unroll
                for (int i2 = 0; i2 < J2; ++i2) {
                    unsigned o = rb;
                    if constexpr (K0 > 0) o = b0 + (unsigned)i0 * ib0;
                    if constexpr (K1 > 0) o += (unsigned)i1 * ib1;
                    if constexpr (K2 > 0) o += (unsigned)i2 * ib2;
                    const bool in = ((m0 >> i0) & (K1 > 0 ? m1 >> i1 : 1) & (K2 > 0 ? m2 >> i2 : 1) & 1) != 0;
                    so[(i0 * J1 + i1) * J2 + i2] = in ? o : 0u;
                }
    };
    typename X::Row xr[J];
    {
        unsigned so[J];
        offsets(t0, so);
#pragma unroll
        for (int k = 0; k < J; ++k) {
            xr[k] = xs.load_so(vl, so[k]);
            // loads leave in step order, the order the loop consumes them
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (int t = t0; t < t1; ++t) {
        const NvFbS &d = op.fb.S[t];
        Fb4<TAcc> f0, f1, f2;
        if constexpr (K0 > 0) f0 = *reinterpret_cast<const Fb4<TAcc> *>(fw + d.tab[0] * 4);
        if constexpr (K1 > 0) f1 = *reinterpret_cast<const Fb4<TAcc> *>(fw + d.tab[1] * 4);
        if constexpr (K2 > 0) f2 = *reinterpret_cast<const Fb4<TAcc> *>(fw + d.tab[2] * 4);
        // w: every step but the middle one of an all-odd shape, wc: that one
        TAcc w[NS], wc[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) w[s] = wc[s] = (TAcc)0;
        // sums the rows in flight; with next, each row's registers then take
        // the next monomial's row
        auto sum_rows = [&](auto next, const unsigned (&sn)[J]) {
#pragma unroll
            for (int i0 = 0; i0 < J0; ++i0)
#pragma unroll
                for (int i1 = 0; i1 < J1; ++i1)
#pragma unroll
                    for (int i2 = 0; i2 < J2; ++i2) {
                        const int k = (i0 * J1 + i1) * J2 + i2;
                        TAcc h = (TAcc)1;
                        if constexpr (K0 > 0) h = f0.v[i0];
                        if constexpr (K1 > 0) h *= f1.v[i1];
                        if constexpr (K2 > 0) h *= f2.v[i2];
                        const bool mid = odd && 2 * i0 + 1 == K0 && (K1 == 0 || 2 * i1 + 1 == K1) &&
                                         (K2 == 0 || 2 * i2 + 1 == K2);
                        if (mid) X::template fma_row<TAcc>(xr[k], h, wc);
                        else X::template fma_row<TAcc>(xr[k], h, w);
                        if constexpr (decltype(next)::value) {
                            xr[k] = xs.load_so(vl, sn[k]);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
        };
        unsigned sn[J];
        if (t + 1 < t1) {
            offsets(t + 1, sn);
            sum_rows(std::true_type{}, sn);
        } else {
            sum_rows(std::false_type{}, sn);
        }
        if (d.nd > 0) {
            TAcc fd = fw[d.dtab[0] * 4];
            if (d.nd > 1) fd *= fw[d.dtab[1] * 4];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                w[s] *= fd;
                if constexpr (odd) wc[s] *= fd;
            }
        }
        // wc stays zero unless the shape has a middle step
        TAcc wf[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) wf[s] = odd ? w[s] + wc[s] : w[s];
        fb_mix<NS, TAcc, C0, C1, odd>(cm + ((size_t)(t - tfirst) * NC + C0 - CB) * sym_size(NS), d, w, wf, V);
    }
}

// y += sum_{steps [s0, s1)} h(p) src[p + stride]: the fast steps of one
// channel or term over the wave's LDS row vb, src published there first.
template <int NS, typename TAcc>
__device__ __forceinline__ void fb_fast(const NvOpDev &op, int s0, int s1, TAcc *vb, int lane, const uint8_t *dig,
                                        const TAcc *ftab, int tid, const TAcc (&src)[NS], TAcc (&y)[NS]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) vb[lane * NS + s] = src[s];
    __builtin_amdgcn_wave_barrier();
    const int nmax = op.nmax;
    for (int k = s0; k < s1; ++k) {
        const NvStep st = op.fb.steps[k];
        TAcc h = ftab[st.code[0] * nmax + dig[st.mode[0] * kBlock + tid]];
#pragma unroll
        for (int j = 1; j < NV_MAXF; ++j)
            if (j < st.nf) h *= ftab[st.code[j] * nmax + dig[st.mode[j] * kBlock + tid]];
        const TAcc *v = vb + (lane + st.stride) * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s) y[s] += h * v[s];
    }
    __builtin_amdgcn_wave_barrier();
}

// The off-diagonal part of the wave's block.
template <int NS, typename TIn, typename TAcc, bool SLAB>
__device__ __forceinline__ void fb_offdiag(const NvOpDev &op, const XRes<NS, TIn> &xs, unsigned vl, unsigned rb,
                                           int lane, const uint8_t *dig, const TAcc *fw, const int *fwm,
                                           const TAcc *ftab, int tid, TAcc *vb, TAcc (&y)[NS]) {
    // phase 0: channels 4.. (quadratic fast monomials), fed by the slow monomials of degree <= 1;
    // they go through LDS before the others start, which keeps six channels in registers
    const int *g0 = op.fb.sgrp[0];
    auto quadratic = [&](auto c0) {
        constexpr int C0 = decltype(c0)::value, C1 = C0 + 3;
        if (op.fb.nch <= C0) return;
        TAcc W[3][NS];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int s = 0; s < NS; ++s) W[c][s] = (TAcc)0;
        fb_slow<NS, TIn, TAcc, C0, C1, 2, 0, 0>(op, xs, vl, rb, fw, fwm, g0[0], g0[1], W);
        fb_slow<NS, TIn, TAcc, C0, C1, 0, 0, 0>(op, xs, vl, rb, fw, fwm, g0[7], g0[8], W);
#pragma unroll
        for (int c = C0; c < C1; ++c)
            if (c < op.fb.nch)
                fb_fast<NS, TAcc>(op, op.fb.chs[c], op.fb.chs[c + 1], vb, lane, dig, ftab, tid, W[c - C0], y);
    };
    quadratic(std::integral_constant<int, 4>{});
    quadratic(std::integral_constant<int, 7>{});
    // phase 1: channels 0..3, slow degree <= 2 (the monomials of phase 0 again: their few rows are
    // cheaper read twice than their channels held)
    TAcc V[4][NS];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int s = 0; s < NS; ++s) V[c][s] = (TAcc)0;
    const int *g1 = op.fb.sgrp[1];
    fb_slow<NS, TIn, TAcc, 0, 4, 2, 0, 0>(op, xs, vl, rb, fw, fwm, g0[0], g0[1], V);
    fb_slow<NS, TIn, TAcc, 0, 4, 0, 0, 0>(op, xs, vl, rb, fw, fwm, g0[7], g0[8], V);
    fb_slow<NS, TIn, TAcc, 0, 4, 2, 0, 0>(op, xs, vl, rb, fw, fwm, g1[0], g1[1], V);
    fb_slow<NS, TIn, TAcc, 0, 4, 3, 0, 0>(op, xs, vl, rb, fw, fwm, g1[1], g1[2], V);
    fb_slow<NS, TIn, TAcc, 0, 4, 2, 2, 0>(op, xs, vl, rb, fw, fwm, g1[3], g1[4], V);
    fb_slow<NS, TIn, TAcc, 0, 4, 0, 0, 0>(op, xs, vl, rb, fw, fwm, g1[7], g1[8], V);
#pragma unroll
    for (int c = 1; c < 4; ++c)
        if (c < op.fb.nch) fb_fast<NS, TAcc>(op, op.fb.chs[c], op.fb.chs[c + 1], vb, lane, dig, ftab, tid, V[c], y);
    // phase 2: channel 0 only, where most of the slow steps are unless the slab pass has the
    // monomials of degree three (without them four states in FP64 take 96 registers instead of 110)
    TAcc Y[1][NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) Y[0][s] = V[0][s];
    const int *g2 = op.fb.sgrp[2], *e2 = SLAB ? op.slab.s2end : g2 + 1;
    fb_slow<NS, TIn, TAcc, 0, 1, 2, 0, 0>(op, xs, vl, rb, fw, fwm, g2[0], e2[0], Y);
    fb_slow<NS, TIn, TAcc, 0, 1, 3, 0, 0>(op, xs, vl, rb, fw, fwm, g2[1], e2[1], Y);
    fb_slow<NS, TIn, TAcc, 0, 1, 2, 2, 0>(op, xs, vl, rb, fw, fwm, g2[3], e2[3], Y);
    fb_slow<NS, TIn, TAcc, 0, 1, 0, 0, 0>(op, xs, vl, rb, fw, fwm, g2[7], e2[7], Y);
    if constexpr (!SLAB) {
        fb_slow<NS, TIn, TAcc, 0, 1, 4, 0, 0>(op, xs, vl, rb, fw, fwm, g2[2], e2[2], Y);
        fb_slow<NS, TIn, TAcc, 0, 1, 3, 2, 0>(op, xs, vl, rb, fw, fwm, g2[4], e2[4], Y);
        fb_slow<NS, TIn, TAcc, 0, 1, 2, 3, 0>(op, xs, vl, rb, fw, fwm, g2[5], e2[5], Y);
        fb_slow<NS, TIn, TAcc, 0, 1, 2, 2, 2>(op, xs, vl, rb, fw, fwm, g2[6], e2[6], Y);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) y[s] += Y[0][s];
    if (op.fb.npure > 0) {
        TAcc xr[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) xr[s] = (TAcc)0;
        xs.template fma_so<TAcc>(vl, rb, (TAcc)1, xr);
        const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
        for (int k = 0; k < op.fb.npure; ++k) {
            const NvFbPure u = op.fb.pure[k];
            TAcc fd = (TAcc)1;
            if (u.nd > 0) fd = fw[u.dtab[0] * 4];
            if (u.nd > 1) fd *= fw[u.dtab[1] * 4];
            const TAcc *C = cm + (size_t)u.cm * NS * NS;
            TAcc v[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                TAcc a = (TAcc)0;
#pragma unroll
                for (int s2 = 0; s2 < NS; ++s2) a += C[s * NS + s2] * xr[s2];
                v[s] = fd * a;
            }
            fb_fast<NS, TAcc>(op, u.s0, u.s1, vb, lane, dig, ftab, tid, v, y);
        }
    }
}

// LDS of the fast-block kernels: factor table, the digits of one row per
// thread, four wave rows of (64 + 2 halo) lanes x NS values, four wave
// tables of ntab factor rows x 4 and four of ntab validity masks.
__host__ __device__ inline size_t fb_lds_layout(const NvOpDev &op, size_t el, size_t *dig_off, size_t *vb_off,
                                                size_t *fw_off) {
    const size_t a = ((size_t)op.ncodes * op.nmax * el + 15) & ~(size_t)15;
    const size_t b = a + (((size_t)op.M * kBlock + 15) & ~(size_t)15);
    const size_t c = b + ((4 * (size_t)(64 + 2 * op.fb.halo) * op.ns * el + 15) & ~(size_t)15);
    if (dig_off) *dig_off = a;
    if (vb_off) *vb_off = b;
    if (fw_off) *fw_off = c;
    // factor rows, then one validity mask per row
    return c + 4 * (size_t)op.fb.ntab * (4 * el + sizeof(int));
}

// Common prologue: factor table and digits in LDS, the wave's block, its LDS
// row and its factor rows.
template <typename TAcc> struct FbWave {
    const TAcc *ftab;
    uint8_t *dig;
    TAcc *vb;
    const TAcc *fw;
    const int *fwm;
    int lane, wave, blk, row0;
    bool inblk, live;
};
template <typename TAcc> __device__ __forceinline__ FbWave<TAcc> fb_prologue(const NvOpDev &op, int b) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    FbWave<TAcc> w;
    size_t dig_off, vb_off, fw_off;
    fb_lds_layout(op, sizeof(TAcc), &dig_off, &vb_off, &fw_off);
    TAcc *ft = reinterpret_cast<TAcc *>(lds_raw);
    const int nt = op.ncodes * op.nmax;
    const TAcc *g = ftab_of<TAcc>(op);
    for (int i = threadIdx.x; i < nt; i += blockDim.x) ft[i] = g[i];
    w.ftab = ft;
    w.dig = lds_raw + dig_off;
    const int tid = threadIdx.x;
    w.lane = tid & 63;
    w.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    w.blk = b * 4 + w.wave;
    w.inblk = w.blk < op.fb.nblk;
    {
        // block t of the sweep: its slow digits in the sweep's mode order
        int t = w.blk, row0 = 0;
        for (int j = 0; j < op.fb.nord; ++j) {
            const int nf = op.fb.ordnf[j];
            const int q = t / nf;
            row0 += (t - q * nf) * op.fb.ordshft[j];
            t = q;
        }
        w.row0 = row0;
    }
    w.live = w.inblk && w.lane < op.fb.P;
    if (w.live) digits_energy(op, w.row0 + w.lane, w.dig, tid);
    else for (int m = 0; m < op.M; ++m) w.dig[m * kBlock + tid] = 0;
    const int rowlen = (64 + 2 * op.fb.halo) * op.ns;
    TAcc *vrow = reinterpret_cast<TAcc *>(lds_raw + vb_off) + (size_t)w.wave * rowlen;
    for (int i = w.lane; i < rowlen; i += 64) vrow[i] = (TAcc)0;
    w.vb = vrow + (size_t)op.fb.halo * op.ns;
    __syncthreads();
    // the wave's factor rows at its slow digits (those of its first lane), and
    // their masks of slots inside the basis (factor nonzero)
    TAcc *fw = reinterpret_cast<TAcc *>(lds_raw + fw_off) + (size_t)w.wave * op.fb.ntab * 4;
    int *fwm = reinterpret_cast<int *>(lds_raw + fw_off + 4 * (size_t)op.fb.ntab * 4 * sizeof(TAcc)) +
               (size_t)w.wave * op.fb.ntab;
    const TAcc *tab = fbtab_of<TAcc>(op);
    for (int k = w.lane; k < op.fb.ntab; k += 64) {
        const int n = w.dig[op.fb.tabmode[k] * kBlock + w.wave * 64];
        int m = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const TAcc f = tab[((size_t)k * op.nmax + n) * 4 + i];
            fw[k * 4 + i] = f;
            m |= (f != (TAcc)0) << i;
        }
        fwm[k] = m;
    }
    __builtin_amdgcn_wave_barrier();
    w.fw = fw;
    w.fwm = fwm;
    return w;
}

// ------------------------------------------------------------------------
// Slab pass (tables in NvSlabDev): yt = the terms of degree three over the
// slow modes, interleaved as x.  The fast-block sweep reads every step of such
// a term through L1, 560 of its 680 row loads on the 88.5M-element cubic
// operator; here S_G is gathered once per row and its L neighbours come from
// LDS: 164 row loads and 200 LDS reads a row there.
// ------------------------------------------------------------------------
// y += the row of the slab pass.
template <int NS, typename TAcc>
__device__ __forceinline__ void add_slab(const void *yt, int r, TAcc (&y)[NS]) {
    constexpr int P = nv_lo_stride(NS);
    const IlRow<TAcc, P> v = reinterpret_cast<const IlRow<TAcc, P> *>(yt)[r];
#pragma unroll
    for (int s = 0; s < NS; ++s) y[s] += v.v[s];
}

template <typename T> __device__ __forceinline__ const T *slabtab_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *slabtab_of<double>(const NvOpDev &op) { return op.slab.tab64; }
template <> __device__ __forceinline__ const float *slabtab_of<float>(const NvOpDev &op) { return op.slab.tab32; }
template <typename T> __device__ __forceinline__ const T *slabltab_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *slabltab_of<double>(const NvOpDev &op) { return op.slab.ltab64; }
template <> __device__ __forceinline__ const float *slabltab_of<float>(const NvOpDev &op) { return op.slab.ltab32; }

template <int A, int B, int C> struct SlabShape { static constexpr int k0 = A, k1 = B, k2 = C; };

// u_k = S_G x at the thread's R rows for a monomial of shape (K0, K1, K2): up to eight rows in
// flight at a time.  Word t of tab names the factor row of slot t; a step outside the basis reads
// the zero margin.
template <int NS, typename TIn, typename TAcc, int R, int K0, int K1, int K2>
__device__ __forceinline__ void slab_gather(int base, const int32_t *inc, const int32_t *tab,
                                            const XRes<NS, TIn> &xs, const unsigned (&vl)[R], unsigned rb,
                                            const TAcc *fw, const int *fwm, TAcc (&u)[R][NS]) {
    using X = XRes<NS, TIn>;
    constexpr unsigned kEl = X::kEl;
    constexpr int J1 = K1 ? K1 : 1, J2 = K2 ? K2 : 1, JI = J1 * J2;
    // slots of the first factor per batch of loads
    constexpr int kIn = sizeof(TAcc) == 8 ? 6 : 8;
    constexpr int B0 = K0 * JI * R <= kIn ? K0 : K0 % 2 == 0 && 2 * JI * R <= kIn ? 2 : 1;
    const int m0 = __builtin_amdgcn_readfirstlane(fwm[tab[0]]);
    int m1 = 1, m2 = 1;
    if constexpr (K1 > 0) m1 = __builtin_amdgcn_readfirstlane(fwm[tab[1]]);
    if constexpr (K2 > 0) m2 = __builtin_amdgcn_readfirstlane(fwm[tab[2]]);
    const Fb4<TAcc> f0 = *reinterpret_cast<const Fb4<TAcc> *>(fw + tab[0] * 4);
    Fb4<TAcc> f1{}, f2{};
    if constexpr (K1 > 0) f1 = *reinterpret_cast<const Fb4<TAcc> *>(fw + tab[1] * 4);
    if constexpr (K2 > 0) f2 = *reinterpret_cast<const Fb4<TAcc> *>(fw + tab[2] * 4);
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int s = 0; s < NS; ++s) u[k][s] = (TAcc)0;
    const unsigned b0 = rb + (unsigned)base * kEl;
    const unsigned ib0 = (unsigned)inc[0] * kEl, ib1 = (unsigned)inc[1] * kEl, ib2 = (unsigned)inc[2] * kEl;
#pragma unroll
    for (int h0 = 0; h0 < K0; h0 += B0) {
        typename X::Row xr[B0 * JI][R];
#pragma unroll
        for (int i0 = 0; i0 < B0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < J1; ++i1)
#pragma unroll
                for (int i2 = 0; i2 < J2; ++i2) {
                    unsigned o = b0 + (unsigned)(h0 + i0) * ib0;
                    if constexpr (K1 > 0) o += (unsigned)i1 * ib1;
                    if constexpr (K2 > 0) o += (unsigned)i2 * ib2;
                    const bool in = ((m0 >> (h0 + i0)) & (K1 > 0 ? m1 >> i1 : 1) & (K2 > 0 ? m2 >> i2 : 1) & 1) != 0;
                    const unsigned so = in ? o : 0u;
#pragma unroll
                    for (int k = 0; k < R; ++k) xr[(i0 * J1 + i1) * J2 + i2][k] = xs.load_so(vl[k], so);
                }
#pragma unroll
        for (int i0 = 0; i0 < B0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < J1; ++i1)
#pragma unroll
                for (int i2 = 0; i2 < J2; ++i2) {
                    TAcc h = f0.v[h0 + i0];
                    if constexpr (K1 > 0) h *= f1.v[i1];
                    if constexpr (K2 > 0) h *= f2.v[i2];
#pragma unroll
                    for (int k = 0; k < R; ++k) X::template fma_row<TAcc>(xr[(i0 * J1 + i1) * J2 + i2][k], h, u[k]);
                }
    }
}

// LDS: two buffers of R rows per thread, the G factor rows and masks, the L factors.
__host__ __device__ inline size_t slab_lds(const NvOpDev &op, size_t el, int threads, int R, size_t *fw_off,
                                           size_t *lt_off) {
    const size_t a = 2 * (size_t)R * threads * op.ns * el;
    const size_t b = a + (size_t)op.slab.ntab * (4 * el + sizeof(int));
    const size_t c = (b + 15) & ~(size_t)15;
    if (fw_off) *fw_off = a;
    if (lt_off) *lt_off = c;
    return c + (size_t)op.slab.nl * op.nmax * 9 * el;
}

// A workgroup takes r rows of every L point for one set of G digits; a thread
// takes R of them, row and row + r/R: with R = 2 a point's rows are a whole
// 128-byte line (64-byte rows of lines cost the L2 twice their bytes), and the
// neighbours' offsets and factors serve both.
constexpr int slab_max_threads(int R, int bytes) { return R == 1 ? 1024 : bytes == 4 ? 640 : 320; }

template <int NS, typename TIn, typename TAcc, int NL, int R>
__global__ __launch_bounds__(slab_max_threads(R, sizeof(TAcc))) __attribute__((amdgpu_waves_per_eu(R == 2 && sizeof(TAcc) == 8 ? 4 : 1))) void hv_slab_kernel(NvOpDev op, const void *__restrict__ xin,
                                                       void *__restrict__ yt, int r) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const NvSlabDev &sl = op.slab;
    const int T = blockDim.x, tid = threadIdx.x;
    size_t fw_off, lt_off;
    slab_lds(op, sizeof(TAcc), T, R, &fw_off, &lt_off);
    TAcc *ub = reinterpret_cast<TAcc *>(lds_raw);
    TAcc *fw = reinterpret_cast<TAcc *>(lds_raw + fw_off);
    int *fwm = reinterpret_cast<int *>(fw + (size_t)sl.ntab * 4);
    TAcc *lt = reinterpret_cast<TAcc *>(lds_raw + lt_off);
    // Every XCD (workgroup b runs on XCD b % 8) takes an eighth of the G points, one chunk of rows
    // after the other: all of them work on the same few rows of every point at a time, which the
    // Infinity Cache holds.
    const int gper = (sl.gpts + 7) >> 3, at = blockIdx.x >> 3;
    const int chunk = at / gper, g = (int)(blockIdx.x & 7) * gper + (at - chunk * gper);
    if (g >= sl.gpts) return;
    {
        const TAcc *tab = slabtab_of<TAcc>(op), *ltab = slabltab_of<TAcc>(op);
        for (int k = tid; k < sl.ntab; k += T) {
            const int n = (g / sl.tabdiv[2 * k]) % sl.tabdiv[2 * k + 1];
            int m = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const TAcc f = tab[((size_t)k * op.nmax + n) * 4 + i];
                fw[k * 4 + i] = f;
                m |= (f != (TAcc)0) << i;
            }
            fwm[k] = m;
        }
        for (int k = tid; k < NL * op.nmax * 9; k += T) lt[k] = ltab[k];
    }
    __syncthreads();
    const int rt = r / R;
    const int pt = tid / rt, row = tid - pt * rt;
    const bool live = pt < sl.pts;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    constexpr int kNsp = nv_lo_stride(NS);
    constexpr unsigned kEl = XRes<NS, TIn>::kEl;
    const XRes<NS, TIn> xs(reinterpret_cast<const TX *>(xin) - (size_t)op.fb.pad * kNsp, op.D + 2 * op.fb.pad);
    const int inrow = pt * op.fb.P + chunk * r + row;   // row within the G point's block
    const int row0 = g * sl.pts * op.fb.P;
    unsigned vl[R];
#pragma unroll
    for (int k = 0; k < R; ++k) vl[k] = live ? (unsigned)(inrow + k * rt) * kEl : 0x80000000u;
    const unsigned rb = (unsigned)(row0 + op.fb.pad) * kEl;
    // per L mode the LDS distance of the neighbours at -2..2 (0 where the neighbour is outside the
    // basis, whose factor is 0, and for threads without a point) and the factors of q and q^2 (those
    // of q^3, needed once, stay in LDS)
    TAcc f1[NL][2], f2[NL][3];
    int o1[NL][2], o2[NL][3], dn[NL], st[NL];
    {
        int rest = live ? pt : 0, str = rt * NS;
#pragma unroll
        for (int q = NL - 1; q >= 0; --q) {
            const int nf = sl.lnf[q];
            const int d = rest / nf, n = rest - d * nf;
            rest = d;
            const TAcc *t = lt + ((size_t)q * op.nmax + n) * 9;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f1[q][i] = t[i];
                const int m = n - 1 + 2 * i;
                o1[q][i] = live && m >= 0 && m < nf ? (2 * i - 1) * str : 0;
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                f2[q][i] = t[2 + i];
                const int m = n - 2 + 2 * i;
                o2[q][i] = live && m >= 0 && m < nf ? (2 * i - 2) * str : 0;
            }
            dn[q] = n;
            st[q] = live ? str : 0;
            str *= nf;
        }
    }
    const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
    TAcc y[R][NS], u[R][NS], z[R][NS];
    // y starts from the leading pass's result
#pragma unroll
    for (int k = 0; k < R; ++k) {
        IlRow<TAcc, kNsp> v;
        if (sl.kl > 0 && live) v = reinterpret_cast<const IlRow<TAcc, kNsp> *>(yt)[row0 + inrow + k * rt];
#pragma unroll
        for (int s = 0; s < NS; ++s) y[k][s] = sl.kl > 0 && live ? v.v[s] : (TAcc)0;
    }
    // publishes u in the buffer the previous monomial did not use (whose readers have all passed the
    // barrier before this one's) and returns the thread's own first row there
    int flip = 0;
    auto publish = [&]() -> const TAcc * {
        TAcc *own = ub + (size_t)(flip * R * T + tid) * NS;
        flip ^= 1;
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int s = 0; s < NS; ++s) own[k * T * NS + s] = u[k][s];
        __syncthreads();
        return own;
    };
    auto clear = [&]() {
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int s = 0; s < NS; ++s) z[k][s] = (TAcc)0;
    };
    // z += h u at LDS distance o
    auto take = [&](const TAcc *p, int o, TAcc h) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const TAcc *v = p + k * T * NS + o;
#pragma unroll
            for (int s = 0; s < NS; ++s) z[k][s] += h * v[s];
        }
    };
    auto mix = [&](int c, const TAcc (&w)[R][NS]) {
        const TAcc *C = cm + (size_t)c * NS * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2)
#pragma unroll
                for (int k = 0; k < R; ++k) y[k][s] += C[s * NS + s2] * w[k][s2];
    };
    // S_G = 1: the cubic monomials of the L modes
    {
#pragma unroll
        for (int k = 0; k < R; ++k) {
#pragma unroll
            for (int s = 0; s < NS; ++s) u[k][s] = (TAcc)0;
            xs.template fma_so<TAcc>(vl[k], rb, (TAcc)1, u[k]);
        }
        const TAcc *p = publish();
#pragma unroll
        for (int a = 0; a < NL; ++a) {
            if (sl.c3[a] >= 0) {
                clear();
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int m = dn[a] - 3 + 2 * i;
                    take(p, m >= 0 && m < sl.lnf[a] ? (2 * i - 3) * st[a] : 0,
                         lt[((size_t)a * op.nmax + dn[a]) * 9 + 5 + i]);
                }
                mix(sl.c3[a], z);
            }
#pragma unroll
            for (int b = 0; b < NL; ++b) {
                if (b == a) continue;
                const int c = sl.c21[a * 2 + (b < a ? b : b - 1)];
                if (c < 0) continue;
                clear();
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) take(p, o2[a][i] + o1[b][j], f2[a][i] * f1[b][j]);
                mix(c, z);
            }
        }
        if constexpr (NL == 3) {
            if (sl.c111 >= 0) {
                clear();
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int k = 0; k < 2; ++k)
                            take(p, o1[0][i] + o1[1][j] + o1[2][k], f1[0][i] * f1[1][j] * f1[2][k]);
                mix(sl.c111, z);
            }
        }
    }
    // S_G of degree 1: the quadratic monomials of the L modes
    for (int t = sl.ggrp[0]; t < sl.ggrp[1]; ++t) {
        const NvSlabG &d = sl.G[t];
        slab_gather<NS, TIn, TAcc, R, 2, 0, 0>(d.base, d.inc, d.tab, xs, vl, rb, fw, fwm, u);
        const TAcc *p = publish();
#pragma unroll
        for (int a = 0; a < NL; ++a) {
            if (d.c2[a] >= 0) {
                clear();
#pragma unroll
                for (int i = 0; i < 3; ++i) take(p, o2[a][i], f2[a][i]);
                mix(d.c2[a], z);
            }
#pragma unroll
            for (int b = a + 1; b < NL; ++b) {
                if (d.c11[a + b - 1] < 0) continue;
                clear();
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) take(p, o1[a][i] + o1[b][j], f1[a][i] * f1[b][j]);
                mix(d.c11[a + b - 1], z);
            }
        }
    }
    // S_G of degree 2: the L modes themselves
    auto linear = [&](const NvSlabG &d) {
        const TAcc *p = publish();
#pragma unroll
        for (int a = 0; a < NL; ++a) {
            if (d.c1[a] < 0) continue;
            clear();
#pragma unroll
            for (int i = 0; i < 2; ++i) take(p, o1[a][i], f1[a][i]);
            mix(d.c1[a], z);
        }
    };
    for (int t = sl.ggrp[1]; t < sl.ggrp[2]; ++t) {
        const NvSlabG &d = sl.G[t];
        slab_gather<NS, TIn, TAcc, R, 3, 0, 0>(d.base, d.inc, d.tab, xs, vl, rb, fw, fwm, u);
        linear(d);
    }
    for (int t = sl.ggrp[2]; t < sl.ggrp[3]; ++t) {
        const NvSlabG &d = sl.G[t];
        slab_gather<NS, TIn, TAcc, R, 2, 2, 0>(d.base, d.inc, d.tab, xs, vl, rb, fw, fwm, u);
        linear(d);
    }
    // S_G of degree 3 feeds y
    auto direct = [&](auto shape, int q) {
        constexpr int K0 = decltype(shape)::k0, K1 = decltype(shape)::k1, K2 = decltype(shape)::k2;
        for (int t = sl.sgrp[q]; t < sl.sgrp[q + 1]; ++t) {
            const NvFbS &d = sl.S[t];
            slab_gather<NS, TIn, TAcc, R, K0, K1, K2>(d.base, d.inc, d.tab, xs, vl, rb, fw, fwm, u);
            mix(d.cm[0], u);
        }
    };
    direct(SlabShape<4, 0, 0>{}, 2);
    direct(SlabShape<3, 2, 0>{}, 4);
    direct(SlabShape<2, 3, 0>{}, 5);
    direct(SlabShape<2, 2, 2>{}, 6);
    if (live) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            IlRow<TAcc, kNsp> v;
#pragma unroll
            for (int s = 0; s < kNsp; ++s) v.v[s] = s < NS ? y[k][s] : (TAcc)0;
            reinterpret_cast<IlRow<TAcc, kNsp> *>(yt)[row0 + inrow + k * rt] = v;
        }
    }
}

// Leading pass: yt = the terms of degree three within modes 0..KL-1, over r rows
// of every point of them.  A workgroup holds the rows in LDS (147 KB at 2304
// points of four FP32 or two FP64 rows of four states) and each thread takes
// point after point; the memory sees every row once.
template <typename T> __device__ __forceinline__ const T *leadtab_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *leadtab_of<double>(const NvOpDev &op) { return op.slab.ktab64; }
template <> __device__ __forceinline__ const float *leadtab_of<float>(const NvOpDev &op) { return op.slab.ktab32; }

template <int NS, typename TIn, typename TAcc, int KL>
__global__ __launch_bounds__(1024) void hv_lead_kernel(NvOpDev op, const void *__restrict__ xin,
                                                       void *__restrict__ yt, int r) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const NvSlabDev &sl = op.slab;
    constexpr int kNsp = nv_lo_stride(NS);
    const int tid = threadIdx.x, items = sl.kpts * r;
    TAcc *ub = reinterpret_cast<TAcc *>(lds_raw);
    TAcc *kt = reinterpret_cast<TAcc *>(lds_raw + (((size_t)items * NS * sizeof(TAcc) + 15) & ~(size_t)15));
    const TAcc *ktab = leadtab_of<TAcc>(op);
    for (int k = tid; k < KL * op.nmax * 9; k += blockDim.x) kt[k] = ktab[k];
    // rows per point of the leading modes; the workgroup's chunk of them
    const int rest = op.D / sl.kpts, row0 = xcd_block(blockIdx.x, gridDim.x) * r;
    using Row = IlRow<TAcc, kNsp>;
    const Row *x = reinterpret_cast<const Row *>(xin);
#pragma unroll 4
    for (int i = tid; i < items; i += blockDim.x) {
        const int pt = i / r, row = i - pt * r;
        const Row v = x[pt * rest + row0 + row];
#pragma unroll
        for (int s = 0; s < NS; ++s) ub[i * NS + s] = v.v[s];
    }
    __syncthreads();
    const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
    for (int i = tid; i < items; i += blockDim.x) {
        const int pt = i / r, row = i - pt * r;
        TAcc f1[KL][2], f2[KL][3], f3[KL][4];
        int o1[KL], o2[KL], o3[KL];  // LDS distances of one, two and three functions up, and which exist
        unsigned up = 0, dn = 0;     // bit 4 k + j: the neighbour j functions up / down mode k is inside
        int q0 = pt, str = r * NS;
#pragma unroll
        for (int k = KL - 1; k >= 0; --k) {
            const int nf = sl.knf[k];
            const int d = q0 / nf, n = q0 - d * nf;
            q0 = d;
            const TAcc *t = kt + ((size_t)k * op.nmax + n) * 9;
#pragma unroll
            for (int j = 0; j < 2; ++j) f1[k][j] = t[j];
#pragma unroll
            for (int j = 0; j < 3; ++j) f2[k][j] = t[2 + j];
#pragma unroll
            for (int j = 0; j < 4; ++j) f3[k][j] = t[5 + j];
            o1[k] = str;
            o2[k] = 2 * str;
            o3[k] = 3 * str;
#pragma unroll
            for (int j = 1; j < 4; ++j) {
                up |= (unsigned)(n + j < nf) << (4 * k + j);
                dn |= (unsigned)(n - j >= 0) << (4 * k + j);
            }
            str *= nf;
        }
        // distance of the neighbour d functions along mode k, 0 outside the basis (factor 0)
        auto off = [&](int k, int d) {
            const int m = d == 1 || d == -1 ? o1[k] : d == 2 || d == -2 ? o2[k] : o3[k];
            if (d > 0) return (up >> (4 * k + d)) & 1 ? m : 0;
            if (d < 0) return (dn >> (4 * k - d)) & 1 ? -m : 0;
            return 0;
        };
        const TAcc *p = ub + i * NS;
        TAcc y[NS], z[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) y[s] = (TAcc)0;
        auto clear = [&]() {
#pragma unroll
            for (int s = 0; s < NS; ++s) z[s] = (TAcc)0;
        };
        auto take = [&](int o, TAcc h) {
#pragma unroll
            for (int s = 0; s < NS; ++s) z[s] += h * p[o + s];
        };
        auto mix = [&](int c) {
            const TAcc *C = cm + (size_t)c * NS * NS;
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int s2 = 0; s2 < NS; ++s2) y[s] += C[s * NS + s2] * z[s2];
        };
#pragma unroll
        for (int a = 0; a < KL; ++a) {
            if (sl.k3[a] >= 0) {
                clear();
#pragma unroll
                for (int j = 0; j < 4; ++j) take(off(a, 2 * j - 3), f3[a][j]);
                mix(sl.k3[a]);
            }
#pragma unroll
            for (int b = 0; b < KL; ++b) {
                if (b == a) continue;
                const int c = sl.k21[a * (NV_LEAD_NL - 1) + (b < a ? b : b - 1)];
                if (c < 0) continue;
                clear();
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int k = 0; k < 2; ++k) take(off(a, 2 * j - 2) + off(b, 2 * k - 1), f2[a][j] * f1[b][k]);
                mix(c);
            }
#pragma unroll
            for (int b = a + 1; b < KL; ++b)
#pragma unroll
                for (int d = b + 1; d < KL; ++d) {
                    const int c = sl.k111[a + b + d - 3];
                    if (c < 0) continue;
                    clear();
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int l = 0; l < 2; ++l)
                                take(off(a, 2 * j - 1) + off(b, 2 * k - 1) + off(d, 2 * l - 1),
                                     f1[a][j] * f1[b][k] * f1[d][l]);
                    mix(c);
                }
        }
        Row v;
#pragma unroll
        for (int s = 0; s < kNsp; ++s) v.v[s] = s < NS ? y[s] : (TAcc)0;
        reinterpret_cast<Row *>(yt)[pt * rest + row0 + row] = v;
    }
}

// Iteration H*v in the fast-block form: y = offdiag(H) q_i, alpha partials.
// Waves per SIMD the compiler must fit (register budget): 8 for FP32 (52
// VGPRs), in FP64 4 (110) with the degree-three slow monomials in the sweep
// and 5 (96) without them.  Four states, 22M rows, all steps in the sweep:
// FP32 10.7 ms at 6, 7 or 8 waves; FP64 23.6 ms at 3 or 4 waves and 28.0 ms
// at 5, where it spills.  Beside the slab pass the FP64 sweep waits on its
// loads (VALU 26% busy): 10.9 ms at 4 waves, 9.2 ms at 5.
// (Above four states the ten channels of NS values need more registers: the
// budget follows the state count.)
constexpr int fb_waves(int ns, int bytes, bool slab) {
    return ns <= 4 ? (bytes == 8 ? (slab ? 5 : 4) : 8) : (bytes == 8 ? 1 : 2);
}
template <int NS, typename TIn, typename TAcc, bool SLAB>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(fb_waves(NS, sizeof(TAcc), SLAB)))) void
hv_fb_iter_kernel(NvOpDev op, LzState st) {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const FbWave<TAcc> w = fb_prologue<TAcc>(op, b);
    const int tid = threadIdx.x;
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    const TX *x = std::is_same<TIn, F64I>::value ? reinterpret_cast<const TX *>(st.v64i)
                                                 : reinterpret_cast<const TX *>(st.vlo);
    constexpr int kNsp = nv_lo_stride(NS);
    constexpr unsigned kEl = XRes<NS, TIn>::kEl;
    const XRes<NS, TIn> xs(x - (size_t)op.fb.pad * kNsp, op.D + 2 * op.fb.pad);
    TAcc y[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) y[s] = (TAcc)0;
    // a lane past the block's P rows loads nothing (offset outside the buffer)
    const unsigned vl = w.live ? (unsigned)w.lane * kEl : 0x80000000u;
    const unsigned rb = (unsigned)(w.row0 + op.fb.pad) * kEl;
    if (w.inblk) fb_offdiag<NS, TIn, TAcc, SLAB>(op, xs, vl, rb, w.lane, w.dig, w.fw, w.fwm, w.ftab, tid, w.vb, y);
    double part = 0.0;
    // q_i, dg and y are touched once per launch (non-temporal on the largest vectors, so that
    // they do not displace the rows of x that neighbouring blocks gather from L2)
    auto epilogue = [&](auto nt) {
        constexpr bool NT = decltype(nt)::value;
        const int r = w.row0 + w.lane;
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = ld_once<NT>(&q[(size_t)s * op.D + r]);
#pragma unroll
        for (int s = 0; s < NS; ++s) dv[s] = ld_once<NT>(&op.dg[(size_t)s * op.D + r]) * v[s];
        if (op.offstate) diag_offstate<NS>(op, w.dig, tid, v, dv);
        TAcc *yo = reinterpret_cast<TAcc *>(st.y);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            st_once<NT>(y[s], &yo[(size_t)s * op.D + r]);
            part += v[s] * (dv[s] + (double)y[s]);
        }
    };
    if (SLAB && w.live) add_slab<NS, TAcc>(st.yt, w.row0 + w.lane, y);
    if (w.live) {
        if (op.stream_nt) epilogue(std::true_type{});
        else epilogue(std::false_type{});
    }
    const double bs = block_sum(part);
    if (tid == 0) st.partials[b] = bs;
}

// Standalone y = H x in the fast-block form: xin is the interleaved copy of x
// (FP32 or FP64, with its margins), x the FP64 vector for the diagonal part.
template <int NS, typename TIn, typename TAcc, bool SLAB>
__global__ __launch_bounds__(kBlock) void hv_fb_full_kernel(NvOpDev op, const void *__restrict__ xin,
                                                            const void *__restrict__ yt,
                                                            const double *__restrict__ x, double *__restrict__ yfull) {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const FbWave<TAcc> w = fb_prologue<TAcc>(op, b);
    const int tid = threadIdx.x;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    constexpr int kNsp = nv_lo_stride(NS);
    constexpr unsigned kEl = XRes<NS, TIn>::kEl;
    const XRes<NS, TIn> xs(reinterpret_cast<const TX *>(xin) - (size_t)op.fb.pad * kNsp, op.D + 2 * op.fb.pad);
    TAcc y[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) y[s] = (TAcc)0;
    const unsigned vl = w.live ? (unsigned)w.lane * kEl : 0x80000000u;
    const unsigned rb = (unsigned)(w.row0 + op.fb.pad) * kEl;
    if (w.inblk) fb_offdiag<NS, TIn, TAcc, SLAB>(op, xs, vl, rb, w.lane, w.dig, w.fw, w.fwm, w.ftab, tid, w.vb, y);
    if (w.live) {
        const int r = w.row0 + w.lane;
        if constexpr (SLAB) add_slab<NS, TAcc>(yt, r, y);
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = x[(size_t)s * op.D + r];
        diag_apply<NS>(op, r, w.dig, tid, v, dv);
#pragma unroll
        for (int s = 0; s < NS; ++s) yfull[(size_t)s * op.D + r] = dv[s] + (double)y[s];
    }
}

// ---- fast-block H*v launchers ----
static size_t hv_fb_lds(const NvOpDev &op, int prec) {
    return fb_lds_layout(op, prec == 0 ? 8 : 4, nullptr, nullptr, nullptr);
}

bool hv_fb_use(const NvOpDev &op, int prec) {
    if (!op.tshape || !op.fb.on || (prec != 0 && prec != 1)) return false;
    const int64_t el = (int64_t)nv_lo_stride(op.ns) * (prec == 0 ? 8 : 4);
    return (int64_t)op.D * el >= op.fb_min_bytes && shaped_ok(op, el) && hv_fb_lds(op, prec) <= 64 * 1024 &&
           ((int64_t)op.D + 2 * (int64_t)op.fb.pad) * el < ((int64_t)1 << 31);
}

int hv_fb_parts(const NvOpDev &op) { return (op.fb.nblk + 3) / 4; }

// ---- slab pass launcher ----
size_t hv_slab_bytes(const NvOpDev &op, int prec) {
    return op.slab.on ? (size_t)op.D * nv_lo_stride(op.ns) * (prec == 0 ? 8 : 4) : 0;
}

template <int NS, int NL>
static hipError_t slab_go(const NvOpDev &op, int prec, const void *xin, void *yt, hipStream_t s) {
    const int r = prec == 0 ? op.slab.r64 : op.slab.r32, R = prec == 0 ? op.slab.R64 : op.slab.R32;
    const unsigned T = (unsigned)(((size_t)op.slab.pts * (r / R) + 63) / 64 * 64);
    const unsigned grid = (unsigned)(8 * ((op.slab.gpts + 7) / 8) * (op.fb.P / r));
    const size_t lds = slab_lds(op, prec == 0 ? 8 : 4, (int)T, R, nullptr, nullptr);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(T), lds, s, op, xin, yt, r); };
    if (prec == 0) {
        if (R == 2) go(hv_slab_kernel<NS, F64I, double, NL, 2>);
        else go(hv_slab_kernel<NS, F64I, double, NL, 1>);
    } else {
        if (R == 2) go(hv_slab_kernel<NS, float, float, NL, 2>);
        else go(hv_slab_kernel<NS, float, float, NL, 1>);
    }
    return hipGetLastError();
}

static size_t lead_lds(const NvOpDev &op, int prec) {
    const size_t el = prec == 0 ? 8 : 4;
    const size_t rows = (size_t)op.slab.kpts * (prec == 0 ? op.slab.kr64 : op.slab.kr32);
    return ((rows * op.ns * el + 15) & ~(size_t)15) + (size_t)op.slab.kl * op.nmax * 9 * el;
}

// fn(kernel) for the leading pass of this operator and precision
template <int NS, typename Fn> static hipError_t with_lead(const NvOpDev &op, int prec, Fn fn) {
    switch (op.slab.kl) {
    case 2: return prec == 0 ? fn(hv_lead_kernel<NS, F64I, double, 2>) : fn(hv_lead_kernel<NS, float, float, 2>);
    case 3: return prec == 0 ? fn(hv_lead_kernel<NS, F64I, double, 3>) : fn(hv_lead_kernel<NS, float, float, 3>);
    case 4: return prec == 0 ? fn(hv_lead_kernel<NS, F64I, double, 4>) : fn(hv_lead_kernel<NS, float, float, 4>);
    default: return hipErrorInvalidValue;
    }
}

template <int NS> static hipError_t lead_prepare(const NvOpDev &op) {
    if constexpr (NS <= 4) {
        for (int prec = 0; prec < 2; ++prec) {
            hipError_t e = with_lead<NS>(op, prec, [&](auto kernel) {
                return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, NV_LEAD_LDS);
            });
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    } else {
        return hipErrorInvalidValue;
    }
}

hipError_t hv_slab_prepare(const NvOpDev &op) {
    if (!op.slab.on || op.slab.kl == 0) return hipSuccess;
    NV_DISPATCH_NS(lead_prepare, op)
}

template <int NS>
static hipError_t slab_ns(const NvOpDev &op, int prec, const void *xin, void *yt, hipStream_t s) {
    if constexpr (NS > 4) {
        return hipErrorInvalidValue;  // the tables are built for at most four states
    } else {
        if (!xin || !yt) return hipErrorInvalidValue;
        if (op.slab.kl > 0) {
            const int r = prec == 0 ? op.slab.kr64 : op.slab.kr32;
            const unsigned grid = (unsigned)(op.D / op.slab.kpts / r);
            hipError_t e = with_lead<NS>(op, prec, [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(grid), dim3(1024), lead_lds(op, prec), s, op, xin, yt, r);
                return hipGetLastError();
            });
            if (e != hipSuccess) return e;
        }
        switch (op.slab.nl) {
        case 1: return slab_go<NS, 1>(op, prec, xin, yt, s);
        case 2: return slab_go<NS, 2>(op, prec, xin, yt, s);
        case 3: return slab_go<NS, 3>(op, prec, xin, yt, s);
        default: return hipErrorInvalidValue;
        }
    }
}

// The forms that leave the degree-three slow monomials to the slab pass (which goes first), and those
// that do not: no slab pass, or no buffer for its result.
template <int NS, bool SLAB>
static hipError_t fb_iter_go(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    const size_t lds = hv_fb_lds(op, prec);
    const unsigned g = (unsigned)hv_fb_parts(op);
    if (prec == 0)
        hipLaunchKernelGGL((hv_fb_iter_kernel<NS, F64I, double, SLAB>), dim3(g), dim3(kBlock), lds, s, op, st);
    else
        hipLaunchKernelGGL((hv_fb_iter_kernel<NS, float, float, SLAB>), dim3(g), dim3(kBlock), lds, s, op, st);
    return hipGetLastError();
}

template <int NS>
static hipError_t fb_iter_ns(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    if constexpr (NS <= 4) {
        if (op.slab.on && st.yt) {
            hipError_t e = slab_ns<NS>(op, prec, prec == 0 ? (const void *)st.v64i : st.vlo, st.yt, s);
            return e != hipSuccess ? e : fb_iter_go<NS, true>(op, prec, st, s);
        }
    }
    return fb_iter_go<NS, false>(op, prec, st, s);
}

template <int NS, bool SLAB>
static hipError_t fb_full_go(const NvOpDev &op, int prec, const void *xin, void *yt, const double *x, double *y,
                             hipStream_t s) {
    const size_t lds = hv_fb_lds(op, prec);
    const unsigned g = (unsigned)hv_fb_parts(op);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(g), dim3(kBlock), lds, s, op, xin, yt, x, y); };
    if (prec == 0) go(hv_fb_full_kernel<NS, F64I, double, SLAB>);
    else go(hv_fb_full_kernel<NS, float, float, SLAB>);
    return hipGetLastError();
}

template <int NS>
static hipError_t fb_full_ns(const NvOpDev &op, int prec, const void *xin, void *yt, const double *x, double *y,
                             hipStream_t s) {
    if constexpr (NS <= 4) {
        if (op.slab.on && yt) {
            hipError_t e = slab_ns<NS>(op, prec, xin, yt, s);
            return e != hipSuccess ? e : fb_full_go<NS, true>(op, prec, xin, yt, x, y, s);
        }
    }
    return fb_full_go<NS, false>(op, prec, xin, yt, x, y, s);
}

hipError_t launch_hv_fb_full(const NvOpDev &op, int prec, const double *x, const void *xin, void *yt, double *y,
                             hipStream_t s) {
    NV_DISPATCH_NS(fb_full_ns, op, prec, xin, yt, x, y, s)
}

hipError_t launch_hv_fb_iter(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    NV_DISPATCH_NS(fb_iter_ns, op, prec, st, s)
}


}  // namespace nv
