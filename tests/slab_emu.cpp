// CPU emulation of the slab pass (hv_slab_kernel), for the CPU test suite.
//
// Builds the operator with the library's own host code (nv_operator.cpp) and
// runs the kernel's walk over the tables it gets, thread by thread of sampled
// workgroups: the gathers through 32-bit byte offsets and validity masks into
// the padded interleaved copy of x, the published rows, the L neighbours by
// their LDS distances.  Every read is bounds-checked against the buffers the
// kernel has, a neighbour at a nonzero factor must be the right point, and the
// result is compared with the step lists of the terms the pass takes.  The
// monomials the fast-block sweep keeps (phase 2 up to slab_s2end) must not
// hold any of those terms, and must hold every other one.
#include <cmath>
#include <set>
#include <string>
#include <vector>

#include "nv_operator.hpp"

using namespace nv;

namespace {
double xval(int64_t i) { return std::sin(0.37 * (double)i + 0.1) + 0.01 * (double)(i % 7); }
const int kShape[NV_FB_NSLOW][3] = {{2, 0, 0}, {3, 0, 0}, {4, 0, 0}, {2, 2, 0},
                                    {3, 2, 0}, {2, 3, 0}, {2, 2, 2}, {0, 0, 0}};
}  // namespace

// el: 4 or 8, the element size whose rows per workgroup and offsets are walked.
// Returns the largest difference relative to the largest reference value.
extern "C" double slab_emulate(const nv_problem *prob, int el, long maxgroups, int *on, int *bad, int *shape) {
    Operator op;
    std::string err;
    *on = 0;
    *bad = 0;
    if (!build_operator(*prob, op, err)) return -1.0;
    *on = op.slab;
    if (!op.slab) return 0.0;
    const int ns = (int)op.ns, nsp = nv_lo_stride(ns), P = op.fb_P, NL = op.slab_nl, gl = op.slab_gl, mf = op.fb_mf;
    const int r = el == 8 ? op.slab_r64 : op.slab_r32, R = el == 8 ? op.slab_R64 : op.slab_R32, rt = r / R;
    const int64_t D = op.D, pad = op.fb_pad;
    const unsigned kEl = (unsigned)(nsp * el);
    const int T1 = (op.slab_pts * rt + 63) / 64 * 64, T = T1 * R;  // threads; published rows, run-major
    shape[0] = NL;
    shape[1] = gl;
    shape[2] = r;
    shape[3] = T1;
    shape[4] = (int)op.slab_G.size();
    shape[5] = (int)op.slab_S.size();
    if (r % R != 0 || P % r != 0 || T1 > 1024) ++*bad;
    if (2 * (int64_t)T * ns * el + (int64_t)(op.slab_tabdiv.size() / 2) * (4 * el + 4) + 16 +
            (int64_t)NL * op.nmax * 9 * el > 64 * 1024)
        ++*bad;
    const int64_t bufrows = D + 2 * pad;
    std::vector<double> xb((size_t)bufrows * nsp, 0.0);
    for (int64_t q = 0; q < D; ++q)
        for (int s = 0; s < ns; ++s) xb[(size_t)(q + pad) * nsp + s] = xval(s * D + q);
    // the row a load of voffset vl and scalar offset so reads
    auto row_at = [&](unsigned vl, unsigned so) -> int64_t {
        const uint64_t o = (uint64_t)vl + so;
        if (o % kEl != 0 || o / kEl >= (uint64_t)bufrows) {
            ++*bad;
            return 0;
        }
        return (int64_t)(o / kEl);
    };
    std::set<int> mine;
    for (size_t ti = 0; ti < op.terms.size(); ++ti) {
        const Term &t = op.terms[ti];
        int deg = 0, slow = 1;
        for (int j = 0; j < t.cnt; ++j) { deg += t.pow[j]; slow = slow && t.mode[j] < mf; }
        if (op.term_dev[ti] >= 0 && deg == 3 && slow) mine.insert(op.term_dev[ti]);
    }
    // each taken term exactly once here and nowhere in the sweep's remaining lists
    std::multiset<int> here, kept;
    for (int k = 0; k < NV_SLAB_NL; ++k) if (op.slab_c3[k] >= 0) here.insert(op.slab_c3[k]);
    for (int k = 0; k < 6; ++k) if (op.slab_c21[k] >= 0) here.insert(op.slab_c21[k]);
    if (op.slab_c111 >= 0) here.insert(op.slab_c111);
    for (auto &g : op.slab_G)
        for (int k = 0; k < 3; ++k) {
            if (g.c1[k] >= 0) here.insert(g.c1[k]);
            if (g.c2[k] >= 0) here.insert(g.c2[k]);
            if (g.c11[k] >= 0) here.insert(g.c11[k]);
        }
    for (auto &S : op.slab_S) here.insert(S.cm[0]);
    std::set<int> lead;
    for (int v : op.slab_k3) if (v >= 0) { here.insert(v); lead.insert(v); }
    for (int v : op.slab_k21) if (v >= 0) { here.insert(v); lead.insert(v); }
    for (int v : op.slab_k111) if (v >= 0) { here.insert(v); lead.insert(v); }
    const int KL = op.slab_kl, kr = el == 8 ? op.slab_kr64 : op.slab_kr32, kpts = op.slab_kpts;
    if (KL > 0) {
        if (((int64_t)kpts * kr * ns * el + 15) / 16 * 16 + (int64_t)KL * op.nmax * 9 * el > NV_LEAD_LDS || KL < 2 ||
            KL > gl || (D / kpts) % kr != 0)
            ++*bad;
    }
    // the leading pass at one row: LDS neighbours of its point, checked against the vector's rows
    auto lead_row = [&](int64_t row, double *y) {
        const int64_t rest = D / kpts;
        const int pt = (int)(row / rest);
        const int64_t q = row % rest, chunk = q / kr, rr = q % kr;
        int n[NV_LEAD_NL], str[NV_LEAD_NL], p = pt, st = kr;
        for (int k = KL - 1; k >= 0; --k) {
            n[k] = p % (int)op.nfunc[k];
            p /= (int)op.nfunc[k];
            str[k] = st;
            st *= (int)op.nfunc[k];
        }
        auto off = [&](int k, int d) { return n[k] + d >= 0 && n[k] + d < op.nfunc[k] ? d * str[k] : 0; };
        auto f = [&](int k, int w, int i) { return op.slab_ktab[((size_t)k * op.nmax + n[k]) * 9 + (w == 1 ? 0 : w == 2 ? 2 : 5) + i]; };
        double z[4];
        auto take = [&](int o, double h) {
            const int64_t a = (int64_t)pt * kr + rr + o;
            if (a < 0 || a >= (int64_t)kpts * kr) { ++*bad; return; }
            const int64_t src = (a / kr) * rest + chunk * kr + a % kr;
            for (int s = 0; s < ns; ++s) z[s] += h * xval(s * D + src);
        };
        auto mixin = [&](int c) {
            for (int s = 0; s < ns; ++s)
                for (int s2 = 0; s2 < ns; ++s2) y[s] += op.cmat[(size_t)c * ns * ns + s * ns + s2] * z[s2];
        };
        auto clear = [&]() { for (double &v : z) v = 0.0; };
        for (int a = 0; a < KL; ++a) {
            if (op.slab_k3[a] >= 0) {
                clear();
                for (int j = 0; j < 4; ++j) take(off(a, 2 * j - 3), f(a, 3, j));
                mixin(op.slab_k3[a]);
            }
            for (int b = 0; b < KL; ++b) {
                if (b == a) continue;
                const int c = op.slab_k21[a * (NV_LEAD_NL - 1) + (b < a ? b : b - 1)];
                if (c < 0) continue;
                clear();
                for (int j = 0; j < 3; ++j)
                    for (int k = 0; k < 2; ++k) take(off(a, 2 * j - 2) + off(b, 2 * k - 1), f(a, 2, j) * f(b, 1, k));
                mixin(c);
            }
            for (int b = a + 1; b < KL; ++b)
                for (int d = b + 1; d < KL; ++d) {
                    const int c = op.slab_k111[a + b + d - 3];
                    if (c < 0) continue;
                    clear();
                    for (int j = 0; j < 2; ++j)
                        for (int k = 0; k < 2; ++k)
                            for (int l = 0; l < 2; ++l)
                                take(off(a, 2 * j - 1) + off(b, 2 * k - 1) + off(d, 2 * l - 1),
                                     f(a, 1, j) * f(b, 1, k) * f(d, 1, l));
                    mixin(c);
                }
        }
    };
    if (here.size() != mine.size()) ++*bad;
    for (int c : mine) if (here.count(c) != 1) ++*bad;
    for (int ph = 0; ph < 3; ++ph)
        for (int q = 0; q < NV_FB_NSLOW; ++q) {
            const int e = ph == 2 ? op.slab_s2end[q] : op.fb_sgrp[ph][q + 1];
            for (int t = op.fb_sgrp[ph][q]; t < op.fb_sgrp[ph][q + 1]; ++t)
                for (int c = 0; c < NV_FB_NCH; ++c)
                    if (op.fb_S[t].cm[c] >= 0) {
                        if (t < e) kept.insert(op.fb_S[t].cm[c]);
                        else if (!mine.count(op.fb_S[t].cm[c])) ++*bad;
                    }
        }
    for (auto &u : op.fb_pure) kept.insert(u.cm);
    for (int c : mine) if (kept.count(c)) ++*bad;
    if (kept.size() + mine.size() != op.dev_terms.size()) ++*bad;

    double maxdiff = 0.0, maxref = 0.0;
    int64_t done = 0;
    const int nch = P / r, gper = (op.slab_gpts + 7) / 8;
    const int64_t groups = (int64_t)8 * gper * nch;
    std::vector<char> seen((size_t)op.slab_gpts * nch, 0);
    const int64_t step = groups > maxgroups ? groups / maxgroups : 1;
    for (int64_t w0 = 0; w0 < groups; ++w0) {
        const int chunk = (int)((w0 >> 3) / gper), g = (int)(w0 & 7) * gper + (int)((w0 >> 3) % gper);
        if (g >= op.slab_gpts) continue;
        if (chunk >= nch || seen[(int64_t)chunk * op.slab_gpts + g]) { ++*bad; continue; }
        seen[(int64_t)chunk * op.slab_gpts + g] = 1;
        ++done;
        if (w0 % step != 0) continue;
        const int ntab = (int)op.slab_tabdiv.size() / 2;
        std::vector<double> fw((size_t)ntab * 4);
        std::vector<int> fwm(ntab, 0);
        for (int k = 0; k < ntab; ++k) {
            const int n = (g / op.slab_tabdiv[2 * k]) % op.slab_tabdiv[2 * k + 1];
            for (int i = 0; i < 4; ++i) {
                fw[k * 4 + i] = op.slab_tab[((size_t)k * op.nmax + n) * 4 + i];
                fwm[k] |= (fw[k * 4 + i] != 0.0) << i;
            }
        }
        const int64_t row0 = (int64_t)g * op.slab_pts * P;
        const unsigned rb = (unsigned)((row0 + pad) * kEl);
        std::vector<unsigned> vl(T, 0u);
        std::vector<int64_t> myrow(T, -1);
        struct Nb { double f[9]; int o[9]; };
        std::vector<Nb> nb((size_t)T * NL);
        for (int t = 0; t < T; ++t) {
            const int tid = t % T1, run = t / T1;
            const int pt = tid / rt, row = tid % rt;
            const bool live = pt < op.slab_pts;
            const int inrow = pt * P + chunk * r + row + run * rt;
            if (live) {
                vl[t] = (unsigned)inrow * kEl;
                myrow[t] = row0 + inrow;
            }
            int rest = live ? pt : 0, str = rt;
            for (int q = NL - 1; q >= 0; --q) {
                const int nf = (int)op.nfunc[gl + q], n = rest % nf;
                rest /= nf;
                Nb &b = nb[(size_t)t * NL + q];
                int at = 0;
                for (int p = 1; p <= 3; ++p)
                    for (int i = 0; i <= p; ++i, ++at) {
                        b.f[at] = op.slab_ltab[((size_t)q * op.nmax + n) * 9 + at];
                        const int m = n - p + 2 * i;
                        b.o[at] = live && m >= 0 && m < nf ? (2 * i - p) * str : 0;
                        // a nonzero factor belongs to a point of the basis, and reaches it
                        if (live && b.f[at] != 0.0) {
                            const int o = tid + b.o[at];
                            if (m < 0 || m >= nf || o < 0 || o >= T1 ||
                                myrow[t] + (int64_t)(2 * i - p) * op.shft[gl + q] !=
                                    row0 + (int64_t)(o / rt) * P + chunk * r + o % rt + run * rt)
                                ++*bad;
                        }
                    }
                str *= nf;
            }
        }
        std::vector<double> y((size_t)T * ns, 0.0), u((size_t)T * ns, 0.0);
        auto mix = [&](int t, int c, const double *z) {
            for (int s = 0; s < ns; ++s)
                for (int s2 = 0; s2 < ns; ++s2) y[(size_t)t * ns + s] += op.cmat[(size_t)c * ns * ns + s * ns + s2] * z[s2];
        };
        auto add = [&](int t, int o, double h, double *z) {
            const int a = t + o;
            if (a < 0 || a >= T || a / T1 != t / T1) { ++*bad; return; }
            for (int s = 0; s < ns; ++s) z[s] += h * u[(size_t)a * ns + s];
        };
        // u = (steps of d) x for every thread; K slots
        auto gather = [&](int64_t base, const int32_t *inc, const int32_t *tab, const int *K, double *out) {
            for (int t = 0; t < T; ++t) {
                double z[4] = {0, 0, 0, 0};
                const int J1 = K[1] ? K[1] : 1, J2 = K[2] ? K[2] : 1;
                for (int i0 = 0; i0 < K[0]; ++i0)
                    for (int i1 = 0; i1 < J1; ++i1)
                        for (int i2 = 0; i2 < J2; ++i2) {
                            if (myrow[t] < 0) continue;
                            unsigned o = rb + (unsigned)base * kEl + (unsigned)i0 * ((unsigned)inc[0] * kEl);
                            double h = fw[tab[0] * 4 + i0];
                            int in = fwm[tab[0]] >> i0;
                            if (K[1]) { o += (unsigned)i1 * ((unsigned)inc[1] * kEl); h *= fw[tab[1] * 4 + i1]; in &= fwm[tab[1]] >> i1; }
                            if (K[2]) { o += (unsigned)i2 * ((unsigned)inc[2] * kEl); h *= fw[tab[2] * 4 + i2]; in &= fwm[tab[2]] >> i2; }
                            const int64_t q = row_at(vl[t], (in & 1) ? o : 0u);
                            if (!(in & 1) && q >= pad) ++*bad;  // the zero margin
                            for (int s = 0; s < ns; ++s) z[s] += h * xb[(size_t)q * nsp + s];
                        }
                for (int s = 0; s < ns; ++s) out[(size_t)t * ns + s] = z[s];
            }
        };
        for (int t = 0; t < T; ++t)
            if (myrow[t] >= 0)
                for (int s = 0; s < ns; ++s) u[(size_t)t * ns + s] = xb[(size_t)row_at(vl[t], rb) * nsp + s];
        for (int t = 0; t < T; ++t) {
            const Nb *b = &nb[(size_t)t * NL];
            for (int a = 0; a < NL; ++a) {
                if (op.slab_c3[a] >= 0) {
                    double z[4] = {0, 0, 0, 0};
                    for (int i = 0; i < 4; ++i) add(t, b[a].o[5 + i], b[a].f[5 + i], z);
                    mix(t, op.slab_c3[a], z);
                }
                for (int l = 0; l < NL; ++l) {
                    if (l == a) continue;
                    const int c = op.slab_c21[a * 2 + (l < a ? l : l - 1)];
                    if (c < 0) continue;
                    double z[4] = {0, 0, 0, 0};
                    for (int i = 0; i < 3; ++i)
                        for (int j = 0; j < 2; ++j) add(t, b[a].o[2 + i] + b[l].o[j], b[a].f[2 + i] * b[l].f[j], z);
                    mix(t, c, z);
                }
            }
            if (NL == 3 && op.slab_c111 >= 0) {
                double z[4] = {0, 0, 0, 0};
                for (int i = 0; i < 2; ++i)
                    for (int j = 0; j < 2; ++j)
                        for (int k = 0; k < 2; ++k)
                            add(t, b[0].o[i] + b[1].o[j] + b[2].o[k], b[0].f[i] * b[1].f[j] * b[2].f[k], z);
                mix(t, op.slab_c111, z);
            }
        }
        static const int kG[3][3] = {{2, 0, 0}, {3, 0, 0}, {2, 2, 0}};
        for (int z0 = 0; z0 < 3; ++z0)
            for (int e = op.slab_ggrp[z0]; e < op.slab_ggrp[z0 + 1]; ++e) {
                const NvSlabG &d = op.slab_G[e];
                gather(d.base, d.inc, d.tab, kG[z0], u.data());
                for (int t = 0; t < T; ++t) {
                    const Nb *b = &nb[(size_t)t * NL];
                    for (int a = 0; a < NL; ++a) {
                        double z[4] = {0, 0, 0, 0};
                        if (z0 == 0 && d.c2[a] >= 0) {
                            for (int i = 0; i < 3; ++i) add(t, b[a].o[2 + i], b[a].f[2 + i], z);
                            mix(t, d.c2[a], z);
                        }
                        if (z0 > 0 && d.c1[a] >= 0) {
                            for (int i = 0; i < 2; ++i) add(t, b[a].o[i], b[a].f[i], z);
                            mix(t, d.c1[a], z);
                        }
                        for (int l = a + 1; l < NL; ++l) {
                            if (z0 != 0 || d.c11[a + l - 1] < 0) continue;
                            double v[4] = {0, 0, 0, 0};
                            for (int i = 0; i < 2; ++i)
                                for (int j = 0; j < 2; ++j) add(t, b[a].o[i] + b[l].o[j], b[a].f[i] * b[l].f[j], v);
                            mix(t, d.c11[a + l - 1], v);
                        }
                    }
                }
            }
        for (int q = 0; q < NV_FB_NSLOW; ++q)
            for (int e = op.slab_sgrp[q]; e < op.slab_sgrp[q + 1]; ++e) {
                if (q != 2 && q < 4) ++*bad;  // only the shapes of degree three
                gather(op.slab_S[e].base, op.slab_S[e].inc, op.slab_S[e].tab, kShape[q], u.data());
                for (int t = 0; t < T; ++t) mix(t, op.slab_S[e].cm[0], &u[(size_t)t * ns]);
            }
        // the step lists of the same terms
        for (int t = 0; t < T; ++t) {
            if (myrow[t] < 0) continue;
            const int64_t row = myrow[t];
            if (KL > 0) lead_row(row, &y[(size_t)t * ns]);
            double ref[4] = {0, 0, 0, 0};
            for (int c : mine) {
                double z[4] = {0, 0, 0, 0};
                for (int k = 0; k < op.dev_terms[c].nsteps; ++k) {
                    const NvStep &st = op.dev_steps[op.dev_terms[c].first + k];
                    double h = 1.0;
                    for (int j = 0; j < st.nf; ++j)
                        h *= op.ftab[(size_t)st.code[j] * op.nmax + (row / op.shft[st.mode[j]]) % op.nfunc[st.mode[j]]];
                    if (h == 0.0) continue;
                    for (int s = 0; s < ns; ++s) z[s] += h * xval(s * D + row + st.stride);
                }
                for (int s = 0; s < ns; ++s)
                    for (int s2 = 0; s2 < ns; ++s2) ref[s] += op.cmat[(size_t)c * ns * ns + s * ns + s2] * z[s2];
            }
            for (int s = 0; s < ns; ++s) {
                maxref = std::fmax(maxref, std::fabs(ref[s]));
                maxdiff = std::fmax(maxdiff, std::fabs(ref[s] - y[(size_t)t * ns + s]));
            }
        }
    }
    if (done != (int64_t)op.slab_gpts * nch) ++*bad;  // every chunk of every point, once
    return maxref > 0.0 ? maxdiff / maxref : 0.0;
}
