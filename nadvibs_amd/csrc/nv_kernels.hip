// HIP kernels of the Lanczos path for gfx950 (64-wide wavefronts).
//
//  * hv_*          matrix-free H*v over the state-major tensor x[s][n_1..n_M]
//                  (last mode fastest): one thread per vibrational index r
//                  computes all states; the mode digits of r and the factor
//                  table sit in LDS; coupling matrices are read as uniform
//                  (scalar) loads.
//  * normalize / lanczos_step   the three-term recurrence in FP64 with the
//                  dots reduced to per-block partials and summed by a
//                  one-block finish kernel (fixed summation order:
//                  reproducible run to run).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "nv_hvcore.hpp"

namespace nv {

// dg[s][r] = E(r) + D_ss(r): harmonic energy, constant term and the Delta=0
// part of the all-even monomials of the diagonal blocks.
template <int NS>
__global__ __launch_bounds__(kBlock) void diag_precompute_kernel(NvOpDev op, double *dg) {
    __shared__ uint8_t dig[NV_MAXM * kBlock];
    const int tid = threadIdx.x;
    const int r = blockIdx.x * kBlock + tid;
    if (r >= op.D) return;
    const double E = digits_energy(op, r, dig, tid);
    double d[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) d[s] = E + op.dconst[s * NS + s];
    for (int t = 0; t < op.ndterms; ++t) {
        const NvDiagTerm dt = op.dterms[t];
        double h = 1.0;
#pragma unroll
        for (int j = 0; j < NV_MAXF; ++j)
            if (j < dt.nf) h *= op.ftab64[dt.code[j] * op.nmax + dig[dt.mode[j] * kBlock + tid]];
        const double *C = op.dcmat + (size_t)t * NS * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s) d[s] += h * C[s * NS + s];
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) dg[(size_t)s * op.D + r] = d[s];
}

// ------------------------------------------------------------------------
// H*v: off-diagonal (in vibrational space) terms, Source/top.f90:758-808.
// acc[s] = sum_t sum_s' C_t[s][s'] sum_{steps} prod_j f_j(n) x[s'][r+stride]
// ------------------------------------------------------------------------
template <int NS, typename TIn, typename TAcc>
__device__ __forceinline__ void offdiag_accumulate(const NvOpDev &op, const TIn *__restrict__ x, int r,
                                                   const uint8_t *dig, const TAcc *ftab, int tid,
                                                   TAcc (&acc)[NS]) {
    const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = (TAcc)0;
    for (int t = 0; t < op.nterms; ++t) {
        const NvTerm tm = op.terms[t];
        TAcc w[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) w[s] = (TAcc)0;
        for (int q = 0; q < tm.nsteps; ++q) {
            const NvStep st = op.steps[tm.first + q];
            TAcc h = ftab[st.code[0] * op.nmax + dig[st.mode[0] * kBlock + tid]];
#pragma unroll
            for (int j = 1; j < NV_MAXF; ++j)
                if (j < st.nf) h *= ftab[st.code[j] * op.nmax + dig[st.mode[j] * kBlock + tid]];
            if (h != (TAcc)0) {
                const int idx = r + st.stride;
                if constexpr (std::is_same<TIn, double>::value) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) w[s] += h * load_acc<TIn, TAcc>(x + (size_t)s * op.D + idx);
                } else {
                    // interleaved low-precision copy: the states of a row are adjacent
                    const TIn *xr = x + (size_t)idx * nv_lo_stride(NS);
#pragma unroll
                    for (int s = 0; s < NS; ++s) w[s] += h * load_acc<TIn, TAcc>(xr + s);
                }
            }
        }
        const TAcc *C = cm + (size_t)t * NS * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            TAcc a = acc[s];
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2) a += C[s * NS + s2] * w[s2];
            acc[s] = a;
        }
    }
}

// The same for two rows of one thread (r0 and r1, digits at dig0 and dig1): the step descriptors are read once for both, and the two rows'
// table and vector loads are independent, so they overlap.  A row that is
// not live (past the end) has zero digits and is skipped.
template <int NS, typename TIn, typename TAcc>
__device__ __forceinline__ void offdiag_accumulate2(const NvOpDev &op, const TIn *__restrict__ x, int r0, int r1,
                                                    bool l0, bool l1, const uint8_t *dig0, const uint8_t *dig1,
                                                    const TAcc *ftab, int tid, TAcc (&acc0)[NS], TAcc (&acc1)[NS]) {
    const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        acc0[s] = (TAcc)0;
        acc1[s] = (TAcc)0;
    }
    for (int t = 0; t < op.nterms; ++t) {
        const NvTerm tm = op.terms[t];
        TAcc w0[NS], w1[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            w0[s] = (TAcc)0;
            w1[s] = (TAcc)0;
        }
        for (int q = 0; q < tm.nsteps; ++q) {
            const NvStep st = op.steps[tm.first + q];
            TAcc h0 = ftab[st.code[0] * op.nmax + dig0[st.mode[0] * kBlock + tid]];
            TAcc h1 = ftab[st.code[0] * op.nmax + dig1[st.mode[0] * kBlock + tid]];
#pragma unroll
            for (int j = 1; j < NV_MAXF; ++j)
                if (j < st.nf) {
                    h0 *= ftab[st.code[j] * op.nmax + dig0[st.mode[j] * kBlock + tid]];
                    h1 *= ftab[st.code[j] * op.nmax + dig1[st.mode[j] * kBlock + tid]];
                }
            if (l0 && h0 != (TAcc)0) {
                const int idx = r0 + st.stride;
                if constexpr (std::is_same<TIn, double>::value) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) w0[s] += h0 * load_acc<TIn, TAcc>(x + (size_t)s * op.D + idx);
                } else {
                    const TIn *xr = x + (size_t)idx * nv_lo_stride(NS);
#pragma unroll
                    for (int s = 0; s < NS; ++s) w0[s] += h0 * load_acc<TIn, TAcc>(xr + s);
                }
            }
            if (l1 && h1 != (TAcc)0) {
                const int idx = r1 + st.stride;
                if constexpr (std::is_same<TIn, double>::value) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) w1[s] += h1 * load_acc<TIn, TAcc>(x + (size_t)s * op.D + idx);
                } else {
                    const TIn *xr = x + (size_t)idx * nv_lo_stride(NS);
#pragma unroll
                    for (int s = 0; s < NS; ++s) w1[s] += h1 * load_acc<TIn, TAcc>(xr + s);
                }
            }
        }
        const TAcc *C = cm + (size_t)t * NS * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            TAcc a0 = acc0[s], a1 = acc1[s];
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2) {
                a0 += C[s * NS + s2] * w0[s2];
                a1 += C[s * NS + s2] * w1[s2];
            }
            acc0[s] = a0;
            acc1[s] = a1;
        }
    }
}

// ------------------------------------------------------------------------
// Shaped off-diagonal H*v.  The same sum as offdiag_accumulate, with the
// steps of a term generated from its shape (NvTermShape): the digits and the
// per-mode factors f_j(Delta_j) are read once per term, the step loop is
// unrolled, a step's factor is f_0 * f_1 * f_2 (the step kernel's product
// order) and its offset a scalar.  Neighbour rows come through buffer
// resources sized to the vector: an offset outside it (a step that leaves the
// basis, whose factor is 0; a negative offset wraps past 2^31) loads 0, so
// there is no branch per step.
// ------------------------------------------------------------------------
// The terms of shape group g; R rows per thread (digits of row q at
// dig + q * M * kBlock), row q's byte offset in the vector vo[q].  SKIP
// points the load of a step whose factor is 0 outside the buffer (it then
// moves no memory), where a plain out-of-basis offset may land on another row.
// With S > 1 (a power of two) only every S-th term is taken, those of index
// part modulo S.
template <int NS, typename TIn, typename TAcc, int R, bool SKIP, int S, int K0, int K1, int K2>
__device__ __forceinline__ void shaped_group(const NvOpDev &op, const XRes<NS, TIn> &xs, const unsigned (&vo)[R],
                                             const uint8_t *dig, const TAcc *ftab, int tid, int g, int part,
                                             TAcc (&acc)[R][NS]) {
    constexpr int J1 = K1 ? K1 : 1, J2 = K2 ? K2 : 1;
    // all slots odd: the middle of the product is Delta = 0 (diagonal part)
    constexpr bool odd = (K0 & 1) && (K1 == 0 || (K1 & 1)) && (K2 == 0 || (K2 & 1));
    const TAcc *__restrict__ cm = cmat_of<TAcc>(op);
    const int t1 = op.tgrp[g + 1];
    for (int t = op.tgrp[g] + ((part - op.tgrp[g]) & (S - 1)); t < t1; t += S) {
        const NvTermShape d = op.tshape[t];
        TAcc f0[R][K0], f1[R][J1], f2[R][J2];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const uint8_t *dq = dig + q * op.M * kBlock + tid;
            const int n0 = dq[d.mode[0] * kBlock];
#pragma unroll
            for (int i = 0; i < K0; ++i) f0[q][i] = ftab[d.code[0][i] * op.nmax + n0];
            if constexpr (K1 > 0) {
                const int n1 = dq[d.mode[1] * kBlock];
#pragma unroll
                for (int i = 0; i < K1; ++i) f1[q][i] = ftab[d.code[1][i] * op.nmax + n1];
            }
            if constexpr (K2 > 0) {
                const int n2 = dq[d.mode[2] * kBlock];
#pragma unroll
                for (int i = 0; i < K2; ++i) f2[q][i] = ftab[d.code[2][i] * op.nmax + n2];
            }
        }
        TAcc w[R][NS];
#pragma unroll
        for (int q = 0; q < R; ++q)
#pragma unroll
            for (int s = 0; s < NS; ++s) w[q][s] = (TAcc)0;
#pragma unroll
        for (int i0 = 0; i0 < K0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < J1; ++i1)
#pragma unroll
                for (int i2 = 0; i2 < J2; ++i2) {
                    if (odd && 2 * i0 + 1 == K0 && (K1 == 0 || 2 * i1 + 1 == K1) && (K2 == 0 || 2 * i2 + 1 == K2))
                        continue;
                    int off = d.base + i0 * d.inc[0];
                    if constexpr (K1 > 0) off += i1 * d.inc[1];
                    if constexpr (K2 > 0) off += i2 * d.inc[2];
                    const unsigned ob = (unsigned)off * XRes<NS, TIn>::kEl;
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        TAcc h = f0[q][i0];
                        if constexpr (K1 > 0) h *= f1[q][i1];
                        if constexpr (K2 > 0) h *= f2[q][i2];
                        unsigned o = vo[q] + ob;
                        if constexpr (SKIP) o = h != (TAcc)0 ? o : 0x80000000u;
                        xs.template fma<TAcc>(o, h, w[q]);
                    }
                }
        const TAcc *C = cm + (size_t)d.cm * NS * NS;
#pragma unroll
        for (int q = 0; q < R; ++q)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                TAcc a = acc[q][s];
#pragma unroll
                for (int s2 = 0; s2 < NS; ++s2) a += C[s * NS + s2] * w[q][s2];
                acc[q][s] = a;
            }
    }
}

template <int NS, typename TIn, typename TAcc, int R, bool SKIP, int S = 1>
__device__ __forceinline__ void offdiag_shaped(const NvOpDev &op, const XRes<NS, TIn> &xs, const unsigned (&vo)[R],
                                               const uint8_t *dig, const TAcc *ftab, int tid, TAcc (&acc)[R][NS],
                                               int part = 0) {
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[q][s] = (TAcc)0;
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 2, 0, 0>(op, xs, vo, dig, ftab, tid, 0, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 3, 0, 0>(op, xs, vo, dig, ftab, tid, 1, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 4, 0, 0>(op, xs, vo, dig, ftab, tid, 2, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 2, 2, 0>(op, xs, vo, dig, ftab, tid, 3, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 3, 2, 0>(op, xs, vo, dig, ftab, tid, 4, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 2, 3, 0>(op, xs, vo, dig, ftab, tid, 5, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 1, 2, 0>(op, xs, vo, dig, ftab, tid, 6, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 2, 1, 0>(op, xs, vo, dig, ftab, tid, 7, part, acc);
    shaped_group<NS, TIn, TAcc, R, SKIP, S, 2, 2, 2>(op, xs, vo, dig, ftab, tid, 8, part, acc);
}

template <typename TAcc>
__device__ __forceinline__ TAcc *stage_tables(const NvOpDev &op, uint8_t *&dig) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    TAcc *ftab = reinterpret_cast<TAcc *>(lds_raw);
    const int nt = op.ncodes * op.nmax;
    const TAcc *g = ftab_of<TAcc>(op);
    for (int i = threadIdx.x; i < nt; i += blockDim.x) ftab[i] = g[i];
    size_t off = ((size_t)nt * sizeof(TAcc) + 15) & ~(size_t)15;
    dig = lds_raw + off;
    return ftab;
}

// Standalone y = H x (x, y double).  TAcc selects the precision of the
// off-diagonal part; the diagonal part is always FP64.
template <int NS, typename TAcc>
__global__ __launch_bounds__(kBlock) void hv_full_kernel(NvOpDev op, const double *__restrict__ x,
                                                          double *__restrict__ y) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int r = xcd_block(blockIdx.x, gridDim.x) * kBlock + tid;
    const bool live = r < op.D;
    if (live) digits_energy(op, r, dig, tid);
    __syncthreads();
    if (!live) return;
    TAcc acc[NS];
    offdiag_accumulate<NS, double, TAcc>(op, x, r, dig, ftab, tid, acc);
    double v[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = x[(size_t)s * op.D + r];
    diag_apply<NS>(op, r, dig, tid, v, dv);
#pragma unroll
    for (int s = 0; s < NS; ++s) y[(size_t)s * op.D + r] = dv[s] + (double)acc[s];
}

// Iteration H*v: y = offdiag(H) q_i in TAcc, alpha(i) = q_i . (H q_i) in FP64.
template <int NS, typename TIn, typename TAcc>
__global__ __launch_bounds__(kBlock) void hv_iter_kernel(NvOpDev op, LzState st) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int r = xcd_block(blockIdx.x, gridDim.x) * kBlock + tid;
    const bool live = r < op.D;
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    const TIn *x = st.vlo ? reinterpret_cast<const TIn *>(st.vlo) : reinterpret_cast<const TIn *>(q);
    if (live) digits_energy(op, r, dig, tid);
    __syncthreads();
    double part = 0.0;
    if (live) {
        TAcc acc[NS];
        offdiag_accumulate<NS, TIn, TAcc>(op, x, r, dig, ftab, tid, acc);
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r];
        diag_apply<NS>(op, r, dig, tid, v, dv);
        TAcc *y = reinterpret_cast<TAcc *>(st.y);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y[(size_t)s * op.D + r] = acc[s];
            part += v[s] * (dv[s] + (double)acc[s]);
        }
    }
    const double b = block_sum(part);
    if (tid == 0) st.partials[blockIdx.x] = b;
}

// hv_iter_kernel with two rows per thread: block b covers the rows of the
// one-row kernel's blocks 2b and 2b+1 and writes their two partials, so alpha
// is the same sum in the same order.
template <int NS, typename TIn, typename TAcc>
__global__ __launch_bounds__(kBlock) void hv_iter2_kernel(NvOpDev op, LzState st) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    uint8_t *dig1 = dig + op.M * kBlock;
    const int tid = threadIdx.x;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = 2 * b * kBlock + tid, r1 = r0 + kBlock;
    const bool l0 = r0 < op.D, l1 = r1 < op.D;
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    const TIn *x = st.vlo ? reinterpret_cast<const TIn *>(st.vlo) : reinterpret_cast<const TIn *>(q);
    if (l0) digits_energy(op, r0, dig, tid);
    else for (int k = 0; k < op.M; ++k) dig[k * kBlock + tid] = 0;
    if (l1) digits_energy(op, r1, dig1, tid);
    else for (int k = 0; k < op.M; ++k) dig1[k * kBlock + tid] = 0;
    __syncthreads();
    double part0 = 0.0, part1 = 0.0;
    if (l0) {
        TAcc acc0[NS], acc1[NS];
        offdiag_accumulate2<NS, TIn, TAcc>(op, x, r0, r1, l0, l1, dig, dig1, ftab, tid, acc0, acc1);
        TAcc *y = reinterpret_cast<TAcc *>(st.y);
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r0];
        diag_apply<NS>(op, r0, dig, tid, v, dv);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y[(size_t)s * op.D + r0] = acc0[s];
            part0 += v[s] * (dv[s] + (double)acc0[s]);
        }
        if (l1) {
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r1];
            diag_apply<NS>(op, r1, dig1, tid, v, dv);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                y[(size_t)s * op.D + r1] = acc1[s];
                part1 += v[s] * (dv[s] + (double)acc1[s]);
            }
        }
    }
    const double s0 = block_sum(part0);
    const double s1 = block_sum(part1);
    if (tid == 0) {
        st.partials[2 * b] = s0;
        st.partials[2 * b + 1] = s1;
    }
}

// hv_iter_kernel over the shaped terms; R rows per thread.  Block b covers
// the rows of the one-row kernel's blocks R*b .. R*b+R-1 and writes their
// partials, so alpha is the same sum in the same order.  Rows past the end
// compute on zero digits and out-of-range loads; they are not written.
template <int NS, typename TIn, typename TAcc, int R, bool SKIP>
__global__ __launch_bounds__(kBlock) void hv_shaped_iter_kernel(NvOpDev op, LzState st) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    const TX *x = std::is_same<TIn, F64I>::value ? reinterpret_cast<const TX *>(st.v64i)
                  : st.vlo                       ? reinterpret_cast<const TX *>(st.vlo)
                                                 : reinterpret_cast<const TX *>(q);
    int r[R];
    bool live[R];
    unsigned vo[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        r[k] = (R * b + k) * kBlock + tid;
        live[k] = r[k] < op.D;
        vo[k] = (unsigned)r[k] * XRes<NS, TIn>::kEl;
        uint8_t *dk = dig + k * op.M * kBlock;
        if (live[k]) digits_energy(op, r[k], dk, tid);
        else for (int m = 0; m < op.M; ++m) dk[m * kBlock + tid] = 0;
    }
    __syncthreads();
    const XRes<NS, TIn> xs(x, op.D);
    TAcc acc[R][NS];
    offdiag_shaped<NS, TIn, TAcc, R, SKIP>(op, xs, vo, dig, ftab, tid, acc);
    TAcc *y = reinterpret_cast<TAcc *>(st.y);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        double part = 0.0;
        if (live[k]) {
            double v[NS], dv[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r[k]];
            diag_apply<NS>(op, r[k], dig + k * op.M * kBlock, tid, v, dv);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                y[(size_t)s * op.D + r[k]] = acc[k][s];
                part += v[s] * (dv[s] + (double)acc[k][s]);
            }
        }
        const double bs = block_sum(part);
        if (tid == 0) st.partials[R * b + k] = bs;
    }
}

// hv_full_kernel over the shaped terms.
template <int NS, typename TAcc>
__global__ __launch_bounds__(kBlock) void hv_shaped_full_kernel(NvOpDev op, const double *__restrict__ x,
                                                                 double *__restrict__ y) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int r = xcd_block(blockIdx.x, gridDim.x) * kBlock + tid;
    const bool live = r < op.D;
    if (live) digits_energy(op, r, dig, tid);
    else for (int m = 0; m < op.M; ++m) dig[m * kBlock + tid] = 0;
    __syncthreads();
    const XRes<NS, double> xs(x, op.D);
    const unsigned vo[1] = {(unsigned)r * 8u};
    TAcc acc[1][NS];
    offdiag_shaped<NS, double, TAcc, 1, false>(op, xs, vo, dig, ftab, tid, acc);
    if (!live) return;
    double v[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = x[(size_t)s * op.D + r];
    diag_apply<NS>(op, r, dig, tid, v, dv);
#pragma unroll
    for (int s = 0; s < NS; ++s) y[(size_t)s * op.D + r] = dv[s] + (double)acc[0][s];
}

// The off-diagonal rows of a workgroup whose S waves share 64 rows: every wave
// takes each S-th term, and wave 0 gets the sum, in wave order.  For vectors
// that leave the chip idle: with a row per thread, 72,765 rows of a cubic
// three-state operator are 285 workgroups, about one wave a SIMD, and the
// latency of 454 steps one after the other set the time (62 us, 41 with four
// waves a row).
template <int NS, typename TIn, typename TAcc, int S>
__device__ __forceinline__ void offdiag_split(const NvOpDev &op, const XRes<NS, TIn> &xs, int r, const uint8_t *dig,
                                              const TAcc *ftab, int lane, int wave, TAcc (&acc)[1][NS]) {
    __shared__ TAcc part[S - 1][NS][64];
    const unsigned vo[1] = {(unsigned)r * XRes<NS, TIn>::kEl};
    offdiag_shaped<NS, TIn, TAcc, 1, false, S>(op, xs, vo, dig, ftab, lane, acc, wave);
    if (wave > 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) part[wave - 1][s][lane] = acc[0][s];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < S - 1; ++w)
#pragma unroll
            for (int s = 0; s < NS; ++s) acc[0][s] += part[w][s][lane];
    }
}

// hv_shaped_iter_kernel, 64 rows a workgroup of S waves that share the terms
// (offdiag_split); a partial per workgroup.
template <int NS, typename TIn, typename TAcc, int S>
__global__ __launch_bounds__(64 * S) void hv_split_iter_kernel(NvOpDev op, LzState st) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    const TX *x = std::is_same<TIn, F64I>::value ? reinterpret_cast<const TX *>(st.v64i)
                                                 : reinterpret_cast<const TX *>(st.vlo);
    const XRes<NS, TIn> xs(x, op.D);
    const int r = b * 64 + lane;
    const bool live = r < op.D;
    if (wave == 0) {
        if (live) digits_energy(op, r, dig, lane);
        else for (int m = 0; m < op.M; ++m) dig[m * kBlock + lane] = 0;
    }
    __syncthreads();
    TAcc acc[1][NS];
    offdiag_split<NS, TIn, TAcc, S>(op, xs, r, dig, ftab, lane, wave, acc);
    if (wave > 0) return;
    TAcc *y = reinterpret_cast<TAcc *>(st.y);
    double part = 0.0;
    if (live) {
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r];
        diag_apply<NS>(op, r, dig, lane, v, dv);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y[(size_t)s * op.D + r] = acc[0][s];
            part += v[s] * (dv[s] + (double)acc[0][s]);
        }
    }
    part = wave_sum(part);
    if (lane == 0) st.partials[b] = part;
}

// hv_shaped_full_kernel in the same form.
template <int NS, typename TAcc, int S>
__global__ __launch_bounds__(64 * S) void hv_split_full_kernel(NvOpDev op, const double *__restrict__ x,
                                                               double *__restrict__ y) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
    const bool live = r < op.D;
    if (wave == 0) {
        if (live) digits_energy(op, r, dig, lane);
        else for (int m = 0; m < op.M; ++m) dig[m * kBlock + lane] = 0;
    }
    __syncthreads();
    const XRes<NS, double> xs(x, op.D);
    TAcc acc[1][NS];
    offdiag_split<NS, double, TAcc, S>(op, xs, r, dig, ftab, lane, wave, acc);
    if (wave > 0 || !live) return;
    double v[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = x[(size_t)s * op.D + r];
    diag_apply<NS>(op, r, dig, lane, v, dv);
#pragma unroll
    for (int s = 0; s < NS; ++s) y[(size_t)s * op.D + r] = dv[s] + (double)acc[0][s];
}

// ------------------------------------------------------------------------
// Two-pass H*v (tables in NvHv2Dev).  A term t = C_t (x) P_sigma (x) P_phi
// splits into sigma, its powers of the two slowest modes 0 and 1, and phi,
// its monomial over the other modes.  With x_r the row r of x (all states):
//   pass 1: Z_g[r] = sum over the terms with sigma = g of C_t (P_phi x)[r],
//           each distinct phi gathered once per row and fed to every
//           channel g it pairs with;
//   pass 2: y[r] = Z_0[r] + sum_{g > 0} sum_{Delta_0, Delta_1}
//           h_0 h_1 Z_g[r + Delta_0 shft_0 + Delta_1 shft_1].
// The step Delta = 0 of the whole term is diagonal (it lives in the FP64
// diagonal part): pass 1 leaves out phi's zero step for g = 0 only, and pass 2
// takes the pure q_a^2 term's C_t h(2, n_a, 0) x_r out again at Delta_a = 0.
// Pass 1 does the distinct phi's gathers (cubic 4-state operator on 10 modes:
// 936 of the one-pass form's 1760 per row) and all the coupling products;
// pass 2 streams the channels along the two slow modes, a workgroup covering
// every (n_0, n_1) of a few consecutive rows of the faster modes so that each
// channel row is fetched from memory once.
// ------------------------------------------------------------------------
typedef float nv_mf4 __attribute__((ext_vector_type(4)));

// Channel accumulators of pass 1.  VALU form: one row per lane, NS values per
// channel.  MFMA form (FP32, NS <= 4): the coupling products run on the
// matrix cores as v_mfma_f32_4x4x1 (16 blocks of 4 lanes): block b of a wave
// is its rows 4b..4b+3; A = the lane's own phi value of state s', B = row
// (lane & 3) of C_t at column s', so lane 4b+j, register i accumulates row
// 4b+i, state j.  The VALU is left with the gathers.
template <int NS, typename TAcc, bool MF> struct Hv2Acc {
    TAcc a[NV_HV2_NG][NS];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int g = 0; g < NV_HV2_NG; ++g)
#pragma unroll
            for (int s = 0; s < NS; ++s) a[g][s] = (TAcc)0;
    }
    template <int G> __device__ __forceinline__ void mix(const TAcc *C, const TAcc (&u)[NS]) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            TAcc v = a[G][s];
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2) v += C[s * NS + s2] * u[s2];
            a[G][s] = v;
        }
    }
};
template <int NS> struct Hv2Acc<NS, float, true> {
    nv_mf4 a[NV_HV2_NG];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int g = 0; g < NV_HV2_NG; ++g) a[g] = nv_mf4{0.f, 0.f, 0.f, 0.f};
    }
    // C: the lane's row (lane & 3) of the 4x4-padded coupling matrix
    template <int G> __device__ __forceinline__ void mix(const float *C, const float (&u)[NS]) {
        const nv_mf4 c = *reinterpret_cast<const nv_mf4 *>(C);
#pragma unroll
        for (int s2 = 0; s2 < NS; ++s2) a[G] = __builtin_amdgcn_mfma_f32_4x4x1f32(u[s2], c[s2], a[G], 0, 0, 0);
    }
};

// The coupling rows a consumer reads: global C_t (VALU) or the lane's row of
// the padded copy staged in LDS (MFMA).
template <int NS, typename TAcc, bool MF>
__device__ __forceinline__ const TAcc *hv2_cmat(const NvOpDev &op, const float *ldsc, int cm) {
    if constexpr (MF) return reinterpret_cast<const TAcc *>(ldsc + cm * 16 + (threadIdx.x & 3) * 4);
    else return cmat_of<TAcc>(op) + (size_t)cm * NS * NS;
}

// acc[g] += C_g u over the channels: cm[g] is the term's cmat row, or -1
// (uniform over the wave); ucm0 is fed to channel 0, u to the others.
template <int NS, typename TAcc, bool MF>
__device__ __forceinline__ void hv2_feed(const NvOpDev &op, const float *ldsc, Hv2Acc<NS, TAcc, MF> &acc,
                                         const int32_t (&cm)[NV_HV2_NG], const TAcc (&u0)[NS], const TAcc (&u)[NS]) {
    if (cm[0] >= 0) acc.template mix<0>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[0]), u0);
    if (cm[1] >= 0) acc.template mix<1>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[1]), u);
    if (cm[2] >= 0) acc.template mix<2>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[2]), u);
    if (cm[3] >= 0) acc.template mix<3>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[3]), u);
    if (cm[4] >= 0) acc.template mix<4>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[4]), u);
    if (cm[5] >= 0) acc.template mix<5>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[5]), u);
    if (cm[6] >= 0) acc.template mix<6>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[6]), u);
    if (cm[7] >= 0) acc.template mix<7>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[7]), u);
    if (cm[8] >= 0) acc.template mix<8>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[8]), u);
    if (cm[9] >= 0) acc.template mix<9>(hv2_cmat<NS, TAcc, MF>(op, ldsc, cm[9]), u);
}

// The phis of shape group grp: steps gathered as in shaped_group (one row per
// thread, out-of-basis loads pointed outside the vector), then fed to their
// consumers.  u leaves out phi's zero step (for channel 0, where the whole
// step would be diagonal), uf keeps it.
template <int NS, typename TIn, typename TAcc, bool MF, bool SKIP, int K0, int K1, int K2>
__device__ __forceinline__ void hv2_phi_group(const NvOpDev &op, const XRes<NS, TIn> &xs, unsigned vo,
                                              const uint8_t *dig, const TAcc *ftab, const float *ldsc, int tid,
                                              int grp, const TAcc (&xr)[NS], Hv2Acc<NS, TAcc, MF> &acc) {
    constexpr int J1 = K1 ? K1 : 1, J2 = K2 ? K2 : 1;
    constexpr bool zs = (K0 & 1) && (K1 == 0 || (K1 & 1)) && (K2 == 0 || (K2 & 1));
    const NvHv2Dev &h = op.hv2;
    const int p1 = h.pgrp[grp + 1];
    for (int p = h.pgrp[grp]; p < p1; ++p) {
        const NvPhi &ph = h.phi[p];
        const NvTermShape d = ph.sh;
        TAcc f0[K0], f1[J1], f2[J2];
        const uint8_t *dq = dig + tid;
        const int n0 = dq[d.mode[0] * kBlock];
        TAcc fd = (TAcc)1;  // the factors of the modes whose only step is Delta = 0
        for (int j = 0; j < ph.nd; ++j) fd *= ftab[ph.dcode[j] * op.nmax + dq[ph.dmode[j] * kBlock]];
#pragma unroll
        for (int i = 0; i < K0; ++i) f0[i] = ftab[d.code[0][i] * op.nmax + n0] * fd;
        if constexpr (K1 > 0) {
            const int n1 = dq[d.mode[1] * kBlock];
#pragma unroll
            for (int i = 0; i < K1; ++i) f1[i] = ftab[d.code[1][i] * op.nmax + n1];
        } else {
            f1[0] = (TAcc)1;
        }
        if constexpr (K2 > 0) {
            const int n2 = dq[d.mode[2] * kBlock];
#pragma unroll
            for (int i = 0; i < K2; ++i) f2[i] = ftab[d.code[2][i] * op.nmax + n2];
        } else {
            f2[0] = (TAcc)1;
        }
        TAcc u[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) u[s] = (TAcc)0;
#pragma unroll
        for (int i0 = 0; i0 < K0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < J1; ++i1) {
                TAcc h01 = f0[i0];
                if constexpr (K1 > 0) h01 *= f1[i1];
#pragma unroll
                for (int i2 = 0; i2 < J2; ++i2) {
                    if (zs && 2 * i0 + 1 == K0 && (K1 == 0 || 2 * i1 + 1 == K1) && (K2 == 0 || 2 * i2 + 1 == K2))
                        continue;
                    int off = d.base + i0 * d.inc[0];
                    if constexpr (K1 > 0) off += i1 * d.inc[1];
                    if constexpr (K2 > 0) off += i2 * d.inc[2];
                    TAcc hf = h01;
                    if constexpr (K2 > 0) hf *= f2[i2];
                    // plain form: an out-of-basis step reads some row (or 0 past the ends) times 0
                    unsigned o = vo + (unsigned)off * XRes<NS, TIn>::kEl;
                    if constexpr (SKIP) o = hf != (TAcc)0 ? o : 0x80000000u;
                    xs.template fma<TAcc>(o, hf, u);
                }
            }
        TAcc uf[NS];
        if constexpr (zs) {
            TAcc z = f0[(K0 - 1) / 2];
            if constexpr (K1 > 0) z *= f1[(K1 - 1) / 2];
            if constexpr (K2 > 0) z *= f2[(K2 - 1) / 2];
#pragma unroll
            for (int s = 0; s < NS; ++s) uf[s] = u[s] + z * xr[s];
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) uf[s] = u[s];
        }
        hv2_feed<NS, TAcc, MF>(op, ldsc, acc, ph.cm, u, uf);
    }
}

__device__ __forceinline__ size_t hv2_tables_bytes(const NvOpDev &op, size_t el) {
    return (((size_t)op.ncodes * op.nmax * el + 15) & ~(size_t)15) + 2 * (size_t)op.M * kBlock;
}

// Pass 1: Z_g[r] for every channel, x the interleaved copy of the vector
// (FP32, or FP64 as F64I).  Z is [NV_HV2_NG][D][nv_lo_stride(NS)].
template <int NS, typename TIn, typename TAcc, bool MF, bool SKIP>
__global__ __launch_bounds__(kBlock) void hv2_pass1_kernel(NvOpDev op, const void *__restrict__ xin,
                                                            TAcc *__restrict__ Z) {
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    float *ldsc = nullptr;
    if constexpr (MF) {
        extern __shared__ __align__(16) unsigned char lds_raw[];
        ldsc = reinterpret_cast<float *>(lds_raw + hv2_tables_bytes(op, sizeof(float)));
        for (int i = threadIdx.x; i < op.nterms * 16; i += blockDim.x) {
            const int t = i >> 4, j = (i >> 2) & 3, k = i & 3;
            ldsc[i] = (j < NS && k < NS) ? op.cmat32[(size_t)t * NS * NS + j * NS + k] : 0.f;
        }
    }
    const int tid = threadIdx.x;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r = b * kBlock + tid;
    const bool live = r < op.D;
    if (live) digits_energy(op, r, dig, tid);
    else for (int m = 0; m < op.M; ++m) dig[m * kBlock + tid] = 0;
    __syncthreads();
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    const XRes<NS, TIn> xs(reinterpret_cast<const TX *>(xin), op.D);
    const unsigned vo = (unsigned)r * XRes<NS, TIn>::kEl;
    TAcc xr[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) xr[s] = (TAcc)0;
    xs.template fma<TAcc>(vo, (TAcc)1, xr);  // row r itself (0 past the end)
    Hv2Acc<NS, TAcc, MF> acc;
    acc.zero();
    const NvHv2Dev &h = op.hv2;
    hv2_feed<NS, TAcc, MF>(op, ldsc, acc, h.idcm, xr, xr);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 2, 0, 0>(op, xs, vo, dig, ftab, ldsc, tid, 0, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 3, 0, 0>(op, xs, vo, dig, ftab, ldsc, tid, 1, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 4, 0, 0>(op, xs, vo, dig, ftab, ldsc, tid, 2, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 2, 2, 0>(op, xs, vo, dig, ftab, ldsc, tid, 3, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 3, 2, 0>(op, xs, vo, dig, ftab, ldsc, tid, 4, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 2, 3, 0>(op, xs, vo, dig, ftab, ldsc, tid, 5, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 1, 2, 0>(op, xs, vo, dig, ftab, ldsc, tid, 6, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 2, 1, 0>(op, xs, vo, dig, ftab, ldsc, tid, 7, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 2, 2, 2>(op, xs, vo, dig, ftab, ldsc, tid, 8, xr, acc);
    hv2_phi_group<NS, TIn, TAcc, MF, SKIP, 1, 0, 0>(op, xs, vo, dig, ftab, ldsc, tid, 9, xr, acc);
    constexpr int P = nv_lo_stride(NS);
    if constexpr (MF) {
        const int rw = b * kBlock + (tid & ~63) + 4 * ((tid & 63) >> 2);
        const int j = tid & 3;
#pragma unroll
        for (int g = 0; g < NV_HV2_NG; ++g) {
            if (!((h.gmask >> g) & 1)) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (rw + i < op.D && j < NS) Z[((size_t)g * op.D + rw + i) * P + j] = acc.a[g][i];
        }
    } else {
        if (!live) return;
#pragma unroll
        for (int g = 0; g < NV_HV2_NG; ++g) {
            if (!((h.gmask >> g) & 1)) continue;
#pragma unroll
            for (int s = 0; s < NS; ++s) Z[((size_t)g * op.D + r) * P + s] = acc.a[g][s];
        }
    }
}

// Pass 2, one signature channel g of powers (P0, P1) on modes 0 and 1: the
// R2 consecutive rows r0..r0+R2-1 of a thread share (n_0, n_1) and so every
// factor.  Steps leaving the basis have factor 0 (factor table) and their
// loads are pointed outside the buffer; no branch.  A signature whose step
// range was cut by a small basis (s < p) takes the generic loop.
template <int NS, typename TIn, typename TAcc, int R2, int P0, int P1>
__device__ __forceinline__ void hv2_sig_rows(const NvOpDev &op, const NvSigma &sg, const XRes<NS, TIn> &zg, int r0,
                                             int n0, int n1, int nf0, TAcc (&y)[R2][NS]) {
    const NvHv2Dev &h = op.hv2;
    const TAcc *ft = ftab_of<TAcc>(op);
    constexpr unsigned kEl = XRes<NS, TIn>::kEl;
    if (sg.s0 == (P0 ? P0 : -1) && sg.s1 == (P1 ? P1 : -1)) {
        constexpr int K0 = P0 ? P0 + 1 : 1, K1 = P1 ? P1 + 1 : 1;
        TAcc f0[K0], f1[K1];
#pragma unroll
        for (int i = 0; i < K0; ++i) f0[i] = P0 ? ft[sg.code0[i] * op.nmax + n0] : (TAcc)1;
#pragma unroll
        for (int i = 0; i < K1; ++i) f1[i] = P1 ? ft[sg.code1[i] * op.nmax + n1] : (TAcc)1;
#pragma unroll
        for (int i0 = 0; i0 < K0; ++i0)
#pragma unroll
            for (int i1 = 0; i1 < K1; ++i1) {
                const int d0 = P0 ? 2 * i0 - P0 : 0, d1 = P1 ? 2 * i1 - P1 : 0;
                const TAcc f = f0[i0] * f1[i1];
                const int off = (d0 * h.n1 + d1) * h.dr;
#pragma unroll
                for (int k = 0; k < R2; ++k) {
                    const unsigned o = f != (TAcc)0 ? (unsigned)(r0 + k + off) * kEl : 0x80000000u;
                    zg.template fma<TAcc>(o, f, y[k]);
                }
            }
        return;
    }
    const int k0 = sg.s0 < 0 ? 1 : sg.s0 + 1, k1 = sg.s1 < 0 ? 1 : sg.s1 + 1;
    for (int i0 = 0; i0 < k0; ++i0) {
        const int d0 = sg.s0 < 0 ? 0 : 2 * i0 - sg.s0;
        if (n0 + d0 < 0 || n0 + d0 >= nf0) continue;
        const TAcc f0 = sg.s0 < 0 ? (TAcc)1 : ft[sg.code0[i0] * op.nmax + n0];
        for (int i1 = 0; i1 < k1; ++i1) {
            const int d1 = sg.s1 < 0 ? 0 : 2 * i1 - sg.s1;
            if (n1 + d1 < 0 || n1 + d1 >= h.n1) continue;
            const TAcc f1 = sg.s1 < 0 ? (TAcc)1 : ft[sg.code1[i1] * op.nmax + n1];
            const int off = (d0 * h.n1 + d1) * h.dr;
#pragma unroll
            for (int k = 0; k < R2; ++k) zg.template fma<TAcc>((unsigned)(r0 + k + off) * kEl, f0 * f1, y[k]);
        }
    }
}

template <int NS, typename TIn, typename TAcc, int R2, int G, int P0, int P1>
__device__ __forceinline__ void hv2_channel(const NvOpDev &op, const TAcc *Z, int r0, int n0, int n1, int nf0,
                                            TAcc (&y)[R2][NS]) {
    if (!((op.hv2.gmask >> G) & 1)) return;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    const XRes<NS, TIn> zg(reinterpret_cast<const TX *>(Z) + (size_t)G * op.D * nv_lo_stride(NS), op.D);
    hv2_sig_rows<NS, TIn, TAcc, R2, P0, P1>(op, op.hv2.sig[G], zg, r0, n0, n1, nf0, y);
}

// Pass 2: y_off from the channels for R2 consecutive rows per thread; ITER:
// the iteration's epilogue (y in the accumulation type, state-major; alpha
// partials with the FP64 diagonal, one per workgroup), else y = diag x + y_off
// in FP64 (standalone H*v).  Workgroup: the h.nl planes (n_0, n_1) times h.c
// threads of R2 consecutive plane rows each, so that every channel row comes
// from memory once and is reused from the caches for its neighbours.
template <int NS, typename TIn, typename TAcc, bool ITER, int R2>
__global__ __launch_bounds__(kBlock) void hv2_pass2_kernel(NvOpDev op, LzState st, const void *__restrict__ xin,
                                                            const TAcc *__restrict__ Z,
                                                            const double *__restrict__ xfull,
                                                            double *__restrict__ yfull) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    uint8_t *dig = lds_raw;
    const NvHv2Dev &h = op.hv2;
    const int tid = threadIdx.x;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int lpos = tid / h.c;
    const int rest0 = (b * h.c + (tid - lpos * h.c)) * R2;
    const bool inl = lpos < h.nl && rest0 < h.dr;
    const int r0 = inl ? lpos * h.dr + rest0 : 0;
    const int n0 = lpos / h.n1, n1 = lpos - (lpos / h.n1) * h.n1;
    const int nf0 = h.nl / h.n1;
    using TX = typename std::conditional<std::is_same<TIn, F64I>::value, double, TIn>::type;
    constexpr unsigned kEl = XRes<NS, TIn>::kEl;
    TAcc y[R2][NS];
#pragma unroll
    for (int k = 0; k < R2; ++k)
#pragma unroll
        for (int s = 0; s < NS; ++s) y[k][s] = (TAcc)0;
    if (inl) {
        if (h.gmask & 1) {
            const XRes<NS, TIn> z0(reinterpret_cast<const TX *>(Z), op.D);
#pragma unroll
            for (int k = 0; k < R2; ++k)
                if (rest0 + k < h.dr) z0.template fma<TAcc>((unsigned)(r0 + k) * kEl, (TAcc)1, y[k]);
        }
        hv2_channel<NS, TIn, TAcc, R2, 1, 1, 0>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 2, 2, 0>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 3, 3, 0>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 4, 0, 1>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 5, 0, 2>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 6, 0, 3>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 7, 1, 1>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 8, 2, 1>(op, Z, r0, n0, n1, nf0, y);
        hv2_channel<NS, TIn, TAcc, R2, 9, 1, 2>(op, Z, r0, n0, n1, nf0, y);
        // the pure q_a^2 terms at Delta_a = 0 are diagonal: take them out again
        for (int g = 2; g <= 5; g += 3) {
            const NvSigma &sg = h.sig[g];
            if (!((h.gmask >> g) & 1) || sg.corr_cm < 0) continue;
            const TAcc hz = ftab_of<TAcc>(op)[sg.corr_code * op.nmax + (g <= 3 ? n0 : n1)];
            const TAcc *C = cmat_of<TAcc>(op) + (size_t)sg.corr_cm * NS * NS;
            const XRes<NS, TIn> xs(reinterpret_cast<const TX *>(xin), op.D);
#pragma unroll
            for (int k = 0; k < R2; ++k) {
                TAcc xr[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) xr[s] = (TAcc)0;
                xs.template fma<TAcc>((unsigned)(r0 + k) * kEl, (TAcc)1, xr);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    TAcc a = (TAcc)0;
#pragma unroll
                    for (int s2 = 0; s2 < NS; ++s2) a += C[s * NS + s2] * xr[s2];
                    y[k][s] -= hz * a;
                }
            }
        }
    }
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < R2; ++k) {
        const bool live = inl && rest0 + k < h.dr;
        const int r = r0 + k;
        if (op.offstate && live) digits_energy(op, r, dig, tid);
        if (!live) continue;
        double v[NS], dv[NS];
        if constexpr (ITER) {
            const int64_t it = *st.iter;
            const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r];
            diag_apply<NS>(op, r, dig, tid, v, dv);
            TAcc *yo = reinterpret_cast<TAcc *>(st.y);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                yo[(size_t)s * op.D + r] = y[k][s];
                part += v[s] * (dv[s] + (double)y[k][s]);
            }
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = xfull[(size_t)s * op.D + r];
            diag_apply<NS>(op, r, dig, tid, v, dv);
#pragma unroll
            for (int s = 0; s < NS; ++s) yfull[(size_t)s * op.D + r] = dv[s] + (double)y[k][s];
        }
    }
    if constexpr (ITER) {
        const double bs = block_sum(part);
        if (tid == 0) st.partials[b] = bs;
    }
}

// The finishing kernel's sum of parts[0, n) (finish_sum_kernel: strided
// per-thread sums, then the block tree), in every workgroup of kBlock threads.
__device__ __forceinline__ double fold_sum(const double *parts, int n) {
    double s = 0.0;
#pragma unroll 8
    for (int i = threadIdx.x; i < n; i += kBlock) s += parts[i];
    return block_sum(s);
}

// lanczos_step (Source/top.f90:820-842): r = (H q_i - alpha q_i) - beta(i-1) q_{i-1}
// stored in slot i+1, beta(i) = |r|.
template <int NS, typename TAcc, bool NT>
__global__ __launch_bounds__(kBlock) void lanczos_step_kernel(NvOpDev op, LzState st) {
    extern __shared__ __align__(16) unsigned char dig[];  // M*kBlock bytes when states couple through D
    const int tid = threadIdx.x;
    const int r = blockIdx.x * kBlock + tid;
    const int64_t it = *st.iter;
    const double *q = st.V + slot_of(it, st.nslots) * (int64_t)op.N;
    const double *qm = st.V + slot_of(it - 1, st.nslots) * (int64_t)op.N;
    double *res = st.V + slot_of(it + 1, st.nslots) * (int64_t)op.N;
    double a;
    if (st.fold_in) {
        a = fold_sum(st.fold_in, st.fold_n);
        if (blockIdx.x == 0 && tid == 0) st.alpha[it] = a;
    } else {
        a = st.alpha[it];
    }
    const double b = it > 1 ? st.beta[it - 1] : 0.0;
    double part = 0.0;
    if (r < op.D) {
        if (op.offstate) digits_energy(op, r, dig, tid);
        double v[NS], dv[NS];
        // every vector is streamed once
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = ld_once<NT>(&q[(size_t)s * op.D + r]);
#pragma unroll
        for (int s = 0; s < NS; ++s) dv[s] = ld_once<NT>(&op.dg[(size_t)s * op.D + r]) * v[s];
        if (op.offstate) diag_offstate<NS>(op, dig, tid, v, dv);
        const TAcc *y = reinterpret_cast<const TAcc *>(st.y);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const size_t o = (size_t)s * op.D + r;
            double w = dv[s] + (double)ld_once<NT>(&y[o]);
            w = w - a * v[s];
            if (it > 1) w = w - b * ld_once<NT>(&qm[o]);
            st_once<NT>(w, &res[o]);
            part += w * w;
        }
    }
    const double bs = block_sum(part);
    if (tid == 0) (st.fold_out ? st.fold_out : st.partials)[blockIdx.x] = bs;
    if (st.next_iter && blockIdx.x == 0 && tid == 0) *st.next_iter = it + st.next_inc;
}


// update_lanczos (Source/top.f90:646-670): q_i = r / beta(i-1) in place, and
// the copies of q_i that H*v and re-orthogonalisation read.  A thread takes
// the NS states of row r, so an interleaved copy gets one row store.
template <int NS, typename TIn, bool NT>
__global__ __launch_bounds__(kBlock) void normalize_rows_kernel(int64_t N, int64_t D, LzState st) {
    constexpr int NSP = nv_lo_stride(NS);
    const int64_t it = *st.iter + st.iter_add;
    if (st.iter_pub && blockIdx.x == 0 && threadIdx.x == 0) *st.iter_pub = it;
    double *q = st.V + slot_of(it, st.nslots) * N;
    double bprev;
    if (st.fold_in && (!st.fold_cond || *st.fold_cond != 0)) {
        bprev = sqrt(fold_sum(st.fold_in, st.fold_n));
        if (blockIdx.x == 0 && threadIdx.x == 0) st.beta[it - 1] = bprev;
    } else {
        bprev = st.beta[it - 1];
    }
    const double sc = 1.0 / bprev;
    TIn *lo = reinterpret_cast<TIn *>(st.vlo);
    float *vf = st.Vf ? st.Vf + slot_of(it, st.nslots) * st.ldf : nullptr;
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < D; r += (int64_t)gridDim.x * kBlock) {
        double v[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            v[s] = ld_once<NT>(&q[s * D + r]) * sc;
            st_once<NT>(v[s], &q[s * D + r]);
            if (vf) vf[s * D + r] = (float)v[s];
        }
        if (lo) {
            IlRow<TIn, NSP> row;
#pragma unroll
            for (int k = 0; k < NSP; ++k) row.v[k] = from_d<TIn>(k < NS ? v[k] : 0.0);
            reinterpret_cast<IlRow<TIn, NSP> *>(lo)[r] = row;
        }
        if (st.v64i) {
            IlRow<double, NSP> row;
#pragma unroll
            for (int k = 0; k < NSP; ++k) row.v[k] = k < NS ? v[k] : 0.0;
            reinterpret_cast<IlRow<double, NSP> *>(st.v64i)[r] = row;
        }
    }
}

__global__ void set_iter_kernel(int64_t *it, int64_t v, int inc) {
    if (threadIdx.x == 0) *it = inc ? *it + 1 : v;
}

__global__ __launch_bounds__(kBlock) void fill_start_kernel(double *v, int64_t D, int ns, const double *vals) {
    const int64_t N = D * ns;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < N; i += (int64_t)gridDim.x * kBlock) {
        const int64_t s = i / D, r = i - s * D;
        v[i] = r == 0 ? vals[s] : 0.0;
    }
}

__global__ __launch_bounds__(kBlock) void norm_kernel(const double *v, int64_t n, double *partials) {
    double p = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        p += v[i] * v[i];
    const double b = block_sum(p);
    if (threadIdx.x == 0) partials[blockIdx.x] = b;
}

// Sums nparts per-block partials in block order (one block; the kernel
// boundary makes the partials visible) and stores the sum, or its square
// root, at out[*iter] (iter null: out[0]); then, with advance, sets
// *advance = *iter + 1 (the next iteration's counter, in place of a launch).
__global__ __launch_bounds__(kBlock) void finish_sum_kernel(const double *partials, int nparts, double *out,
                                                           const int64_t *iter, int take_sqrt, int64_t *advance) {
    double s = 0.0;
    // loads unrolled ahead of the adds, which keep their order (32 in flight per
    // thread: 86,400 partials are 338 per thread)
#pragma unroll 32
    for (int i = threadIdx.x; i < nparts; i += kBlock) s += partials[i];
    s = block_sum(s);
    if (threadIdx.x == 0) {
        const int64_t k = iter ? *iter : 0;
        out[k] = take_sqrt ? sqrt(s) : s;
        if (advance) *advance = k + 1;
    }
}

hipError_t launch_finish_sum(const double *partials, int nparts, double *out, const int64_t *iter, int take_sqrt,
                             hipStream_t s, int64_t *advance) {
    hipLaunchKernelGGL(finish_sum_kernel, dim3(1), dim3(kBlock), 0, s, partials, nparts, out, iter, take_sqrt,
                       advance);
    return hipGetLastError();
}

// ------------------------------------------------------------------------
// host launchers for the above
// ------------------------------------------------------------------------
size_t hv_lds_bytes(const NvOpDev &op, int prec) {
    const size_t el = prec == 0 ? sizeof(double) : sizeof(float);
    size_t off = ((size_t)op.ncodes * op.nmax * el + 15) & ~(size_t)15;
    return off + 2 * (size_t)op.M * kBlock;  // digits of up to two rows per thread
}

int hv_blocks(const NvOpDev &op) { return (op.D + kBlock - 1) / kBlock; }

static int grid_stride_blocks(int64_t n) {
    int64_t b = (n + kBlock - 1) / kBlock;
    return (int)(b < 8192 ? b : 8192);
}

// Above op.skip_min_bytes of vector (set per context: kSkipMinBytes, or less
// for operators with many out-of-basis steps) the shaped kernels point the
// loads of out-of-basis steps outside the buffer (no memory traffic) instead
// of at a wrong row.
constexpr int64_t kSkipMinBytes = (int64_t)128 << 20;
constexpr int kShapedMaxStates = NV_MAXS;

// The shaped kernels serve operators whose terms all have a shape (ordr <= 3),
// any number of states (up to NV_MAXS), FP64 or FP32, with every row offset inside a 32-bit
// buffer range; op.tshape = nullptr selects the step-table kernels.
bool shaped_ok(const NvOpDev &op, int64_t el) {
    if (!op.tshape || op.ns > kShapedMaxStates) return false;
    return ((int64_t)op.D + 2 * kBlock) * el < ((int64_t)1 << 31);
}

// The Lanczos iteration in FP64 reads the interleaved copy LzState::v64i (one
// 16-byte load per two states).  The standalone and batched H*v read the
// state-major vector, one load per state and step, and keep the step-table
// form above kSkipMinBytes, where its branch over out-of-basis steps wins
// (N = 88.5M, four states: 55.9 against 65.7 ms per H*v).
int64_t hv_skip_min_bytes() { return kSkipMinBytes; }

bool hv_shaped(const NvOpDev &op, int prec) {
    if (prec == 0) return shaped_ok(op, nv_lo_stride(op.ns) * 8);
    if (prec == 1) return shaped_ok(op, nv_lo_stride(op.ns) * 4);
    return false;
}

bool hv_shaped_skip(const NvOpDev &op, int prec) {
    const int64_t vbytes = (int64_t)op.D * nv_lo_stride(op.ns) * (prec == 0 ? 8 : 4);
    return hv_shaped(op, prec) && vbytes > op.skip_min_bytes;
}

// Standalone and batched H*v read the state-major FP64 vector itself.
static bool shaped_state_major(const NvOpDev &op) {
    return shaped_ok(op, 8) && (int64_t)op.D * 8 * op.ns <= kSkipMinBytes;
}

bool hv_shaped_batch(const NvOpDev &op, int prec) { return prec == 0 ? shaped_state_major(op) : hv_shaped(op, prec); }

// The FP64 H*v shares the terms of a row over the kSplitWaves waves of a
// workgroup up to kSplitRows rows (iteration: 64 rows a partial, and no more
// partials than the folded finishing sums take) or kSplitFullRows (standalone,
// no partials).  33 iterations, one wave a row against four: 1,000 rows of two
// states 539 -> 502 us, 3,500 of four states (cubic) 1349 -> 742, 72,765 of
// three (cubic) 2467 -> 1802, 175,616 of two 1139 -> 1013, 262,144 of two
// (cubic) 2781 -> 2528.  Two waves give less below 100,000 rows, eight lose
// above (100,000 rows 1025 -> 943 us with four, 1010 with eight).  Standalone,
// 460,800 rows of three states: 61.2 -> 56.6 us, cubic 298 -> 272.
// kSplitMinRows is no line of speed: below it the shared form is the faster one
// too (33 iterations, 64 rows of two states 462 against 404 us, 432 cubic rows
// of three 1240 against 655).  But such a run soon exhausts its Krylov space,
// after which rounding alone decides the coefficients, and it keeps the sums of
// the batched kernels so that a problem gives the same numbers alone and in a
// batch.
// In FP32 it serves operators of kSplitTerms32 terms or more: those whose
// steps are too many for the run-time compiled kernel.  17 iterations, cubic
// operators of 9 and 10 modes: 1,536 rows of four states 2061 -> 720 us,
// 19,683 of two 1478 -> 646, 104,976 of three 2281 -> 1860, 248,832 of three
// 4093 -> 3793; the error against 64 bits falls by 20 to 40% (four short FP32
// sums instead of one long one: 3.5-5.9e-8 to 2.8-3.7e-8 over six operators).
constexpr int kSplitWaves = 4;
constexpr int kSplitTerms32 = 200;
constexpr int kSplitMinRows = 512;
constexpr int kSplitRows = 64 * 4096;
constexpr int kSplitFullRows = 1 << 19;
static bool hv_split(const NvOpDev &op, int prec, int rows) {
    // beside the tables, the sums of the waves after the first
    return (prec == 0 || (prec == 1 && op.nterms >= kSplitTerms32)) && op.D >= kSplitMinRows && op.D <= rows &&
           hv_lds_bytes(op, 0) + (size_t)(kSplitWaves - 1) * op.ns * 64 * sizeof(double) <= 65536;
}
static unsigned hv_split_blocks(const NvOpDev &op) { return (unsigned)((op.D + 63) / 64); }
int hv_split_waves(const NvOpDev &op, int prec) {
    return hv_shaped(op, prec) && !hv_shaped_skip(op, prec) && hv_split(op, prec, kSplitRows) ? kSplitWaves : 1;
}
static bool hv_split_iter(const NvOpDev &op, int prec, const LzState &st) {
    return (prec == 0 ? (void *)st.v64i : st.vlo) && hv_split_waves(op, prec) > 1;
}

template <int NS>
static hipError_t hv_full_ns(const NvOpDev &op, int prec, const double *x, double *y, hipStream_t s) {
    const size_t lds = hv_lds_bytes(op, prec);
    if constexpr (NS <= kShapedMaxStates) {
        if (shaped_state_major(op)) {
            if (prec == 0 && hv_split(op, prec, kSplitFullRows))
                hipLaunchKernelGGL((hv_split_full_kernel<NS, double, kSplitWaves>), dim3(hv_split_blocks(op)),
                                   dim3(64 * kSplitWaves), lds, s, op, x, y);
            else if (hv_split(op, prec, kSplitFullRows))
                hipLaunchKernelGGL((hv_split_full_kernel<NS, float, kSplitWaves>), dim3(hv_split_blocks(op)),
                                   dim3(64 * kSplitWaves), lds, s, op, x, y);
            else if (prec == 0)
                hipLaunchKernelGGL((hv_shaped_full_kernel<NS, double>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op,
                                   x, y);
            else
                hipLaunchKernelGGL((hv_shaped_full_kernel<NS, float>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op,
                                   x, y);
            return hipGetLastError();
        }
    }
    if (prec == 0)
        hipLaunchKernelGGL((hv_full_kernel<NS, double>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, x, y);
    else
        hipLaunchKernelGGL((hv_full_kernel<NS, float>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, x, y);
    return hipGetLastError();
}

// Two rows per thread pays for the step-table kernel in FP32 on large
// operators (four states, 22M rows: 36.7 -> 29.7 ms per H*v); in FP64 (55.6 ->
// 62.2 ms) and below a few million rows (three states, 0.46M rows: 53.8 ->
// 57.4 us) the one-row kernel is faster.
constexpr int kTwoRowMinRows = 1 << 22;

template <int NS>
static hipError_t hv_iter_ns(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    const size_t lds = hv_lds_bytes(op, prec);
    if constexpr (NS <= kShapedMaxStates) {
        // FP64 runs shaped when the caller keeps the interleaved copy
        // one row per thread: the unrolled terms give the loads enough independence
        // (four states, 22M rows: FP32 17.1 ms against 17.8 ms with two rows; FP64
        // 40.4 against 46.8 ms)
        if (hv_shaped(op, prec) && (prec == 1 || st.v64i)) {
            const unsigned g = (unsigned)hv_blocks(op);
            if (hv_shaped_skip(op, prec)) {
                if (prec == 0)
                    hipLaunchKernelGGL((hv_shaped_iter_kernel<NS, F64I, double, 1, true>), dim3(g), dim3(kBlock), lds,
                                       s, op, st);
                else
                    hipLaunchKernelGGL((hv_shaped_iter_kernel<NS, float, float, 1, true>), dim3(g), dim3(kBlock), lds,
                                       s, op, st);
                return hipGetLastError();
            }
            const bool split = hv_split_iter(op, prec, st);
            if (split && prec == 0)
                hipLaunchKernelGGL((hv_split_iter_kernel<NS, F64I, double, kSplitWaves>), dim3(hv_split_blocks(op)),
                                   dim3(64 * kSplitWaves), lds, s, op, st);
            else if (split)
                hipLaunchKernelGGL((hv_split_iter_kernel<NS, float, float, kSplitWaves>), dim3(hv_split_blocks(op)),
                                   dim3(64 * kSplitWaves), lds, s, op, st);
            else if (prec == 0)
                hipLaunchKernelGGL((hv_shaped_iter_kernel<NS, F64I, double, 1, false>), dim3(g), dim3(kBlock), lds,
                                   s, op, st);
            else
                hipLaunchKernelGGL((hv_shaped_iter_kernel<NS, float, float, 1, false>), dim3(g), dim3(kBlock), lds,
                                   s, op, st);
            return hipGetLastError();
        }
    }
    if (prec != 0 && op.D >= kTwoRowMinRows) {
        const unsigned g = (unsigned)((hv_blocks(op) + 1) / 2);
        if (prec == 1)
            hipLaunchKernelGGL((hv_iter2_kernel<NS, float, float>), dim3(g), dim3(kBlock), lds, s, op, st);
        else
            hipLaunchKernelGGL((hv_iter2_kernel<NS, __hip_bfloat16, float>), dim3(g), dim3(kBlock), lds, s, op, st);
        return hipGetLastError();
    }
    if (prec == 0)
        hipLaunchKernelGGL((hv_iter_kernel<NS, double, double>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    else if (prec == 1)
        hipLaunchKernelGGL((hv_iter_kernel<NS, float, float>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    else
        hipLaunchKernelGGL((hv_iter_kernel<NS, __hip_bfloat16, float>), dim3(hv_blocks(op)), dim3(kBlock), lds, s,
                           op, st);
    return hipGetLastError();
}

// ---- two-pass H*v launchers ----
static size_t hv2_pass1_lds(const NvOpDev &op, int prec);

bool hv2_use(const NvOpDev &op, int prec) {
    if (!op.tshape || !op.hv2.on || (prec != 0 && prec != 1) || (prec == 1 && !op.hv2.f32)) return false;
    const int64_t el = (int64_t)nv_lo_stride(op.ns) * (prec == 0 ? 8 : 4);
    return (int64_t)op.D * el >= op.hv2_min_bytes && ((int64_t)op.D + 2 * kBlock) * el < ((int64_t)1 << 31) &&
           hv2_pass1_lds(op, prec) <= 64 * 1024;
}

size_t hv2_scratch_bytes(const NvOpDev &op, int prec) {
    return (size_t)NV_HV2_NG * op.D * nv_lo_stride(op.ns) * (prec == 0 ? 8 : 4);
}

// Consecutive plane rows per thread of the second pass.
constexpr int kHv2Rows = 4;

int hv2_parts(const NvOpDev &op) {
    const int per = op.hv2.c * kHv2Rows;
    return (op.hv2.dr + per - 1) / per;
}

// The FP32 path keeps the coupling products on the matrix cores up to four states.
static bool hv2_mfma(const NvOpDev &op, int prec) { return prec == 1 && op.ns <= 4 && op.hv2.mfma; }

static size_t hv2_pass1_lds(const NvOpDev &op, int prec) {
    return hv_lds_bytes(op, prec) + (hv2_mfma(op, prec) ? (size_t)op.nterms * 16 * sizeof(float) : 0);
}

template <int NS>
static hipError_t hv2_ns(const NvOpDev &op, int prec, const void *xin, void *Z, const LzState *st,
                         const double *xfull, double *yfull, hipStream_t s) {
    if constexpr (NS > 4) {
        return hipErrorInvalidValue;  // the tables are built for at most four states
    } else {
    const unsigned g1 = (unsigned)hv_blocks(op);
    const size_t l1 = hv2_pass1_lds(op, prec);
    // plain form in FP32 (18.1 against 19.2 ms), skip form in FP64 (37.9 against 40.3 ms)
    const bool skip = op.hv2.skip < 0 ? prec == 0 : op.hv2.skip != 0;
    if (prec == 1) {
        if (hv2_mfma(op, prec)) {
            if (skip)
                hipLaunchKernelGGL((hv2_pass1_kernel<NS, float, float, true, true>), dim3(g1), dim3(kBlock), l1, s,
                                   op, xin, (float *)Z);
            else
                hipLaunchKernelGGL((hv2_pass1_kernel<NS, float, float, true, false>), dim3(g1), dim3(kBlock), l1, s,
                                   op, xin, (float *)Z);
        } else {
            if (skip)
                hipLaunchKernelGGL((hv2_pass1_kernel<NS, float, float, false, true>), dim3(g1), dim3(kBlock), l1, s,
                                   op, xin, (float *)Z);
            else
                hipLaunchKernelGGL((hv2_pass1_kernel<NS, float, float, false, false>), dim3(g1), dim3(kBlock), l1,
                                   s, op, xin, (float *)Z);
        }
    } else {
        if (skip)
            hipLaunchKernelGGL((hv2_pass1_kernel<NS, F64I, double, false, true>), dim3(g1), dim3(kBlock), l1, s, op,
                               xin, (double *)Z);
        else
            hipLaunchKernelGGL((hv2_pass1_kernel<NS, F64I, double, false, false>), dim3(g1), dim3(kBlock), l1, s,
                               op, xin, (double *)Z);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const unsigned g2 = (unsigned)hv2_parts(op);
    const unsigned b2 = (unsigned)(op.hv2.nl * op.hv2.c);
    const size_t l2 = (size_t)op.M * kBlock;
    const LzState none{};
    if (st) {
        if (prec == 1)
            hipLaunchKernelGGL((hv2_pass2_kernel<NS, float, float, true, kHv2Rows>), dim3(g2), dim3(b2), l2, s, op, *st, xin,
                               (const float *)Z, nullptr, nullptr);
        else
            hipLaunchKernelGGL((hv2_pass2_kernel<NS, F64I, double, true, kHv2Rows>), dim3(g2), dim3(b2), l2, s, op, *st, xin,
                               (const double *)Z, nullptr, nullptr);
    } else {
        if (prec == 1)
            hipLaunchKernelGGL((hv2_pass2_kernel<NS, float, float, false, kHv2Rows>), dim3(g2), dim3(b2), l2, s, op, none, xin,
                               (const float *)Z, xfull, yfull);
        else
            hipLaunchKernelGGL((hv2_pass2_kernel<NS, F64I, double, false, kHv2Rows>), dim3(g2), dim3(b2), l2, s, op, none, xin,
                               (const double *)Z, xfull, yfull);
    }
    return hipGetLastError();
    }
}

template <int NS>
static hipError_t step_ns(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    const size_t lds = op.offstate ? (size_t)op.M * kBlock : 0;
    if (prec == 0 && op.stream_nt)
        hipLaunchKernelGGL((lanczos_step_kernel<NS, double, true>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    else if (prec == 0)
        hipLaunchKernelGGL((lanczos_step_kernel<NS, double, false>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    else if (op.stream_nt)
        hipLaunchKernelGGL((lanczos_step_kernel<NS, float, true>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    else
        hipLaunchKernelGGL((lanczos_step_kernel<NS, float, false>), dim3(hv_blocks(op)), dim3(kBlock), lds, s, op, st);
    return hipGetLastError();
}

template <int NS>
static hipError_t diag_ns(const NvOpDev &op, double *dg, hipStream_t s) {
    hipLaunchKernelGGL((diag_precompute_kernel<NS>), dim3(hv_blocks(op)), dim3(kBlock), 0, s, op, dg);
    return hipGetLastError();
}

hipError_t launch_diag_precompute(const NvOpDev &op, double *dg, hipStream_t s) {
    NV_DISPATCH_NS(diag_ns, op, dg, s)
}

hipError_t launch_hv_full(const NvOpDev &op, int prec, const double *x, double *y, hipStream_t s) {
    NV_DISPATCH_NS(hv_full_ns, op, prec, x, y, s)
}

hipError_t launch_hv2_full(const NvOpDev &op, int prec, const double *x, const void *xin, void *Z, double *y,
                           hipStream_t s) {
    NV_DISPATCH_NS(hv2_ns, op, prec, xin, Z, nullptr, x, y, s)
}

// The iteration H*v runs in the fast-block form when the operator has its
// tables and the interleaved copy of q_i exists (FP32: LzState::vlo; FP64:
// LzState::v64i).
static bool fb_iter(const NvOpDev &op, int prec, const LzState &st) {
    return hv_fb_use(op, prec) && (prec == 1 ? st.vlo != nullptr : st.v64i != nullptr);
}

// The iteration H*v runs two-pass when the caller gave the channel scratch
// (LzState::z2) and, in FP64, the interleaved copy of q_i.
static bool hv2_iter(const NvOpDev &op, int prec, const LzState &st) {
    return st.z2 && hv2_use(op, prec) && (prec == 1 || st.v64i);
}

static hipError_t hv_iter_any(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    if (fb_iter(op, prec, st)) return launch_hv_fb_iter(op, prec, st, s);
    if (hv2_iter(op, prec, st)) {
        const void *xin = prec == 1 ? st.vlo : (const void *)st.v64i;
        NV_DISPATCH_NS(hv2_ns, op, prec, xin, st.z2, &st, nullptr, nullptr, s)
    }
    NV_DISPATCH_NS(hv_iter_ns, op, prec, st, s)
}

int hv_iter_parts(const NvOpDev &op, int prec, const LzState &st) {
    if (fb_iter(op, prec, st)) return hv_fb_parts(op);
    if (hv2_iter(op, prec, st)) return hv2_parts(op);
    return hv_split_iter(op, prec, st) ? (int)hv_split_blocks(op) : hv_blocks(op);
}

static hipError_t step_any(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    NV_DISPATCH_NS(step_ns, op, prec, st, s)
}

hipError_t launch_hv_iter_only(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    return hv_iter_any(op, prec, st, s);
}

hipError_t launch_hv_iter(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    hipError_t e = hv_iter_any(op, prec, st, s);
    if (e != hipSuccess) return e;
    return launch_finish_sum(st.partials, hv_iter_parts(op, prec, st), st.alpha, st.iter, 0, s);
}

hipError_t launch_lanczos_step_only(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    return step_any(op, prec, st, s);
}

hipError_t launch_lanczos_step(const NvOpDev &op, int prec, const LzState &st, hipStream_t s, int64_t *advance) {
    hipError_t e = step_any(op, prec, st, s);
    if (e != hipSuccess) return e;
    return launch_finish_sum(st.partials, hv_blocks(op), st.beta, st.iter, 1, s, advance);
}

template <int NS>
static hipError_t normalize_ns(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    const int g = grid_stride_blocks(op.D);
    const int64_t N = op.N, D = op.D;
    if (op.stream_nt) {
        if (prec == 0 || st.vlo == nullptr)
            hipLaunchKernelGGL((normalize_rows_kernel<NS, double, true>), dim3(g), dim3(kBlock), 0, s, N, D, st);
        else if (prec == 1)
            hipLaunchKernelGGL((normalize_rows_kernel<NS, float, true>), dim3(g), dim3(kBlock), 0, s, N, D, st);
        else
            hipLaunchKernelGGL((normalize_rows_kernel<NS, __hip_bfloat16, true>), dim3(g), dim3(kBlock), 0, s, N, D,
                               st);
    } else {
        if (prec == 0 || st.vlo == nullptr)
            hipLaunchKernelGGL((normalize_rows_kernel<NS, double, false>), dim3(g), dim3(kBlock), 0, s, N, D, st);
        else if (prec == 1)
            hipLaunchKernelGGL((normalize_rows_kernel<NS, float, false>), dim3(g), dim3(kBlock), 0, s, N, D, st);
        else
            hipLaunchKernelGGL((normalize_rows_kernel<NS, __hip_bfloat16, false>), dim3(g), dim3(kBlock), 0, s, N,
                               D, st);
    }
    return hipGetLastError();
}

hipError_t launch_normalize(const NvOpDev &op, int prec, const LzState &st, hipStream_t s) {
    NV_DISPATCH_NS(normalize_ns, op, prec, st, s)
}

// y[r * nsp + s] = (float)x[s * D + r] (the interleaved FP32 copy).
__global__ __launch_bounds__(kBlock) void cast_f32_kernel(const double *x, float *y, int64_t n, int64_t D, int nsp) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const int64_t s = i / D;
        y[(i - s * D) * nsp + s] = (float)x[i];
    }
}

// y[r * nsp + s] = x[s * D + r] (the interleaved FP64 copy).
__global__ __launch_bounds__(kBlock) void cast_f64i_kernel(const double *x, double *y, int64_t n, int64_t D, int nsp) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const int64_t s = i / D;
        y[(i - s * D) * nsp + s] = x[i];
    }
}

hipError_t launch_cast_f64i(const double *x, double *y, int64_t n, int64_t D, int ns, hipStream_t s) {
    hipLaunchKernelGGL(cast_f64i_kernel, dim3(grid_stride_blocks(n)), dim3(kBlock), 0, s, x, y, n, D,
                       nv_lo_stride(ns));
    return hipGetLastError();
}

hipError_t launch_cast_f32(const double *x, float *y, int64_t n, int64_t D, int ns, hipStream_t s) {
    hipLaunchKernelGGL(cast_f32_kernel, dim3(grid_stride_blocks(n)), dim3(kBlock), 0, s, x, y, n, D,
                       nv_lo_stride(ns));
    return hipGetLastError();
}

hipError_t launch_set_iter(int64_t *d_iter, int64_t value, int increment, hipStream_t s) {
    hipLaunchKernelGGL(set_iter_kernel, dim3(1), dim3(64), 0, s, d_iter, value, increment);
    return hipGetLastError();
}

hipError_t launch_fill_start(double *v, int64_t D, int ns, const double *vals_dev, hipStream_t s) {
    hipLaunchKernelGGL(fill_start_kernel, dim3(grid_stride_blocks(D * ns)), dim3(kBlock), 0, s, v, D, ns, vals_dev);
    return hipGetLastError();
}

hipError_t launch_norm_to(const double *v, int64_t n, double *out, double *partials, unsigned *counter,
                          hipStream_t s) {
    (void)counter;
    const int g = grid_stride_blocks(n);
    hipLaunchKernelGGL(norm_kernel, dim3(g), dim3(kBlock), 0, s, v, n, partials);
    return launch_finish_sum(partials, g, out, nullptr, 1, s);
}

// Overlaps of up to kMaxProbes probe vectors with basis vectors j0..j0+nj-1
// (q_j in slot j % nslots of V): grid (chunks, nj), partial dots per chunk in
// part[(k * chunks + chunk) * kMaxProbes + p], summed on the host.
__global__ __launch_bounds__(kBlock) void probe_dots_kernel(ProbeSet ps, const double *__restrict__ V, int64_t nslots,
                                                            int64_t N, int64_t j0, int64_t chunk,
                                                            double *__restrict__ part) {
    const int64_t k = blockIdx.y;
    const double *q = V + ((j0 + k) % nslots) * N;
    const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < N ? lo + chunk : N;
    double acc[kMaxProbes];
#pragma unroll
    for (int p = 0; p < kMaxProbes; ++p) acc[p] = 0.0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const double v = q[i];
#pragma unroll
        for (int p = 0; p < kMaxProbes; ++p)
            if (p < ps.np) acc[p] += v * ps.p[p][i];
    }
#pragma unroll
    for (int p = 0; p < kMaxProbes; ++p) {
        const double t = block_sum(acc[p]);
        if (threadIdx.x == 0) part[(k * gridDim.x + blockIdx.x) * kMaxProbes + p] = t;
    }
}

int probe_chunks(int64_t N) { return (int)std::min<int64_t>(64, (N + 65535) / 65536); }

hipError_t launch_probe_dots(const ProbeSet &ps, const double *V, int64_t nslots, int64_t N, int64_t j0, int64_t nj,
                             double *part, hipStream_t s) {
    const int nc = probe_chunks(N);
    const int64_t chunk = (N + nc - 1) / nc;
    hipLaunchKernelGGL(probe_dots_kernel, dim3(nc, (unsigned)nj), dim3(kBlock), 0, s, ps, V, nslots, N, j0, chunk,
                       part);
    return hipGetLastError();
}

// ------------------------------------------------------------------------
// Batched Lanczos: many operators of uneven size advance one iteration per
// launch sequence.  The rows of every problem are cut into tiles of
// blockDim.x rows; one workgroup per tile, so one launch covers the whole
// batch and the small problems cost no launches of their own.  Each tile
// reads its problem's operator tables and vector offsets.
// ------------------------------------------------------------------------
template <int NS, typename TIn, typename TAcc>
__device__ __forceinline__ void batch_hv_row(const NvOpDev &op, const TIn *x, const double *q, TAcc *y, int r,
                                             const uint8_t *dig, const TAcc *ftab, int tid, double &part) {
    TAcc acc[NS];
    offdiag_accumulate<NS, TIn, TAcc>(op, x, r, dig, ftab, tid, acc);
    double v[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r];
    diag_apply<NS>(op, r, dig, tid, v, dv);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        y[(size_t)s * op.D + r] = acc[s];
        part += v[s] * (dv[s] + (double)acc[s]);
    }
}

__global__ __launch_bounds__(kBlock) void batch_start_kernel(const BatchStart *pts, int64_t n, double *v) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) v[pts[i].at] = pts[i].value;
}

template <typename TIn>
__global__ __launch_bounds__(kBlock) void batch_normalize_kernel(BatchDev b) {
    const BatchTile tl = b.tiles[blockIdx.x];
    const NvOpDev &opg = b.ops[tl.prob];
    const int D = opg.D, ns = opg.ns;
    const int r = tl.row0 + threadIdx.x;
    if (r >= D) return;
    const int64_t it = *b.iter;
    double *q = b.V + slot_of(it, 3) * b.Ntot + b.voff[tl.prob];
    const double sc = 1.0 / b.beta[(int64_t)tl.prob * b.ld + it - 1];
    TIn *lo = b.vlo ? reinterpret_cast<TIn *>(b.vlo) + b.loff[tl.prob] : nullptr;
    const int nsp = nv_lo_stride(ns);
    for (int s = 0; s < ns; ++s) {
        const double v = q[(size_t)s * D + r] * sc;
        q[(size_t)s * D + r] = v;
        if (lo) lo[(size_t)r * nsp + s] = from_d<TIn>(v);
    }
}

template <int NS, typename TIn, typename TAcc>
__global__ __launch_bounds__(kBlock) void batch_hv_kernel(BatchDev b, int t0) {
    const int t = t0 + blockIdx.x;
    const BatchTile tl = b.tiles[t];
    const NvOpDev op = b.ops[tl.prob];
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int r = tl.row0 + tid;
    const bool live = r < op.D;
    const int64_t it = *b.iter;
    const double *q = b.V + slot_of(it, 3) * b.Ntot + b.voff[tl.prob];
    const TIn *x = b.vlo ? reinterpret_cast<const TIn *>(b.vlo) + b.loff[tl.prob] : reinterpret_cast<const TIn *>(q);
    TAcc *y = reinterpret_cast<TAcc *>(b.y) + b.voff[tl.prob];
    if (live) digits_energy(op, r, dig, tid);
    __syncthreads();
    double part = 0.0;
    if (live) batch_hv_row<NS, TIn, TAcc>(op, x, q, y, r, dig, ftab, tid, part);
    const double bs = block_sum(part);
    if (tid == 0) b.partials[t] = bs;
}

// batch_hv_kernel with two rows per thread: a workgroup of bs/2 threads
// covers the tile's bs rows as two halves.
template <int NS, typename TIn, typename TAcc>
__global__ __launch_bounds__(kBlock) void batch_hv2_kernel(BatchDev b, int t0) {
    const int t = t0 + blockIdx.x;
    const BatchTile tl = b.tiles[t];
    const NvOpDev op = b.ops[tl.prob];
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    uint8_t *dig1 = dig + op.M * kBlock;
    const int tid = threadIdx.x;
    const int half = b.bs / 2;
    const int r0 = tl.row0 + tid, r1 = r0 + half;
    const bool l0 = r0 < op.D, l1 = r1 < op.D;
    const int64_t it = *b.iter;
    const double *q = b.V + slot_of(it, 3) * b.Ntot + b.voff[tl.prob];
    const TIn *x = b.vlo ? reinterpret_cast<const TIn *>(b.vlo) + b.loff[tl.prob] : reinterpret_cast<const TIn *>(q);
    TAcc *y = reinterpret_cast<TAcc *>(b.y) + b.voff[tl.prob];
    if (l0) digits_energy(op, r0, dig, tid);
    else for (int k = 0; k < op.M; ++k) dig[k * kBlock + tid] = 0;
    if (l1) digits_energy(op, r1, dig1, tid);
    else for (int k = 0; k < op.M; ++k) dig1[k * kBlock + tid] = 0;
    __syncthreads();
    double part = 0.0;
    if (l0) {
        TAcc acc0[NS], acc1[NS];
        offdiag_accumulate2<NS, TIn, TAcc>(op, x, r0, r1, l0, l1, dig, dig1, ftab, tid, acc0, acc1);
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r0];
        diag_apply<NS>(op, r0, dig, tid, v, dv);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y[(size_t)s * op.D + r0] = acc0[s];
            part += v[s] * (dv[s] + (double)acc0[s]);
        }
        if (l1) {
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r1];
            diag_apply<NS>(op, r1, dig1, tid, v, dv);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                y[(size_t)s * op.D + r1] = acc1[s];
                part += v[s] * (dv[s] + (double)acc1[s]);
            }
        }
    }
    const double bs = block_sum(part);
    if (tid == 0) b.partials[t] = bs;
}

// batch_hv2_kernel / batch_hv_kernel over the shaped terms: R rows per
// thread (row k of a thread at row0 + k * blockDim.x + tid), for batches
// whose every operator has shaped terms.
template <int NS, typename TIn, typename TAcc, int R>
__global__ __launch_bounds__(kBlock) void batch_shaped_kernel(BatchDev b, int t0) {
    const int t = t0 + blockIdx.x;
    const BatchTile tl = b.tiles[t];
    const NvOpDev op = b.ops[tl.prob];
    uint8_t *dig;
    const TAcc *ftab = stage_tables<TAcc>(op, dig);
    const int tid = threadIdx.x;
    const int64_t it = *b.iter;
    const double *q = b.V + slot_of(it, 3) * b.Ntot + b.voff[tl.prob];
    const TIn *x = b.vlo ? reinterpret_cast<const TIn *>(b.vlo) + b.loff[tl.prob] : reinterpret_cast<const TIn *>(q);
    TAcc *y = reinterpret_cast<TAcc *>(b.y) + b.voff[tl.prob];
    int r[R];
    bool live[R];
    unsigned vo[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        r[k] = tl.row0 + k * (int)blockDim.x + tid;
        live[k] = r[k] < op.D;
        vo[k] = (unsigned)r[k] * XRes<NS, TIn>::kEl;
        uint8_t *dk = dig + k * op.M * kBlock;
        if (live[k]) digits_energy(op, r[k], dk, tid);
        else for (int m = 0; m < op.M; ++m) dk[m * kBlock + tid] = 0;
    }
    __syncthreads();
    const XRes<NS, TIn> xs(x, op.D);
    TAcc acc[R][NS];
    offdiag_shaped<NS, TIn, TAcc, R, false>(op, xs, vo, dig, ftab, tid, acc);
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        if (!live[k]) continue;
        double v[NS], dv[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r[k]];
        diag_apply<NS>(op, r[k], dig + k * op.M * kBlock, tid, v, dv);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            y[(size_t)s * op.D + r[k]] = acc[k][s];
            part += v[s] * (dv[s] + (double)acc[k][s]);
        }
    }
    const double bs = block_sum(part);
    if (tid == 0) b.partials[t] = bs;
}

template <int NS, typename TAcc>
__device__ __forceinline__ void batch_step_row(const NvOpDev &op, const double *q, const double *qm, double *res,
                                               const TAcc *y, double a, double bb, int64_t it, int r,
                                               const uint8_t *dig, int tid, double &part) {
    double v[NS], dv[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = q[(size_t)s * op.D + r];
    diag_apply<NS>(op, r, dig, tid, v, dv);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const size_t o = (size_t)s * op.D + r;
        double w = dv[s] + (double)y[o];
        w = w - a * v[s];
        if (it > 1) w = w - bb * qm[o];
        res[o] = w;
        part += w * w;
    }
}

template <int NS, typename TAcc>
__global__ __launch_bounds__(kBlock) void batch_step_kernel(BatchDev b, int t0) {
    extern __shared__ __align__(16) unsigned char dig[];
    const int t = t0 + blockIdx.x;
    const BatchTile tl = b.tiles[t];
    const NvOpDev op = b.ops[tl.prob];
    const int tid = threadIdx.x;
    const int r = tl.row0 + tid;
    const int64_t it = *b.iter;
    const int64_t off = b.voff[tl.prob];
    const double *q = b.V + slot_of(it, 3) * b.Ntot + off;
    const double *qm = b.V + slot_of(it - 1, 3) * b.Ntot + off;
    double *res = b.V + slot_of(it + 1, 3) * b.Ntot + off;
    const TAcc *y = reinterpret_cast<const TAcc *>(b.y) + off;
    const double a = b.alpha[(int64_t)tl.prob * b.ld + it];
    const double bb = it > 1 ? b.beta[(int64_t)tl.prob * b.ld + it - 1] : 0.0;
    double part = 0.0;
    if (r < op.D) {
        if (op.offstate) digits_energy(op, r, dig, tid);
        batch_step_row<NS, TAcc>(op, q, qm, res, y, a, bb, it, r, dig, tid, part);
    }
    const double bs = block_sum(part);
    if (tid == 0) b.partials[t] = bs;
}

// dst[p][it] = (sqrt of) the sum of problem p's tile partials, in tile order.
__global__ __launch_bounds__(256) void batch_finish_kernel(BatchDev b, double *dst, int take_sqrt) {
    const int p = blockIdx.x;
    const int t0 = b.tile0[2 * p], t1 = b.tile0[2 * p + 1];
    double s = 0.0;
    for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) s += b.partials[t];
    s = block_sum(s);
    if (threadIdx.x == 0) {
        const int64_t it = *b.iter;
        dst[(int64_t)p * b.ld + it] = take_sqrt ? sqrt(s) : s;
    }
}

hipError_t launch_batch_start(const BatchStart *pts, int64_t n, double *v, hipStream_t s) {
    hipLaunchKernelGGL(batch_start_kernel, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, pts, n, v);
    return hipGetLastError();
}

size_t batch_hv_lds(const NvOpDev &op, int prec) { return hv_lds_bytes(op, prec); }

hipError_t launch_batch_normalize(const BatchDev &b, int prec, hipStream_t s) {
    if (prec == 0 || b.vlo == nullptr)
        hipLaunchKernelGGL((batch_normalize_kernel<double>), dim3(b.T), dim3(b.bs), 0, s, b);
    else
        hipLaunchKernelGGL((batch_normalize_kernel<float>), dim3(b.T), dim3(b.bs), 0, s, b);
    return hipGetLastError();
}

// The tuned form of the batched H*v: shaped or step-table kernels, and in FP32
// one or two rows per thread (two rows need workgroups of at least one wave).
template <int NS>
static void batch_hv_ns(const BatchDev &b, int prec, size_t lds, int t0, int nt, hipStream_t s) {
    const bool two = prec != 0 && b.rows == 2 && b.bs >= 128;
    if constexpr (NS <= kShapedMaxStates) {
        if (b.shaped[prec == 0 ? 0 : 1] && !b.steps) {
            if (prec == 0)
                hipLaunchKernelGGL((batch_shaped_kernel<NS, double, double, 1>), dim3(nt), dim3(b.bs), lds, s, b, t0);
            else if (b.rows == 4 && b.bs >= 256)
                hipLaunchKernelGGL((batch_shaped_kernel<NS, float, float, 4>), dim3(nt), dim3(b.bs / 4), lds, s, b,
                                   t0);
            else if (two)
                hipLaunchKernelGGL((batch_shaped_kernel<NS, float, float, 2>), dim3(nt), dim3(b.bs / 2), lds, s, b,
                                   t0);
            else
                hipLaunchKernelGGL((batch_shaped_kernel<NS, float, float, 1>), dim3(nt), dim3(b.bs), lds, s, b, t0);
            return;
        }
    }
    if (prec == 0)
        hipLaunchKernelGGL((batch_hv_kernel<NS, double, double>), dim3(nt), dim3(b.bs), lds, s, b, t0);
    else if (two)
        hipLaunchKernelGGL((batch_hv2_kernel<NS, float, float>), dim3(nt), dim3(b.bs / 2), lds, s, b, t0);
    else
        hipLaunchKernelGGL((batch_hv_kernel<NS, float, float>), dim3(nt), dim3(b.bs), lds, s, b, t0);
}

template <int NS>
static void batch_step_ns(const BatchDev &b, int prec, size_t lds, int t0, int nt, hipStream_t s) {
    if (prec == 0)
        hipLaunchKernelGGL((batch_step_kernel<NS, double>), dim3(nt), dim3(b.bs), lds, s, b, t0);
    else
        hipLaunchKernelGGL((batch_step_kernel<NS, float>), dim3(nt), dim3(b.bs), lds, s, b, t0);
}

#define NV_BATCH_DISPATCH(fn, ns, ...)                                                                            \
    switch (ns) {                                                                                                 \
    case 1: fn<1>(__VA_ARGS__); break;                                                                            \
    case 2: fn<2>(__VA_ARGS__); break;                                                                            \
    case 3: fn<3>(__VA_ARGS__); break;                                                                            \
    case 4: fn<4>(__VA_ARGS__); break;                                                                            \
    case 5: fn<5>(__VA_ARGS__); break;                                                                            \
    case 6: fn<6>(__VA_ARGS__); break;                                                                            \
    case 7: fn<7>(__VA_ARGS__); break;                                                                            \
    case 8: fn<8>(__VA_ARGS__); break;                                                                            \
    case 9: fn<9>(__VA_ARGS__); break;                                                                            \
    case 10: fn<10>(__VA_ARGS__); break;                                                                          \
    default: return hipErrorInvalidValue;                                                                         \
    }

hipError_t launch_batch_hv(const BatchDev &b, const BatchGroup *groups, int ngroups, int prec, size_t lds,
                           hipStream_t s) {
    for (int g = 0; g < ngroups; ++g) {
        NV_BATCH_DISPATCH(batch_hv_ns, groups[g].ns, b, prec, lds, groups[g].t0, groups[g].nt, s)
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(batch_finish_kernel, dim3(b.P), dim3(256), 0, s, b, b.alpha, 0);
    return hipGetLastError();
}

hipError_t launch_batch_step(const BatchDev &b, const BatchGroup *groups, int ngroups, int prec, size_t lds,
                             hipStream_t s) {
    for (int g = 0; g < ngroups; ++g) {
        NV_BATCH_DISPATCH(batch_step_ns, groups[g].ns, b, prec, lds, groups[g].t0, groups[g].nt, s)
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(batch_finish_kernel, dim3(b.P), dim3(256), 0, s, b, b.beta, 1);
    return hipGetLastError();
}

}  // namespace nv
