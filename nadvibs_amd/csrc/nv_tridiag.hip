// Tridiagonal eigensolve (restates GIVENS, Source/yarkony.f90:91-543, for a
// tridiagonal input: the Householder stage and the back transformation are
// identities there).  The matrix arrives divided by its Frobenius norm.
//
// Everything here is a chain of n dependent steps per root, so the time is
// (steps) x (latency of a step); the kernels keep divisions, memory latency
// and control flow out of the chain.  MI355X, n = 2000 (before: the quotient
// form of the Sturm sequence over LDS, one row of the factors in flight, one
// thread for the clusters, a workgroup per column to normalise):
//   bisection          7.76 -> 0.59 ms, and 0.10 ms for the shared grid
//   inverse iteration  4.99 -> 1.20 ms
//   clusters           0.19 -> 0.005 ms
//   normalisation      0.20 -> 0.06 ms
// and a whole nv_ritz call with the envelope of its sticks 14.05 -> 2.14 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "nv_kernels.hpp"

namespace nv {

#define NV_EPS 1.1102230246251565e-16          /* 2^-53, determine_epsilon */
#define NV_HUGE 1.7976931348623157e308
#define NV_DEL1 (NV_EPS / 100.0)
#define NV_DELTA (NV_EPS * NV_EPS * 100.0)
#define NV_DELBIG (NV_HUGE * NV_DELTA / 1000.0)
#define NV_THETA1 (1000.0 / NV_HUGE)
#define NV_TOLER (NV_EPS * 100.0)

__device__ __forceinline__ double tri_block_sum(double v) {
    __shared__ double red[4];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// 1/d and a/d by Newton's iteration on the hardware estimate (two steps reach
// FP64; the quotient gets one residual correction).  Divisors too small for the
// estimate take the IEEE division.
__device__ __forceinline__ double tri_rcp(double d) {
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    return fma(fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ double tri_div(double a, double d) {
    const double m = fabs(d);
    if (m < 1e-280 || m > 1e280) return a / d;
    const double r = tri_rcp(d), q = a * r;
    return fma(fma(-d, q, a), r, q);
}

// Number of eigenvalues below x: sign changes of the leading principal minors
// of T - x, p_j = (d_j - x) p_{j-1} - e_{j-1}^2 p_{j-2}.  The quotients
// p_j / p_{j-1} are the pivots whose signs GIVENS counts
// (Source/yarkony.f90:360-389); the product form has one fma in the chain
// where the quotient has a division.  The minors are rescaled by a power of
// two every kSturm steps: |d - x| <= 2 and e^2 <= 1, so they grow by less than
// 2.5 a step.  A zero minor counts as a nonnegative pivot followed by a
// negative one, as there.  That does not hold where several rows are exactly
// decoupled (e^2 at its floor, kTriMinE2) and x is their common diagonal: the
// minors can then underflow to zero between two rescalings, and the sign
// changes after them are lost.  The search meets such an x only in the last
// ulps of that diagonal's own roots; on the CPU, 96,000 roots of matrices with
// repeated diagonals and zero couplings came within 1.7 * 2^-53 of the norm of
// a bisection in 113-bit arithmetic.  de is read with scalar loads, the next
// kSturm rows while these are used.
constexpr int kSturm = 8;
static_assert(kSturm <= kTriPad, "the prefetch reads kSturm rows past the matrix");

__device__ __forceinline__ void sturm_step(double d, double e2, double x, double &p1, double &p2, int &changes) {
    const double p = fma(d - x, p1, -(e2 * p2));
    changes += (int)((unsigned)(__double2hiint(p) ^ __double2hiint(p1)) >> 31);
    p2 = p1;
    p1 = p;
}

__device__ __forceinline__ int sturm_below(const double2 *__restrict__ de, int n, double x) {
    double p1 = 1.0, p2 = 0.0;
    int changes = 0;
    double2 cur[kSturm];
#pragma unroll
    for (int u = 0; u < kSturm; ++u) cur[u] = de[u];
    int j = 0;
    for (; j + kSturm <= n; j += kSturm) {
        double2 nxt[kSturm];
#pragma unroll
        for (int u = 0; u < kSturm; ++u) nxt[u] = de[j + kSturm + u];
#pragma unroll
        for (int u = 0; u < kSturm; ++u) sturm_step(cur[u].x, cur[u].y, x, p1, p2, changes);
        const int k = -__builtin_amdgcn_frexp_exp(fmax(fabs(p1), fabs(p2)));
        p1 = __builtin_amdgcn_ldexp(p1, k);
        p2 = __builtin_amdgcn_ldexp(p2, k);
#pragma unroll
        for (int u = 0; u < kSturm; ++u) cur[u] = nxt[u];
    }
#pragma unroll
    for (int u = 0; u < kSturm; ++u)
        if (j + u < n) sturm_step(cur[u].x, cur[u].y, x, p1, p2, changes);
    return changes;
}

// Sturm counts at the grid points every root's search starts from.
__device__ __forceinline__ double grid_point(int k, int K) { return -1.0 + 2.0 * ((double)(k + 1) / (double)(K + 1)); }

__global__ __launch_bounds__(64) void tri_grid_kernel(int n, const double2 *__restrict__ de, int K,
                                                      int32_t *__restrict__ cnt) {
    const int k = blockIdx.x * 64 + threadIdx.x;
    const int c = sturm_below(de, n, grid_point(k < K ? k : K - 1, K));
    if (k < K) cnt[k] = c;
}

// L lanes per root: multisection.  Each round takes Sturm counts at L interior
// points of [lo, hi] and keeps the sub-interval where the count reaches i + 1
// (count(lo) < i + 1 <= count(hi) throughout), so a round shrinks the interval
// (L + 1)-fold where bisection halves it.  When the points no longer fall
// strictly inside (a few ulps left) it bisects, and it stops at adjacent
// doubles; the root is hi, as in the bisection of GIVENS
// (Source/yarkony.f90:345-400).  The grid's counts replace the first rounds,
// which would be the same for every root.  The chain is bound by the issue of
// about seven FP64 instructions a step, so L falls as n grows to keep about
// one wave per SIMD.
template <int L>
__global__ __launch_bounds__(64) void tri_bisect_kernel(int n, const double2 *__restrict__ de, int K,
                                                        const int32_t *__restrict__ cnt, double *__restrict__ root) {
    constexpr int R = 64 / L;
    const int lane = threadIdx.x & (L - 1), grp = threadIdx.x / L;
    const int i = blockIdx.x * R + grp;
    const int want = (i < n ? i : n - 1) + 1;
    double lo = -1.0, hi = 1.0;
    if (K > 0) {
        int a = -1, b = K;  // count(a) < want <= count(b)
        while (b - a > 1) {
            const int m = (a + b) >> 1;
            if (cnt[m] >= want) b = m;
            else a = m;
        }
        if (a >= 0) lo = grid_point(a, K);
        if (b < K) hi = grid_point(b, K);
    }
    bool bis = false;
    for (int guard = 0; guard < 8192; ++guard) {
        const double mid = (lo + hi) * 0.5;
        const bool done = mid == lo || mid == hi;
        if (__all(done)) break;
        const double x = bis ? mid : lo + (hi - lo) * ((double)(lane + 1) / (double)(L + 1));
        const bool inside = x > lo && x < hi;
        const int c = sturm_below(de, n, x);
        const bool ge = inside ? c >= want : x >= hi;
        unsigned long long ball = __ballot(ge) >> (grp * L);
        if (L < 64) ball &= (1ull << (L & 63)) - 1;
        if (done) continue;
        if (bis) {
            if (ball & 1) hi = mid;
            else lo = mid;
            bis = false;
            continue;
        }
        const int k = ball ? __ffsll(ball) - 1 : L;  // first point at or above the root
        const double f = (hi - lo);
        const double xk = lo + f * ((double)(k + 1) / (double)(L + 1)), xl = lo + f * ((double)k / (double)(L + 1));
        const double new_hi = k < L ? xk : hi;
        const double new_lo = k == 0 ? lo : xl;
        if ((new_lo > lo && new_lo < new_hi) || new_hi < hi) {
            lo = new_lo > lo ? new_lo : lo;
            hi = new_hi;
        } else {
            bis = true;
        }
    }
    if (lane == 0 && i < n) root[i] = hi;
}

// Back substitution of one root through its pivoted factors, from v in place
// (Source/yarkony.f90:790-780).  Rows go in chunks of kBack: the next chunk's
// rows load while this one's are solved, and the pivots' reciprocals stay out
// of the chain, which is one fma and one product a row.  Rows whose value
// outgrows the reference's overflow guard (DELBIG) redo their chunk one by one
// with its rescaling.
constexpr int kBack = 16;

struct BackChunk {
    double u2[kBack], u3[kBack], u4[kBack], v[kBack];
};

__device__ __forceinline__ void back_load(BackChunk &c, int n, int i, int top, const double *__restrict__ U2,
                                          const double *__restrict__ U3, const double *__restrict__ U4,
                                          const double *v) {
#pragma unroll
    for (int k = 0; k < kBack; ++k) {
        const int l = top - k > 0 ? top - k : 0;
        const size_t o = (size_t)l * n + i;
        c.u2[k] = U2[o];
        c.u3[k] = U3[o];
        c.u4[k] = U4[o];
        c.v[k] = v[o];
    }
}

__device__ __forceinline__ double tri_pivot(double t) { return fabs(t) < NV_DELTA ? NV_DELTA : t; }

// Rows top .. max(top - kBack + 1, 0) of one root as the reference solves them.
__device__ __forceinline__ void back_rows_guarded(int n, int i, int top, const double *U2, const double *U3,
                                               const double *U4, double *v) {
    for (int l = top; l >= 0 && l > top - kBack; --l) {
        while (true) {
            const double v1 = l + 1 < n ? v[(size_t)(l + 1) * n + i] : 0.0;
            const double v2 = l + 2 < n ? v[(size_t)(l + 2) * n + i] : 0.0;
            const double e = v[(size_t)l * n + i] - v1 * U3[(size_t)l * n + i] - v2 * U4[(size_t)l * n + i];
            // a non-finite value cannot be rescaled and ends the sweep instead of looping
            if (fabs(e) > NV_DELBIG && isfinite(e)) {
                for (int k = 0; k < n; ++k) v[(size_t)k * n + i] /= NV_DELBIG;
                continue;
            }
            v[(size_t)l * n + i] = e / tri_pivot(U2[(size_t)l * n + i]);
            break;
        }
    }
}

__device__ __forceinline__ void tri_backsolve(int n, int i, const double *U2, const double *U3, const double *U4, double *v) {
    BackChunk cur, nxt;
    back_load(cur, n, i, n - 1, U2, U3, U4, v);
    double v1 = 0.0, v2 = 0.0;
    for (int top = n - 1; top >= 0; top -= kBack) {
        back_load(nxt, n, i, top - kBack, U2, U3, U4, v);
        double out[kBack];
        double a1 = v1, a2 = v2;
        bool big = false;
#pragma unroll
        for (int k = 0; k < kBack; ++k) {
            const double e = fma(-a1, cur.u3[k], fma(-a2, cur.u4[k], cur.v[k]));
            big = big || (top - k >= 0 && !(fabs(e) <= NV_DELBIG));
            out[k] = e * tri_rcp(tri_pivot(cur.u2[k]));
            a2 = a1;
            a1 = out[k];
        }
        if (!big) {
#pragma unroll
            for (int k = 0; k < kBack; ++k)
                if (top - k >= 0) v[(size_t)(top - k) * n + i] = out[k];
            v1 = a1;
            v2 = a2;
        } else {
            back_rows_guarded(n, i, top, U2, U3, U4, v);
            const int l = top - kBack + 1;
            if (l >= 0) {
                v1 = v[(size_t)l * n + i];
                v2 = l + 1 < n ? v[(size_t)(l + 1) * n + i] : 0.0;
            }
            // the rows ahead may have been rescaled
            back_load(nxt, n, i, top - kBack, U2, U3, U4, v);
        }
        cur = nxt;
    }
}

// Inverse iteration for root i: factor T - root (partial pivoting), start
// from ones (or the reference's multiplicative generator inside a cluster),
// back solve, forward sweep, back solve.  Vectors are stored component-major:
// vec[j*n + i], a lane per root, so a row of 64 roots is one 512-byte access.
__global__ __launch_bounds__(64) void tri_inverse_kernel(int n, const double *__restrict__ d,
                                                         const double *__restrict__ e,
                                                         const double *__restrict__ root,
                                                         const int32_t *__restrict__ ia,
                                                         const int64_t *__restrict__ rank, double *lu, double *vec) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= n) return;
    const size_t nn = (size_t)n * n;
    double *U2 = lu, *U3 = lu + nn, *U4 = lu + 2 * nn, *U5 = lu + 3 * nn;
    const double ar = root[i];
    const bool member = ia[i] != 0;
    // inside a cluster: x <- 4099 x mod 2^23 after n*rank[i] draws from 2^23-3
    constexpr uint32_t kMod = 1u << 23;
    uint32_t x = kMod - 3;
    if (member) {
        uint64_t k = (uint64_t)n * (uint64_t)rank[i];
        uint64_t p = 4099 % kMod, acc = 1;
        while (k) {
            if (k & 1) acc = (acc * p) % kMod;
            p = (p * p) % kMod;
            k >>= 1;
        }
        x = (uint32_t)((x * acc) % kMod);
    }
    auto start_value = [&]() {
        if (!member) return 1.0;
        x = (uint32_t)((4099ull * x) % kMod);
        return (double)x / (double)(kMod / 2) - 1.0;
    };
    double el1 = d[0] - ar;
    double el2 = n > 1 ? e[0] : 0.0;
    double first = 0.0;  // the pivot of row 0
#pragma unroll 4
    for (int j = 0; j + 1 < n; ++j) {
        const double bj = e[j], dj = d[j + 1] - ar;
        const double bj1 = j + 2 < n ? e[j + 1] : 0.0;
        const bool swap = fabs(el1) <= fabs(bj);
        // one division serves both branches
        const double den = swap ? bj : el1;
        double t = tri_div(swap ? el1 : bj, den);
        if (swap && !(fabs(bj) > NV_THETA1)) t = 1.0;
        const double u3 = swap ? dj : el2;
        const size_t o = (size_t)j * n + i;
        U2[o] = den;
        U3[o] = u3;
        U4[o] = (swap && j + 2 < n) ? bj1 : 0.0;
        U5[o] = t;
        vec[o] = start_value();
        if (j == 0) first = den;
        const double other = swap ? el2 : dj;
        el1 = other - t * u3;
        el2 = swap ? -t * bj1 : bj1;
    }
    {
        const size_t o = (size_t)(n - 1) * n + i;
        U2[o] = el1;
        U3[o] = 0.0;
        U4[o] = 0.0;
        vec[o] = start_value();
        if (n == 1) first = el1;
    }
    tri_backsolve(n, i, U2, U3, U4, vec);
    // forward sweep (Source/yarkony.f90:890-830); a swapped row uses the last
    // pivot of the back substitution as multiplier, as the reference does
    const double t1 = tri_pivot(first);
    double el = vec[i];
    double nv[kBack], nu2[kBack], nu5[kBack];
    auto fwd_load = [&](int j0) {
#pragma unroll
        for (int k = 0; k < kBack; ++k) {
            const int j = j0 + k + 1 < n ? j0 + k : (n > 1 ? n - 2 : 0);
            const size_t o = (size_t)j * n + i;
            nv[k] = vec[n > 1 ? o + n : o];
            nu2[k] = U2[o];
            nu5[k] = U5[o];
        }
    };
    if (n > 1) fwd_load(0);
    for (int j0 = 0; j0 + 1 < n; j0 += kBack) {
        double cv[kBack], c2[kBack], c5[kBack];
#pragma unroll
        for (int k = 0; k < kBack; ++k) {
            cv[k] = nv[k];
            c2[k] = nu2[k];
            c5[k] = nu5[k];
        }
        fwd_load(j0 + kBack);
#pragma unroll
        for (int k = 0; k < kBack; ++k) {
            const int j = j0 + k;
            if (j + 1 < n) {
                const double nxt = cv[k];
                const bool swap = c2[k] == e[j];
                vec[(size_t)j * n + i] = swap ? nxt : el;
                el = swap ? el - nxt * t1 : nxt - el * c5[k];
            }
        }
    }
    vec[(size_t)(n - 1) * n + i] = el;
    tri_backsolve(n, i, U2, U3, U4, vec);
}

// Normalisation (Source/yarkony.f90:900-920): max |v|, sum of (v/max)^2,
// scale, flush components below eps/100 to zero.  Kc columns per workgroup
// for the roots that stand alone: a row of Kc roots is one 64-byte access,
// where a workgroup per column touches 64 bytes for each 8 (n = 2000: 197 us).
constexpr int kNormCols = 8;
constexpr int kNormRows = 256 / kNormCols;

__device__ __forceinline__ bool in_cluster(int n, int i, const int32_t *ia) {
    return ia[i] != 0 || (i + 1 < n && ia[i + 1] > 0);
}

__global__ __launch_bounds__(256) void tri_norm_kernel(int n, const int32_t *__restrict__ ia, double *__restrict__ vec) {
    __shared__ double red[kNormRows][kNormCols];
    const int c = threadIdx.x % kNormCols, r = threadIdx.x / kNormCols;
    const int i = blockIdx.x * kNormCols + c;
    const bool on = i < n && !in_cluster(n, i, ia);
    double mx = 0.0;
    if (on)
#pragma unroll 8
        for (int j = r; j < n; j += kNormRows) mx = fmax(mx, fabs(vec[(size_t)j * n + i]));
    red[r][c] = mx;
    __syncthreads();
    for (int k = 0; k < kNormRows; ++k) mx = fmax(mx, red[k][c]);
    __syncthreads();
    double s = 0.0;
    if (on)
#pragma unroll 8
        for (int j = r; j < n; j += kNormRows) {
            const double q = vec[(size_t)j * n + i] / mx;
            s += q * q;
        }
    red[r][c] = s;
    __syncthreads();
    s = 0.0;
    for (int k = 0; k < kNormRows; ++k) s += red[k][c];
    const double t = 1.0 / (sqrt(s) * mx);
    if (on)
#pragma unroll 8
        for (int j = r; j < n; j += kNormRows) {
            double v = vec[(size_t)j * n + i] * t;
            if (fabs(v) < NV_DEL1) v = 0.0;
            vec[(size_t)j * n + i] = v;
        }
}

__device__ void tri_normalize_block(int n, int i, double *vec) {
    __shared__ double red[16];
    double mx = 0.0;
    for (int j = threadIdx.x; j < n; j += blockDim.x) mx = fmax(fabs(vec[(size_t)j * n + i]), mx);
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) mx = fmax(mx, red[w]);
    double s = 0.0;
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const double q = vec[(size_t)j * n + i] / mx;
        s += q * q;
    }
    s = tri_block_sum(s);
    const double t = 1.0 / (sqrt(s) * mx);
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        double v = vec[(size_t)j * n + i] * t;
        if (fabs(v) < NV_DEL1) v = 0.0;
        vec[(size_t)j * n + i] = v;
    }
    __syncthreads();
}

// Gram-Schmidt inside clusters of near-equal roots (Source/yarkony.f90:800-870)
// and normalisation: the workgroup of a cluster's first root walks its members
// in order.
__global__ __launch_bounds__(256) void tri_finish_kernel(int n, const int32_t *ia, double *vec) {
    const int i = blockIdx.x;
    if (ia[i] != 0 || !in_cluster(n, i, ia)) return;
    tri_normalize_block(n, i, vec);
    for (int m = i + 1; m < n && ia[m] > 0; ++m) {
        for (int j1 = 1; j1 <= ia[m]; ++j1) {
            const int k = m - j1;
            double t = 0.0;
            for (int j = threadIdx.x; j < n; j += blockDim.x) t += vec[(size_t)j * n + m] * vec[(size_t)j * n + k];
            t = tri_block_sum(t);
            for (int j = threadIdx.x; j < n; j += blockDim.x) vec[(size_t)j * n + m] -= t * vec[(size_t)j * n + k];
            __syncthreads();
        }
        tri_normalize_block(n, m, vec);
    }
}

// ia[i]: position of root i in its cluster (neighbours closer than TOLER);
// rank[i]: cluster members before it.  A cluster starts at a break, so ia is
// the distance to the last break and rank the non-breaks before i: two scans
// in one workgroup, a contiguous run of roots per thread.
__global__ __launch_bounds__(1024) void tri_cluster_kernel(int n, const double *__restrict__ root,
                                                           int32_t *__restrict__ ia, int64_t *__restrict__ rank) {
    __shared__ int last[1024], brk[1024];
    const int t = threadIdx.x;
    const int per = (n + 1023) / 1024;
    const int i0 = t * per < n ? t * per : n, i1 = i0 + per < n ? i0 + per : n;
    auto is_break = [&](int i) { return i == 0 || !(fabs(root[i - 1] - root[i]) < NV_TOLER); };
    int l = -1, b = 0;
    for (int i = i0; i < i1; ++i)
        if (is_break(i)) {
            l = i;
            ++b;
        }
    last[t] = l;
    brk[t] = b;
    for (int off = 1; off < 1024; off <<= 1) {
        __syncthreads();
        const int lp = t >= off ? last[t - off] : -1, bp = t >= off ? brk[t - off] : 0;
        __syncthreads();
        last[t] = last[t] > lp ? last[t] : lp;
        brk[t] += bp;
    }
    __syncthreads();
    l = t > 0 ? last[t - 1] : -1;
    b = t > 0 ? brk[t - 1] : 0;
    for (int i = i0; i < i1; ++i) {
        rank[i] = i - b;
        if (is_break(i)) {
            l = i;
            ++b;
        }
        ia[i] = i - l;
    }
}

// The grid's counts cost one chain of n steps, which stands for log(K) / log(L + 1)
// rounds of every root's search; below 256 rows a chain is shorter than a launch.
int tri_grid_points(int64_t n) { return n >= 256 ? 16384 : 0; }

hipError_t launch_tridiag(int64_t n64, const TriWork &w, hipStream_t s) {
    const int n = (int)n64;
    const double2 *de = reinterpret_cast<const double2 *>(w.de);
    const int K = tri_grid_points(n);
    if (K) hipLaunchKernelGGL(tri_grid_kernel, dim3((unsigned)(K / 64)), dim3(64), 0, s, n, de, K, w.cnt);
    // about one wave per SIMD (256 CUs of four)
    if (n <= 1024)
        hipLaunchKernelGGL(tri_bisect_kernel<64>, dim3((unsigned)n), dim3(64), 0, s, n, de, K, w.cnt, w.root);
    else if (n <= 2048)
        hipLaunchKernelGGL(tri_bisect_kernel<32>, dim3((unsigned)((n + 1) / 2)), dim3(64), 0, s, n, de, K, w.cnt,
                           w.root);
    else
        hipLaunchKernelGGL(tri_bisect_kernel<16>, dim3((unsigned)((n + 3) / 4)), dim3(64), 0, s, n, de, K, w.cnt,
                           w.root);
    hipLaunchKernelGGL(tri_cluster_kernel, dim3(1), dim3(1024), 0, s, n, w.root, w.ia, w.rank);
    hipLaunchKernelGGL(tri_inverse_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, n, w.d, w.e, w.root, w.ia,
                       w.rank, w.lu, w.vec);
    hipLaunchKernelGGL(tri_norm_kernel, dim3((unsigned)((n + kNormCols - 1) / kNormCols)), dim3(256), 0, s, n, w.ia,
                       w.vec);
    hipLaunchKernelGGL(tri_finish_kernel, dim3((unsigned)n), dim3(256), 0, s, n, w.ia, w.vec);
    return hipGetLastError();
}

}  // namespace nv
