// Bilinear forms of the Krylov gradient and the projected vectors, on the
// FP64 matrix cores.
//
// The gradient needs G_t[a][c] = sum_r u_a[r] (P_t v_c)[r] for every monomial
// P_t of order <= 2, over many pairs (u, v).  Position operators of different
// modes commute and are symmetric, so with U_0 = u, U_k = q_k u (and V_l alike)
//   q_l          -> U_0 . V_l
//   q_k q_l      -> U_k . V_l            (k < l)
//   q_k^2        -> U_k . V_k  and a diagonal rest: the truncated product q_k q_k
//                   is q_k^2 less nf/2 on the last function, since <n|q q|n> =
//                   n/2 + (n + 1)/2 with the second half missing there.  So the
//                   part of q_k^2 off the diagonal is U_k . V_k - sum w_k u v with
//                   w_k = n_k + 1/2 less nf_k/2 on the last function.
// One product of a ((M + 1) ns) x rows block with a rows x ((M + 1) ns) block
// gives every form at once, and a second small one the sums weighted with
// n_k + 1/2, with the last function and with 1.  A row then needs 2 M + 1
// neighbours of u and of v, where the term-by-term kernel reads every step of
// every term through L2 again (27 terms of a six-mode operator: 1.2 GB a pair
// of vectors, 176 us for 460,800 rows of three states and 22 us for its sums;
// here 41 us).  What is left is bound by the issue of the wave that forms the
// columns: matrix products 13 us, loads 20 us of the 41.  Loads of the next chunk
// in flight during the products need 270 registers, one wave per SIMD: 82 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "nv_kernels.hpp"

namespace nv {

typedef double nv_d4 __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4: lane l gives A[l % 16][l / 16] and B[l / 16][l % 16] and
// holds D[l / 16 + 4 v][l % 16] in register v.
__device__ __forceinline__ nv_d4 mfma16(double a, double b, nv_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Rows of a chunk: lanes 0..31 of a wave form the U block of 32 rows, lanes
// 32..63 the V block of the same rows.
constexpr int kCRows = 32;
constexpr int kCLd = kCRows + 4;  // row stride in LDS: 16 columns at 8 words apart take every bank once

// The columns of one tile: kMpt whole modes (mode-major, ns states each), so
// that the pairs k <= l fill the upper triangle of tiles.
__host__ __device__ constexpr int modes_per_tile(int ns) { return 16 / ns; }

// The digits of a row come from FP64 reciprocals: (rest + 1/2) / nf is at least
// 1/(2 nf) from an integer, far more than the rounding, and a 32-bit integer
// division costs some thirty instructions.
__device__ __forceinline__ int next_digit(int &rest, int nf, double inv) {
    const int d = (int)((rest + 0.5) * inv);
    const int n = rest - d * nf;
    rest = d;
    return n;
}

// All loads of a row leave before any is used; MM bounds the modes (it sizes the
// registers).  A neighbour outside the basis repeats the row itself, at factor 0.
template <int NS, int TU, int NW, int MM>
__global__ __launch_bounds__(256) void bilinear_kernel(GradModes g, const double *__restrict__ ub, int64_t ldu,
                                                      const double *__restrict__ vb, int64_t ldv, int64_t vslot0,
                                                      int64_t vslots, int m, double *__restrict__ part) {
    constexpr int MPT = modes_per_tile(NS);
    constexpr int NT = TU * (TU + 1) / 2;
    __shared__ double tab[4][2][TU * 16][kCLd];
    __shared__ uint8_t dig[4][16][kCRows];
    __shared__ double sq[256];  // <n|q|n+1>
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < 256; i += 256) sq[i] = sqrt((i + 1) / 2.0);
    for (int i = tid; i < 4 * 2 * TU * 16 * kCLd; i += 256) (&tab[0][0][0][0])[i] = 0.0;
    for (int i = tid; i < 4 * 16 * kCRows; i += 256) (&dig[0][0][0])[i] = 0;
    __syncthreads();
    const int side = lane >> 5, rr = lane & 31;
    const int i16 = lane & 15, k4 = lane >> 4;
    nv_d4 acc[NT], wacc[NW];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = nv_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NW; ++t) wacc[t] = nv_d4{0.0, 0.0, 0.0, 0.0};
    const int D = g.D;
    // this lane's weight rows: mode, last function (rows M..2M-1, else -1), 1 for the row of
    // ones and -1 past it
    int wk[NW], wlast[NW], wkind[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t) {
        const int w = t * 16 + i16;
        wk[t] = w < g.M ? w : (w < 2 * g.M ? w - g.M : 0);
        wlast[t] = w >= g.M && w < 2 * g.M ? g.nf[wk[t]] - 1 : -1;
        wkind[t] = w < 2 * g.M ? 0 : (w == 2 * g.M ? 1 : -1);
    }
    const int chunks = (D + kCRows - 1) / kCRows;
    // XCD x takes one contiguous range of rows, so the neighbours along the slow modes stay in its L2
    const int nb = gridDim.x, b = blockIdx.x, x = b & 7, q8 = nb >> 3, rem = nb & 7;
    const int bb = x * q8 + (x < rem ? x : rem) + (b >> 3);
    const int c0 = (int)((int64_t)chunks * bb / nb) + wave, c1 = (int)((int64_t)chunks * (bb + 1) / nb);
    auto vector_of = [&](int j) {
        return side ? vb + ((vslot0 + j) % vslots) * ldv : ub + (int64_t)j * ldu;
    };
    for (int j = blockIdx.y; j < m; j += gridDim.y) {
        const double *src = vector_of(j);
        for (int c = c0; c < c1; c += 4) {
            const int r = c * kCRows + rr;
            const bool live = r < D;
            const int rs = live ? r : 0;
            double own[NS], up[MM][NS], dn[MM][NS], fu[MM], fd[MM];
            int rest = rs;
#pragma unroll
            for (int a = 0; a < NS; ++a) own[a] = src[(int64_t)a * D + rs];
#pragma unroll
            for (int q = 0; q < MM; ++q) {
                const int k = g.M - 1 - q;
                if (k >= 0) {
                    const int nf = g.nf[k], sh = g.shft[k];
                    const int n = next_digit(rest, nf, g.inv[k]);
                    const bool hu = n + 1 < nf, hd = n > 0;
                    const int ru = hu ? rs + sh : rs, rd = hd ? rs - sh : rs;
#pragma unroll
                    for (int a = 0; a < NS; ++a) {
                        up[q][a] = src[(int64_t)a * D + ru];
                        dn[q][a] = src[(int64_t)a * D + rd];
                    }
                    fu[q] = live && hu ? sq[n] : 0.0;
                    fd[q] = live && hd ? sq[n - 1] : 0.0;
                    if (side == 0) dig[wave][k][rr] = (uint8_t)n;
                }
            }
            // this row's columns: u, then q_k u for every mode
#pragma unroll
            for (int a = 0; a < NS; ++a) tab[wave][side][a][rr] = live ? own[a] : 0.0;
#pragma unroll
            for (int q = 0; q < MM; ++q) {
                const int k = g.M - 1 - q;
                if (k >= 0) {
                    const int col = ((k + 1) / MPT) * 16 + ((k + 1) % MPT) * NS;
#pragma unroll
                    for (int a = 0; a < NS; ++a)
                        tab[wave][side][col + a][rr] = fma(fu[q], up[q][a], fd[q] * dn[q][a]);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll 2
            for (int s = 0; s < kCRows / 4; ++s) {
                const int row = 4 * s + k4;
                double av[TU], bv[TU];
#pragma unroll
                for (int t = 0; t < TU; ++t) {
                    av[t] = tab[wave][0][t * 16 + i16][row];
                    bv[t] = tab[wave][1][t * 16 + i16][row];
                }
                int at = 0;
#pragma unroll
                for (int t = 0; t < TU; ++t)
#pragma unroll
                    for (int t2 = t; t2 < TU; ++t2) {
                        acc[at] = mfma16(av[t], bv[t2], acc[at]);
                        ++at;
                    }
                // weights x (u_a v_c): n_k + 1/2, then the last function's nf/2, then 1
                const int a = i16 / NS, cc = i16 % NS;
                const double uv = i16 < NS * NS ? tab[wave][0][a < NS ? a : 0][row] * tab[wave][1][cc][row] : 0.0;
#pragma unroll
                for (int t = 0; t < NW; ++t) {
                    const int n = dig[wave][wk[t]][row];
                    double wt = n + 0.5;
                    if (wlast[t] >= 0) wt = n == wlast[t] ? 0.5 * (n + 1) : 0.0;
                    if (wkind[t] != 0) wt = wkind[t] > 0 ? 1.0 : 0.0;
                    wacc[t] = mfma16(wt, uv, wacc[t]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the four waves' sums through LDS (the columns are no longer needed), one
    // partial per workgroup and tile
    double *red = &tab[0][0][0][0];  // 4 x 256 doubles
    const int64_t wg = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
#pragma unroll
    for (int t = 0; t < NT + NW; ++t) {
        const nv_d4 v = t < NT ? acc[t < NT ? t : 0] : wacc[t < NT ? 0 : t - NT];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave * 256 + (k4 + 4 * e) * 16 + i16] = v[e];
        __syncthreads();
        part[(wg * (NT + NW) + t) * 256 + tid] = (red[tid] + red[256 + tid]) + (red[512 + tid] + red[768 + tid]);
    }
}

// acc[tile][256] += the partials of every workgroup, in order within four strided sums.
__global__ __launch_bounds__(1024) void bilinear_finish_kernel(int nwg, int nt, const double *__restrict__ part,
                                                               double *__restrict__ acc) {
    __shared__ double red[1024];
    const int e = threadIdx.x & 255, q = threadIdx.x >> 8, t = blockIdx.x;
    double s = 0.0;
#pragma unroll 8
    for (int w = q; w < nwg; w += 4) s += part[((int64_t)w * nt + t) * 256 + e];
    red[threadIdx.x] = s;
    __syncthreads();
    if (q == 0) acc[t * 256 + e] += (red[e] + red[256 + e]) + (red[512 + e] + red[768 + e]);
}

// Forms of order <= 2 over at most four states and fifteen modes whose columns
// fit three tiles (ns = 4: eleven modes, ns = 3: fourteen); the term-by-term
// kernel serves the rest.
static int bilinear_tu(int ns, int M) { return (M + 1 + modes_per_tile(ns) - 1) / modes_per_tile(ns); }
static int bilinear_nw(int M) { return (2 * M + 1 + 15) / 16; }

bool bilinear_ok(int ns, int M, int ordr) { return ordr <= 2 && ns <= 4 && M <= 15 && bilinear_tu(ns, M) <= 3; }

int bilinear_tiles(int ns, int M) {
    const int tu = bilinear_tu(ns, M);
    return tu * (tu + 1) / 2 + bilinear_nw(M);
}

int bilinear_index(int ns, int M, int k, int a, int l, int c) {
    const int mpt = modes_per_tile(ns), tu = bilinear_tu(ns, M);
    const int t = k / mpt, t2 = l / mpt;
    const int tile = t * tu - t * (t - 1) / 2 + (t2 - t);
    return tile * 256 + ((k % mpt) * ns + a) * 16 + (l % mpt) * ns + c;
}

int bilinear_weight_index(int ns, int M, int w, int a, int c) {
    const int tu = bilinear_tu(ns, M);
    return (tu * (tu + 1) / 2 + w / 16) * 256 + (w % 16) * 16 + a * ns + c;
}

// Two workgroups a CU when the rows and the pairs allow it; each takes a
// contiguous range of chunks of every gridDim.y-th pair.
static dim3 bilinear_grid(int64_t D, int m) {
    const int64_t chunks = (D + kCRows - 1) / kCRows;
    const int gx = (int)std::min<int64_t>(512, (chunks + 3) / 4);
    const int gy = (int)std::min<int64_t>(m, (512 + gx - 1) / gx);
    return dim3((unsigned)gx, (unsigned)gy);
}

size_t bilinear_part_bytes(int ns, int M, int64_t D, int m) {
    const dim3 g = bilinear_grid(D, m);
    return (size_t)g.x * g.y * bilinear_tiles(ns, M) * 256 * sizeof(double);
}

template <int NS, int TU, int NW, int MM>
static hipError_t bilinear_launch(const GradModes &g, const double *u, int64_t ldu, const double *v, int64_t ldv,
                                  int64_t slot0, int64_t nslots, int m, double *part, double *acc, hipStream_t s) {
    const dim3 grid = bilinear_grid(g.D, m);
    constexpr int nt = TU * (TU + 1) / 2 + NW;
    bilinear_kernel<NS, TU, NW, MM><<<grid, 256, 0, s>>>(g, u, ldu, v, ldv, slot0, nslots, m, part);
    bilinear_finish_kernel<<<nt, 1024, 0, s>>>((int)(grid.x * grid.y), nt, part, acc);
    return hipGetLastError();
}

template <int NS>
static hipError_t bilinear_ns(const GradModes &g, const double *u, int64_t ldu, const double *v, int64_t ldv,
                              int64_t slot0, int64_t nslots, int m, double *part, double *acc, hipStream_t s) {
    const int M = g.M;
    // modes MIN..MM: up to 7 fill one tile of weights, 11 and 15 take two
#define NV_T(TU, MIN, MM)                                                                                            \
    if constexpr (TU >= (MIN + NS_TILE) / NS_TILE && TU <= (MM + NS_TILE) / NS_TILE)                                 \
        if (tu == TU)                                                                                                \
            return bilinear_launch<NS, TU, (2 * MM + 16) / 16, MM>(g, u, ldu, v, ldv, slot0, nslots, m, part, acc, s);
#define NV_B(MIN, MM)             \
    if (M >= MIN && M <= MM) {    \
        NV_T(1, MIN, MM)          \
        NV_T(2, MIN, MM)          \
        NV_T(3, MIN, MM)          \
    }
    constexpr int NS_TILE = modes_per_tile(NS);
    const int tu = bilinear_tu(NS, M);
    NV_B(1, 4) NV_B(5, 7) NV_B(8, 11) NV_B(12, 15)
#undef NV_B
#undef NV_T
    return hipErrorInvalidValue;
}

hipError_t launch_bilinear(const GradModes &g, int ns, const double *u, int64_t ldu, const double *v, int64_t ldv,
                           int64_t slot0, int64_t nslots, int m, double *part, double *acc, hipStream_t s) {
    switch (ns) {
        case 1: return bilinear_ns<1>(g, u, ldu, v, ldv, slot0, nslots, m, part, acc, s);
        case 2: return bilinear_ns<2>(g, u, ldu, v, ldv, slot0, nslots, m, part, acc, s);
        case 3: return bilinear_ns<3>(g, u, ldu, v, ldv, slot0, nslots, m, part, acc, s);
        case 4: return bilinear_ns<4>(g, u, ldu, v, ldv, slot0, nslots, m, part, acc, s);
        default: return hipErrorInvalidValue;
    }
}

// ---- Y = V S ----------------------------------------------------------------
// Y[c0+c][r] = sum_k S(k, c0+c) V_k[r], k = 0..n-1.  V_k at V + ((slot0 + k) %
// nslots) * N (the basis or a circular segment buffer); S component-major with
// row stride ldv, vec[k*ldv + i] = component k of root i.
//
// A product of n x nc by N x n: FP64 on the matrix cores, kRitzChunk outputs per
// pass over the basis.  A wave holds kRitzChunk x 32 outputs (128 accumulator
// registers) and walks the basis four vectors at a time; S comes from LDS,
// staged kRitzKB vectors at a time, and the loads of the next four vectors are
// in flight during the products of these.  The vector form (16 outputs per pass,
// one element per thread) read the basis four times as often: 120 vectors of 1.38M
// elements into 120 outputs 3.2 -> 1.05 ms.
// T tiles of 16 outputs (fewer than four when fewer are left).
template <int T>
__global__ __launch_bounds__(256) void ritz_vectors_kernel(const double *__restrict__ V, int64_t N, int n,
                                                          const double *__restrict__ vec, int64_t ldv, int64_t c0,
                                                          int nc, int64_t slot0, int64_t nslots,
                                                          double *__restrict__ Y) {
    // rows 16 doubles apart in the banks: the four rows of a read take each bank twice
    __shared__ double s[kRitzKB][T * 16 + 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i16 = lane & 15, k4 = lane >> 4;
    const int64_t r0 = ((int64_t)blockIdx.x * 4 + wave) * 32 + i16, r1 = r0 + 16;
    // rows past the end repeat the last one; they are not written
    const int64_t ra = r0 < N ? r0 : N - 1, rb = r1 < N ? r1 : N - 1;
    nv_d4 acc[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t][0] = acc[t][1] = nv_d4{0.0, 0.0, 0.0, 0.0};
    // vector k of this lane's four; past the last one its coefficient is zero
    auto at = [&](int k) { return V + ((slot0 + (k < n ? k : n - 1)) % nslots) * N; };
    double xa = at(k4)[ra], xb = at(k4)[rb];
    for (int k0 = 0; k0 < n; k0 += kRitzKB) {
        __syncthreads();
        for (int t = threadIdx.x; t < kRitzKB * T * 16; t += 256) {
            const int kk = t / (T * 16), cc = t % (T * 16);
            s[kk][cc] = (k0 + kk < n && cc < nc) ? vec[(int64_t)(k0 + kk) * ldv + c0 + cc] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < kRitzKB; kk += 4) {
            if (k0 + kk >= n) break;
            const double *p = at(k0 + kk + 4 + k4);
            const double na = p[ra], nb = p[rb];
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const double a = s[kk + k4][t * 16 + i16];
                acc[t][0] = mfma16(a, xa, acc[t][0]);
                acc[t][1] = mfma16(a, xb, acc[t][1]);
            }
            xa = na;
            xb = nb;
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = t * 16 + k4 + 4 * e;
            if (c >= nc) continue;
            if (r0 < N) Y[(c0 + c) * N + r0] = acc[t][0][e];
            if (r1 < N) Y[(c0 + c) * N + r1] = acc[t][1][e];
        }
}

hipError_t launch_ritz_vectors(const double *V, int64_t N, int64_t n, const double *vec, int64_t nroots, double *Y,
                               hipStream_t s) {
    return launch_ritz_vectors(V, N, n, vec, n, nroots, 0, n, Y, s);
}

hipError_t launch_ritz_vectors(const double *V, int64_t N, int64_t n, const double *vec, int64_t ldv, int64_t nroots,
                               int64_t slot0, int64_t nslots, double *Y, hipStream_t s) {
    if (n < 1 || n > INT32_MAX || nslots < n || slot0 < 0 || ldv < 1) return hipErrorInvalidValue;
    const unsigned nb = (unsigned)((N + 127) / 128);
    for (int64_t c0 = 0; c0 < nroots; c0 += kRitzChunk) {
        const int nc = (int)(nroots - c0 < kRitzChunk ? nroots - c0 : kRitzChunk);
        auto go = [&](auto kernel) {
            kernel<<<nb, 256, 0, s>>>(V, N, (int)n, vec, ldv, c0, nc, slot0 % nslots, nslots, Y);
        };
        if (nc > 48) go(ritz_vectors_kernel<4>);
        else if (nc > 32) go(ritz_vectors_kernel<3>);
        else if (nc > 16) go(ritz_vectors_kernel<2>);
        else go(ritz_vectors_kernel<1>);
    }
    return hipGetLastError();
}

}  // namespace nv
