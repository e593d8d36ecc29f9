// Device code shared by the H*v kernels (nv_kernels.hip, nv_fastblock.hip):
// the row order over the XCDs, block sums, element types, mode digits, the
// diagonal part, and the buffer loads of the interleaved vectors.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <type_traits>

#include "nv_kernels.hpp"

namespace nv {

// Workgroups of one launch go to the 8 XCDs round-robin (workgroup b to XCD
// b % 8).  H*v gathers x at +-stride of every mode, so a workgroup reads the
// rows of its neighbours along the slow modes; mapping each XCD onto one
// contiguous range of rows keeps that window inside the XCD's own L2.
__device__ __forceinline__ int xcd_block(int b, int g) {
    const int x = b & 7, j = b >> 3, q = g >> 3, rem = g & 7;
    return x * q + (x < rem ? x : rem) + j;
}

// ------------------------------------------------------------------------
// reductions
// ------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Block-wide sum; every thread gets the result.  blockDim.x <= 1024.
static __device__ __forceinline__ double block_sum(double v) {
    __shared__ double red[16];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    const int nw = (blockDim.x + 63) >> 6;
    double t = 0.0;
    for (int i = 0; i < nw; ++i) t += red[i];
    return t;
}

// ------------------------------------------------------------------------
// element types
// ------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ float to_f(T v);
template <> __device__ __forceinline__ float to_f<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f<__hip_bfloat16>(__hip_bfloat16 v) { return __bfloat162float(v); }

template <typename TIn, typename TAcc> __device__ __forceinline__ TAcc load_acc(const TIn *p);
template <> __device__ __forceinline__ double load_acc<double, double>(const double *p) { return *p; }
template <> __device__ __forceinline__ float load_acc<float, float>(const float *p) { return *p; }
template <> __device__ __forceinline__ float load_acc<__hip_bfloat16, float>(const __hip_bfloat16 *p) {
    return __bfloat162float(*p);
}
template <> __device__ __forceinline__ float load_acc<double, float>(const double *p) { return (float)*p; }

template <typename T> __device__ __forceinline__ T from_d(double v);
template <> __device__ __forceinline__ double from_d<double>(double v) { return v; }
template <> __device__ __forceinline__ float from_d<float>(double v) { return (float)v; }
template <> __device__ __forceinline__ __hip_bfloat16 from_d<__hip_bfloat16>(double v) {
    return __float2bfloat16((float)v);
}

template <typename T> __device__ __forceinline__ const T *ftab_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *ftab_of<double>(const NvOpDev &op) { return op.ftab64; }
template <> __device__ __forceinline__ const float *ftab_of<float>(const NvOpDev &op) { return op.ftab32; }
template <typename T> __device__ __forceinline__ const T *cmat_of(const NvOpDev &op);
template <> __device__ __forceinline__ const double *cmat_of<double>(const NvOpDev &op) { return op.cmat64; }
template <> __device__ __forceinline__ const float *cmat_of<float>(const NvOpDev &op) { return op.cmat32; }

// ------------------------------------------------------------------------
// mode digits and the diagonal part
// ------------------------------------------------------------------------
// Writes the digits n_k of r into dig[k*kBlock + tid]; returns E(r).
__device__ __forceinline__ double digits_energy(const NvOpDev &op, int r, uint8_t *dig, int tid) {
    unsigned rr = (unsigned)r;
    double e = 0.0;
    for (int k = op.M - 1; k >= 0; --k) {
        const unsigned nf = (unsigned)op.nfunc[k];
        const unsigned q = rr / nf;
        const unsigned d = rr - q * nf;
        rr = q;
        dig[k * kBlock + tid] = (uint8_t)d;
        e += ((double)d + 0.5) * op.omega[k];
    }
    return e;
}

// The vibrationally diagonal part of H (Source/top.f90:712-756) splits into
// the state-diagonal E(n) + D_ss(n), precomputed once into op.dg, and the
// inter-state part D_ss'(n), s != s', evaluated per row when present.
template <int NS>
__device__ __forceinline__ void diag_offstate(const NvOpDev &op, const uint8_t *dig, int tid,
                                              const double (&v)[NS], double (&out)[NS]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        double a = 0.0;
#pragma unroll
        for (int s2 = 0; s2 < NS; ++s2)
            if (s2 != s) a += op.dconst[s * NS + s2] * v[s2];
        out[s] += a;
    }
    for (int t = 0; t < op.ndterms; ++t) {
        const NvDiagTerm dt = op.dterms[t];
        double h = 1.0;
#pragma unroll
        for (int j = 0; j < NV_MAXF; ++j)
            if (j < dt.nf) h *= op.ftab64[dt.code[j] * op.nmax + dig[dt.mode[j] * kBlock + tid]];
        const double *C = op.dcmat + (size_t)t * NS * NS;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double a = 0.0;
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2)
                if (s2 != s) a += C[s * NS + s2] * v[s2];
            out[s] += h * a;
        }
    }
}

// out[s] = sum_s' (E + D)(n)_{ss'} v[s'] in FP64.  dig is only read when
// states are coupled through D.
template <int NS>
__device__ __forceinline__ void diag_apply(const NvOpDev &op, int r, const uint8_t *dig, int tid,
                                           const double (&v)[NS], double (&out)[NS]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) out[s] = op.dg[(size_t)s * op.D + r] * v[s];
    if (op.offstate) diag_offstate<NS>(op, dig, tid, v, out);
}

// ------------------------------------------------------------------------
// neighbour rows through buffer resources
// ------------------------------------------------------------------------
typedef float nv_f2 __attribute__((ext_vector_type(2)));
typedef float nv_f3 __attribute__((ext_vector_type(3)));
typedef float nv_f4 __attribute__((ext_vector_type(4)));

// Word 3 of the buffer resource: data format 32 (bits 15-18 = 4); the
// run-time compiled kernels use the same value.
constexpr int kBufFlags = 0x00020000;

template <int NS, typename TIn> struct XRes;

// One interleaved row as loaded (P = nv_lo_stride values), held apart from its
// use so that a loop can keep loads of the next iteration in flight.
template <int P> struct FRow { nv_f4 v[P / 4]; };
template <> struct FRow<1> { float v; };
template <> struct FRow<2> { nv_f2 v; };
template <> struct FRow<3> { nv_f3 v; };

// interleaved FP32 copy, x[r * nv_lo_stride(NS) + s]: one load per row up to
// four states, 16-byte loads of the states present beyond
template <int NS> struct XRes<NS, float> {
    static constexpr unsigned kEl = nv_lo_stride(NS) * 4;
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ XRes(const float *x, int D)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, (int)((unsigned)D * kEl), kBufFlags)) {}
    template <typename TAcc>
    __device__ __forceinline__ void fma(unsigned o, TAcc h, TAcc (&w)[NS]) const { fma_so<TAcc>(o, 0u, h, w); }
    // offset o (per lane) plus so (wave-uniform, a scalar register)
    template <typename TAcc>
    __device__ __forceinline__ void fma_so(unsigned o, unsigned so, TAcc h, TAcc (&w)[NS]) const {
        constexpr int P = nv_lo_stride(NS);
        if constexpr (P == 1) {
            const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, (int)so, 0));
            w[0] += h * (TAcc)v;
        } else if constexpr (P == 2) {
            const nv_f2 v = __builtin_bit_cast(nv_f2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)o, (int)so, 0));
#pragma unroll
            for (int s = 0; s < NS; ++s) w[s] += h * (TAcc)v[s];
        } else if constexpr (P == 3) {
            const nv_f3 v = __builtin_bit_cast(nv_f3, __builtin_amdgcn_raw_buffer_load_b96(r, (int)o, (int)so, 0));
#pragma unroll
            for (int s = 0; s < NS; ++s) w[s] += h * (TAcc)v[s];
        } else if constexpr (P == 4) {
            const nv_f4 v = __builtin_bit_cast(nv_f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, (int)so, 0));
#pragma unroll
            for (int s = 0; s < NS; ++s) w[s] += h * (TAcc)v[s];
        } else {
#pragma unroll
            for (int part = 0; part * 4 < NS; ++part) {
                const nv_f4 v = __builtin_bit_cast(
                    nv_f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(o + 16u * part), (int)so, 0));
#pragma unroll
                for (int s = part * 4; s < NS && s < part * 4 + 4; ++s) w[s] += h * (TAcc)v[s - part * 4];
            }
        }
    }
    using Row = FRow<nv_lo_stride(NS)>;
    __device__ __forceinline__ Row load_so(unsigned o, unsigned so) const {
        constexpr int P = nv_lo_stride(NS);
        Row x;
        if constexpr (P == 1) x.v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, (int)so, 0));
        else if constexpr (P == 2) x.v = __builtin_bit_cast(nv_f2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)o, (int)so, 0));
        else if constexpr (P == 3) x.v = __builtin_bit_cast(nv_f3, __builtin_amdgcn_raw_buffer_load_b96(r, (int)o, (int)so, 0));
        else {
#pragma unroll
            for (int part = 0; part < P / 4; ++part)
                x.v[part] = __builtin_bit_cast(
                    nv_f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(o + 16u * part), (int)so, 0));
        }
        return x;
    }
    template <typename TAcc> static __device__ __forceinline__ void fma_row(const Row &x, TAcc h, TAcc (&w)[NS]) {
        constexpr int P = nv_lo_stride(NS);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if constexpr (P == 1) w[s] += h * (TAcc)x.v;
            else if constexpr (P <= 3) w[s] += h * (TAcc)x.v[s];
            else w[s] += h * (TAcc)x.v[s / 4][s % 4];
        }
    }
};

// state-major FP64 vector, x[s * D + r]: one resource per state
template <int NS> struct XRes<NS, double> {
    static constexpr unsigned kEl = 8;
    __amdgpu_buffer_rsrc_t r[NS];
    __device__ __forceinline__ XRes(const double *x, int D) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            r[s] = __builtin_amdgcn_make_buffer_rsrc((void *)(x + (size_t)s * D), (short)0, (int)((unsigned)D * 8u),
                                                     kBufFlags);
    }
    template <typename TAcc>
    __device__ __forceinline__ void fma(unsigned o, TAcc h, TAcc (&w)[NS]) const {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const double v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r[s], (int)o, 0, 0));
            w[s] += h * (TAcc)v;
        }
    }
};

// interleaved FP64 copy, x[r * nv_lo_stride(NS) + s]: 16-byte loads of two states
struct F64I {};
template <int NS> struct XRes<NS, F64I> {
    static constexpr unsigned kEl = nv_lo_stride(NS) * 8;
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ XRes(const double *x, int D)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, (int)((unsigned)D * kEl), kBufFlags)) {}
    template <typename TAcc>
    __device__ __forceinline__ void fma(unsigned o, TAcc h, TAcc (&w)[NS]) const { fma_so<TAcc>(o, 0u, h, w); }
    template <typename TAcc>
    __device__ __forceinline__ void fma_so(unsigned o, unsigned so, TAcc h, TAcc (&w)[NS]) const {
        typedef double nv_d2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int part = 0; 2 * part < NS; ++part) {
            if (2 * part + 1 < NS) {
                const nv_d2 v = __builtin_bit_cast(
                    nv_d2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(o + 16u * part), (int)so, 0));
                w[2 * part] += h * (TAcc)v[0];
                w[2 * part + 1] += h * (TAcc)v[1];
            } else {
                const double v = __builtin_bit_cast(
                    double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)(o + 16u * part), (int)so, 0));
                w[2 * part] += h * (TAcc)v;
            }
        }
    }
    typedef double nv_rd2 __attribute__((ext_vector_type(2)));
    struct Row {
        nv_rd2 v[NS / 2];
        double t;  // the last state when NS is odd
    };
    __device__ __forceinline__ Row load_so(unsigned o, unsigned so) const {
        Row x;
#pragma unroll
        for (int part = 0; 2 * part + 1 < NS; ++part)
            x.v[part] = __builtin_bit_cast(nv_rd2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(o + 16u * part), (int)so, 0));
        if constexpr (NS % 2 == 1)
            x.t = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)(o + 16u * (NS / 2)), (int)so, 0));
        else
            x.t = 0.0;
        return x;
    }
    template <typename TAcc> static __device__ __forceinline__ void fma_row(const Row &x, TAcc h, TAcc (&w)[NS]) {
#pragma unroll
        for (int s = 0; s + 1 < NS; s += 2) {
            w[s] += h * (TAcc)x.v[s / 2][0];
            w[s + 1] += h * (TAcc)x.v[s / 2][1];
        }
        if constexpr (NS % 2 == 1) w[NS - 1] += h * (TAcc)x.t;
    }
};

// One interleaved row of K values (the H*v input copies), aligned for one
// wide store where its size allows.
__host__ __device__ constexpr size_t il_align(size_t b) {
    return b % 16 == 0 ? 16 : b % 8 == 0 ? 8 : b % 4 == 0 ? 4 : 2;
}
template <typename T, int K> struct alignas(il_align(sizeof(T) * K) < alignof(T) ? alignof(T)
                                                                                  : il_align(sizeof(T) * K)) IlRow {
    T v[K];
};
// rows follow each other without a gap, as H*v reads them (three BF16 values are 6 bytes)
static_assert(sizeof(IlRow<__hip_bfloat16, 1>) == 2 && sizeof(IlRow<__hip_bfloat16, 3>) == 6 &&
                  sizeof(IlRow<float, 3>) == 12 && sizeof(IlRow<double, 3>) == 24,
              "an interleaved row holds its values and nothing else");

__device__ __forceinline__ int64_t slot_of(int64_t i, int64_t nslots) { return i % nslots; }

// A vector element touched once per launch: non-temporal (NT) where the
// vectors are far larger than the caches, plain otherwise (a vector that fits
// the Infinity Cache is read again from it by the next kernel).
template <bool NT, typename T> __device__ __forceinline__ T ld_once(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT, typename T> __device__ __forceinline__ void st_once(T v, T *p) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

}  // namespace nv

// fn<NS>(...) for the operator's number of states
#define NV_DISPATCH_NS(fn, ...)                    \
    switch (op.ns) {                               \
    case 1: return fn<1>(__VA_ARGS__);             \
    case 2: return fn<2>(__VA_ARGS__);             \
    case 3: return fn<3>(__VA_ARGS__);             \
    case 4: return fn<4>(__VA_ARGS__);             \
    case 5: return fn<5>(__VA_ARGS__);             \
    case 6: return fn<6>(__VA_ARGS__);             \
    case 7: return fn<7>(__VA_ARGS__);             \
    case 8: return fn<8>(__VA_ARGS__);             \
    case 9: return fn<9>(__VA_ARGS__);             \
    case 10: return fn<10>(__VA_ARGS__);           \
    default: return hipErrorInvalidValue;          \
    }
