// Shared helpers for the gfx950 KMeans kernels: argument checks, dtype dispatch,
// wave64/block reductions.  Internal to the library; the public ABI is
// include/mi355x_kmeans.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mi355x_kmeans.h"

#define KMX_WAVE 64

#define KMX_REQUIRE_PTR(p) \
    do {                   \
        if ((p) == nullptr) return KMX_ERR_NULL_POINTER; \
    } while (0)

#define KMX_REQUIRE_DTYPE(dt) \
    do {                      \
        if ((dt) != KMX_F32 && (dt) != KMX_F64) return KMX_ERR_BAD_DTYPE; \
    } while (0)

// First statement of every entry point that launches kernels: hipGetLastError reports the
// last error of ANY earlier runtime call of the thread (another library's probe included), so
// a stale one is dropped here and KMX_LAUNCH_CHECK only sees this library's own launches.
#define KMX_ENTRY() (void)hipGetLastError()

#define KMX_LAUNCH_CHECK()                    \
    do {                                      \
        hipError_t e_ = hipGetLastError();    \
        if (e_ != hipSuccess) return (int32_t)e_; \
    } while (0)

static inline size_t kmx_align256(size_t x) { return (x + 255) & ~(size_t)255; }
static inline size_t kmx_dtype_size(int32_t dtype) { return dtype == KMX_F64 ? 8 : 4; }
static inline int64_t kmx_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Number of compute units of the current device (cached); 256 on MI355X.
int32_t kmx_num_cus();

// ---------------------------------------------------------------------------- device side

// W consecutive elements as one memory access that asks for no more alignment than an element has: the
// hardware takes 64- and 128-bit accesses at any multiple of four bytes.  Every row but the first of an
// array whose n is not divisible by four starts off a 16-byte boundary, so three arrays in four used to
// take their rows element by element (per iteration, n = 800 000 against 800 001, us, before: 32 features
// and 64 clusters in fp64 96 / 152, 50 and 100 in fp32 153 / 216).
template <typename T, int W>
struct KmxVec;
template <>
struct KmxVec<float, 1> { typedef float type; };
template <>
struct KmxVec<float, 2> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <>
struct KmxVec<float, 4> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <>
struct KmxVec<double, 1> { typedef double type; };
template <>
struct KmxVec<double, 2> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <>
struct KmxVec<uint32_t, 2> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(4))); };
template <>
struct KmxVec<uint32_t, 4> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(4))); };

// Four consecutive values of a row in memory at i0 (one or two 128-bit accesses when `full`), zero past n.
template <typename T>
__device__ __forceinline__ void kmx_load4(const T* __restrict__ row, int64_t i0, int64_t n, bool full, T (&v)[4]) {
    if (full) {
        constexpr int W = 16 / (int)sizeof(T);
#pragma unroll
        for (int r = 0; r < 4; r += W) {
            const typename KmxVec<T, W>::type q = *reinterpret_cast<const typename KmxVec<T, W>::type*>(row + i0 + r);
#pragma unroll
            for (int e = 0; e < W; ++e) v[r + e] = q[e];
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (i0 + r < n) ? row[i0 + r] : T(0);
    }
}

template <typename T>
__device__ __forceinline__ void kmx_store4(T* __restrict__ row, int64_t i0, int64_t n, bool full, const T (&v)[4]) {
    if (full) {
        constexpr int W = 16 / (int)sizeof(T);
#pragma unroll
        for (int r = 0; r < 4; r += W) {
            typename KmxVec<T, W>::type q;
#pragma unroll
            for (int e = 0; e < W; ++e) q[e] = v[r + e];
            *reinterpret_cast<typename KmxVec<T, W>::type*>(row + i0 + r) = q;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (i0 + r < n) row[i0 + r] = v[r];
    }
}

template <typename T>
__device__ __forceinline__ T kmx_inf();
template <>
__device__ __forceinline__ float kmx_inf<float>() { return __builtin_huge_valf(); }
template <>
__device__ __forceinline__ double kmx_inf<double>() { return __builtin_huge_val(); }

// Whether a value is a NaN or an infinity: all bits of the exponent set.
__device__ __forceinline__ bool kmx_not_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }
__device__ __forceinline__ bool kmx_not_finite(double v) {
    return ((unsigned)(__double_as_longlong(v) >> 32) & 0x7ff00000u) == 0x7ff00000u;
}

// Sum over the 64 lanes of a wave; every lane receives the total.
template <typename T>
__device__ __forceinline__ T kmx_wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, KMX_WAVE);
    return v;
}

// Sum over a block of up to 1024 threads; result valid in thread 0.  `scratch` holds
// at least blockDim.x / 64 elements of T in LDS.  Fixed order, hence reproducible.
template <typename T>
__device__ __forceinline__ T kmx_block_sum(T v, T* scratch) {
    v = kmx_wave_sum(v);
    const int lane = threadIdx.x & (KMX_WAVE - 1);
    const int wave = threadIdx.x / KMX_WAVE;
    const int n_waves = (blockDim.x + KMX_WAVE - 1) / KMX_WAVE;
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    T total = T(0);
    if (threadIdx.x == 0) {
        for (int i = 0; i < n_waves; ++i) total += scratch[i];
    }
    return total;
}

// Hardware floating-point atomic add (LDS or global), result unused.
template <typename T>
__device__ __forceinline__ void kmx_atomic_add(T* addr, T v) {
    unsafeAtomicAdd(addr, v);
}

// (value, index) minimum with the lowest index winning ties.
template <typename T>
__device__ __forceinline__ void kmx_argmin_combine(T& v, int64_t& i, T ov, int64_t oi) {
    if (ov < v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}
