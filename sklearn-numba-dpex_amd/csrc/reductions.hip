// Shared reduction and elementwise kernels for gfx950 (the reference's common/ kernels):
// row/column sums, argmin, half squared norms, broadcast ops, label bookkeeping.
// Sums accumulate in fp64 in a fixed order (thread-strided, wave shuffle tree, wave order,
// block order), so results do not change from run to run.
#include "kmx_common.h"

#include <atomic>
#include <mutex>
#include <type_traits>

namespace {

constexpr int SUM_MAX_BLOCKS_PER_ROW = 256;
constexpr int SUM_COL_CHUNKS = 64;

// A thread's part of a row's sum: 16 bytes per load, two loads in flight; the values behind the last
// whole load go to the first threads of the first workgroup.
template <typename T>
__device__ __forceinline__ double sum_row_part(const T* __restrict__ p, int64_t cols, int square) {
    constexpr int W = 16 / (int)sizeof(T);
    using V = typename KmxVec<T, W>::type;
    const V* __restrict__ pv = reinterpret_cast<const V*>(p);
    const int64_t groups = cols / W;
    const int64_t stride = (int64_t)gridDim.x * 256;
    int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    auto add_one = [&](const T e) {
        const double x = (double)e;
        acc += square ? x * x : x;
    };
    auto add = [&](const V v) {
#pragma unroll
        for (int j = 0; j < W; ++j) add_one(v[j]);
    };
    for (; g + stride < groups; g += 2 * stride) {
        const V a = pv[g];
        const V b = pv[g + stride];
        add(a);
        add(b);
    }
    if (g < groups) add(pv[g]);
    if (blockIdx.x == 0 && groups * W + threadIdx.x < cols) add_one(p[groups * W + threadIdx.x]);
    return acc;
}

template <typename T>
__global__ __launch_bounds__(256) void sum_rows_stage1(const T* __restrict__ in,
                                                       double* __restrict__ partial, int64_t cols,
                                                       int square) {
    const int64_t row = blockIdx.y;
    const T* __restrict__ p = in + (size_t)row * cols;
    const double acc = sum_row_part<T>(p, cols, square);
    __shared__ double scratch[4];
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) partial[(size_t)row * gridDim.x + blockIdx.x] = tot;
}

template <typename T>
__global__ __launch_bounds__(256) void sum_rows_stage2(const double* __restrict__ partial,
                                                       T* __restrict__ out, int n_partials) {
    const int64_t row = blockIdx.x;
    double acc = 0.0;
    for (int j = threadIdx.x; j < n_partials; j += 256) acc += partial[(size_t)row * n_partials + j];
    __shared__ double scratch[4];
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) out[row] = (T)tot;
}

// Row sums in ONE launch (up to SUM_TICKET_ROWS rows): stage 1 as above, then the workgroup of a
// row that gets done last adds the row's partial sums in the order of stage 2 - the same value,
// bit for bit, without the second launch and the gap before it.  The partial sums are handed
// over through device-scope stores, each workgroup waits for its own before it draws its ticket,
// and the last one reads them with device-scope loads (no device-wide fence).
// The tickets live in a device array of the library, zero when the library is loaded and left
// zero by every launch; concurrent launches take different slots of it (handed out in turn).
constexpr int SUM_TICKET_SLOTS = 256;
constexpr int SUM_TICKET_ROWS = 64;
__device__ unsigned int sum_tickets[SUM_TICKET_SLOTS][SUM_TICKET_ROWS];

template <typename T>
__global__ __launch_bounds__(256) void sum_rows_fused(const T* __restrict__ in, double* __restrict__ partial,
                                                      T* __restrict__ out, int64_t cols, int square, int slot) {
    const int64_t row = blockIdx.y;
    const T* __restrict__ p = in + (size_t)row * cols;
    const double acc = sum_row_part<T>(p, cols, square);
    __shared__ double scratch[4];
    __shared__ unsigned int is_last;
    const int n_partials = (int)gridDim.x;
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&partial[(size_t)row * n_partials + blockIdx.x], tot, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        unsigned int* ticket = &sum_tickets[slot][row];
        const unsigned int arrived = atomicAdd(ticket, 1u);
        is_last = arrived == (unsigned int)n_partials - 1u ? 1u : 0u;
        if (is_last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (is_last == 0u) return;
    double acc2 = 0.0;
    for (int j = threadIdx.x; j < n_partials; j += 256)
        acc2 += __hip_atomic_load(&partial[(size_t)row * n_partials + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double tot2 = kmx_block_sum<double>(acc2, scratch);
    if (threadIdx.x == 0) out[row] = (T)tot2;
}

template <typename T>
__global__ __launch_bounds__(256) void sum_cols_stage1(const T* __restrict__ in,
                                                       double* __restrict__ partial, int64_t rows,
                                                       int64_t cols, int64_t rows_per_chunk) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    const int64_t r0 = (int64_t)blockIdx.y * rows_per_chunk;
    int64_t r1 = r0 + rows_per_chunk;
    if (r1 > rows) r1 = rows;
    double acc = 0.0;
    for (int64_t r = r0; r < r1; ++r) acc += (double)in[(size_t)r * cols + c];
    partial[(size_t)blockIdx.y * cols + c] = acc;
}

template <typename T>
__global__ __launch_bounds__(256) void sum_cols_stage2(const double* __restrict__ partial,
                                                       T* __restrict__ out, int64_t cols,
                                                       int n_chunks) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    double acc = 0.0;
    for (int j = 0; j < n_chunks; ++j) acc += partial[(size_t)j * cols + c];
    out[c] = (T)acc;
}

// Single workgroup: n is small wherever the engine needs an argmin (n_local_trials values),
// larger inputs are strided over.
template <typename T>
__global__ __launch_bounds__(1024) void argmin_kernel(const T* __restrict__ values,
                                                      int32_t* __restrict__ out, int64_t n) {
    T best = kmx_inf<T>();
    int64_t arg = INT64_MAX;
    for (int64_t i = threadIdx.x; i < n; i += 1024) {
        const T v = values[i];
        kmx_argmin_combine(best, arg, v, i);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const T ov = __shfl_xor(best, off, 64);
        const int64_t oi = __shfl_xor(arg, off, 64);
        kmx_argmin_combine(best, arg, ov, oi);
    }
    __shared__ T sv[16];
    __shared__ int64_t si[16];
    if ((threadIdx.x & 63) == 0) {
        sv[threadIdx.x >> 6] = best;
        si[threadIdx.x >> 6] = arg;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) kmx_argmin_combine(best, arg, sv[w], si[w]);
        // every value NaN or +inf beyond the first: fall back to the first index
        out[0] = (int32_t)(arg == INT64_MAX ? 0 : arg);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void half_sq_norms_kernel(const T* __restrict__ a_t,
                                                            T* __restrict__ out, int rows,
                                                            int cols) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    T acc = T(0);
    for (int r = 0; r < rows; ++r) {
        const T v = a_t[(size_t)r * cols + c];
        acc += v * v;
    }
    out[c] = acc / T(2);
}

template <typename T>
__global__ __launch_bounds__(256) void broadcast_rows_kernel(T* __restrict__ a,
                                                             const T* __restrict__ v, int64_t rows,
                                                             int64_t cols, int op) {
    const int64_t row = blockIdx.y;
    const T rv = op == 0 ? -v[row] : v[row];
    T* __restrict__ p = a + (size_t)row * cols;
    const int64_t stride = (int64_t)gridDim.x * 256;
    constexpr int W = 16 / (int)sizeof(T);
    using V = typename KmxVec<T, W>::type;
    V* __restrict__ pv = reinterpret_cast<V*>(p);
    const int64_t groups = cols / W;
    for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < groups; g += stride) {
        V x = pv[g];
#pragma unroll
        for (int j = 0; j < W; ++j) x[j] = x[j] + rv;
        pv[g] = x;
    }
    const int64_t c = groups * W + threadIdx.x;  // the values behind the last whole vector
    if (blockIdx.x == 0 && c < cols) p[c] = p[c] + rv;
}

// mean[r] = sums[r] / n in T (in place), stats[0] = sum of mean^2 (fp64, rounded to T).
template <typename T>
__global__ __launch_bounds__(256) void center_mean_kernel(T* __restrict__ mean, T* __restrict__ stats, int64_t rows, T n) {
    __shared__ double scratch[4];
    double acc = 0.0;
    for (int64_t r = threadIdx.x; r < rows; r += 256) {
        const T m = mean[r] / n;
        mean[r] = m;
        acc += (double)m * (double)m;
    }
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) stats[0] = (T)tot;
}

// dst = src - mean per row (dst may be src; left as it is where stats[0] is zero and dst is src) and the
// workgroups' sums of the new values' squares: a pass over X less than centring first and summing then.
template <typename T>
__global__ __launch_bounds__(256) void center_rows_kernel(const T* src, T* dst, const T* __restrict__ mean,
                                                          const T* __restrict__ stats, double* __restrict__ partial,
                                                          int64_t cols) {
    const int64_t row = blockIdx.y;
    const bool any = stats[0] != T(0);  // (NaN: yes)
    const T rv = any ? -mean[row] : T(0);
    const T* p = src + (size_t)row * cols;
    T* q = dst + (size_t)row * cols;
    const bool write = any || src != dst;
    constexpr int W = 16 / (int)sizeof(T);
    using V = typename KmxVec<T, W>::type;
    const int64_t groups = cols / W, stride = (int64_t)gridDim.x * 256;
    double acc = 0.0;
    auto group = [&](const int64_t g, V x) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < W; ++j) {
            if (any) x[j] = x[j] + rv;
            acc += (double)x[j] * (double)x[j];
        }
        if (write) *reinterpret_cast<V*>(q + g * W) = x;
    };
    int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (; g + stride < groups; g += 2 * stride) {  // two loads in flight
        const V a = *reinterpret_cast<const V*>(p + g * W), b = *reinterpret_cast<const V*>(p + (g + stride) * W);
        group(g, a);
        group(g + stride, b);
    }
    if (g < groups) group(g, *reinterpret_cast<const V*>(p + g * W));
    const int64_t c = groups * W + threadIdx.x;  // the values behind the last whole vector
    if (blockIdx.x == 0 && c < cols) {
        const T x = any ? p[c] + rv : p[c];
        acc += (double)x * (double)x;
        if (write) q[c] = x;
    }
    __shared__ double scratch[4];
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) partial[(size_t)row * gridDim.x + blockIdx.x] = tot;
}

// stats[1] = the total of the partial sums, stats[3] = the first weight.
template <typename T>
__global__ __launch_bounds__(1024) void center_total_kernel(const double* __restrict__ partial, int64_t count,
                                                            const T* __restrict__ w, T* __restrict__ stats) {
    __shared__ double scratch[16];
    double acc = 0.0;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < count; i += 1024) acc += partial[i];
    const double tot = kmx_block_sum<double>(acc, scratch);
    if (threadIdx.x == 0) {
        stats[1] = (T)tot;
        stats[3] = w[0];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void broadcast_div_cols_kernel(T* __restrict__ a,
                                                                 const T* __restrict__ v,
                                                                 int64_t rows, int64_t cols) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    const T dv = v[c];
    for (int64_t r = 0; r < rows; ++r) a[(size_t)r * cols + c] = a[(size_t)r * cols + c] / dv;
}

template <typename T>
__global__ __launch_bounds__(256) void divide_by_kernel(T* __restrict__ data, int64_t n, T divisor) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        data[i] = data[i] / divisor;
}

__global__ __launch_bounds__(256) void fill_zero_kernel(unsigned char* __restrict__ data,
                                                        int64_t n_bytes) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    const int64_t n_words = n_bytes / 4;
    uint32_t* w = reinterpret_cast<uint32_t*>(data);
    const bool aligned = (reinterpret_cast<uintptr_t>(data) & 3) == 0;
    if (aligned) {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_words; i += stride) w[i] = 0u;
        for (int64_t i = n_words * 4 + (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_bytes; i += stride)
            data[i] = 0;
    } else {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_bytes; i += stride) data[i] = 0;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void centroid_shifts_kernel(const T* __restrict__ a_t,
                                                              const T* __restrict__ b_t,
                                                              T* __restrict__ out, int d, int k) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= k) return;
    T acc = T(0);
    for (int f = 0; f < d; ++f) {
        const T diff = a_t[(size_t)f * k + c] - b_t[(size_t)f * k + c];
        acc += diff * diff;
    }
    out[c] = acc;
}

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t* __restrict__ p, int64_t n,
                                                       int32_t value, int32_t* extra,
                                                       int32_t extra_value) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) p[i] = value;
    if (extra && blockIdx.x == 0 && threadIdx.x == 0) extra[0] = extra_value;
}

// mapping[l1[i]] = l2[i]; concurrent writers of one slot race, any winner serves: if the two
// labelings agree up to a permutation every writer of a slot stores the same value.
__global__ __launch_bounds__(256) void build_mapping_kernel(const uint32_t* __restrict__ l1,
                                                            const uint32_t* __restrict__ l2,
                                                            int32_t* __restrict__ mapping,
                                                            int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        mapping[l1[i]] = (int32_t)l2[i];
}

__global__ __launch_bounds__(256) void check_mapping_kernel(const uint32_t* __restrict__ l1,
                                                            const uint32_t* __restrict__ l2,
                                                            const int32_t* __restrict__ mapping,
                                                            int32_t* __restrict__ result,
                                                            int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        bad |= mapping[l1[i]] != (int32_t)l2[i];
    if (__any(bad) && (threadIdx.x & 63) == 0) result[0] = 0;
}

// The labels that occur, gathered in LDS (a byte per cluster; the stores of a wave that fall on one
// byte all write 1) before a workgroup touches memory: at most k atomics per workgroup, and those
// only for clusters no other workgroup has reported yet.  With an atomic per label that looks new,
// every wave of the first round queued up at the same few words: 541 us for 70 000 labels of 10
// clusters, 180 us for 100 000 of 20; now 6 us for either (latency of two trips to memory).
constexpr int DISTINCT_LDS_CLUSTERS = 32768;
__global__ __launch_bounds__(256) void count_distinct_lds_kernel(const uint32_t* __restrict__ labels,
                                                                 int32_t* __restrict__ seen,
                                                                 int32_t* __restrict__ result, int64_t n, int k) {
    extern __shared__ __align__(16) unsigned char here[];
    for (int c = threadIdx.x; c < (k + 3) / 4; c += 256) reinterpret_cast<uint32_t*>(here)[c] = 0u;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * 256;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if ((reinterpret_cast<uintptr_t>(labels) & 15) == 0) {
        const uint4* __restrict__ l4 = reinterpret_cast<const uint4*>(labels);
        const int64_t n4 = n / 4;
        for (int64_t g = i; g < n4; g += stride) {
            const uint4 v = l4[g];
            here[v.x] = 1;
            here[v.y] = 1;
            here[v.z] = 1;
            here[v.w] = 1;
        }
        i += n4 * 4;
    }
    for (; i < n; i += stride) here[labels[i]] = 1;
    __syncthreads();
    int fresh = 0;
    for (int c = threadIdx.x; c < k; c += 256)
        if (here[c] != 0 && __builtin_nontemporal_load(seen + c) == 0 && atomicExch(seen + c, 1) == 0) ++fresh;
    fresh = kmx_wave_sum(fresh);
    if ((threadIdx.x & 63) == 0 && fresh > 0) atomicAdd(result, fresh);
}

// more clusters than that: an atomic per label that nobody seems to have reported
__global__ __launch_bounds__(256) void count_distinct_kernel(const uint32_t* __restrict__ labels,
                                                             int32_t* __restrict__ seen,
                                                             int32_t* __restrict__ result,
                                                             int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        const uint32_t l = labels[i];
        if (__builtin_nontemporal_load(seen + l) > 0) continue;
        if (atomicAdd(seen + l, 1) == 0) atomicAdd(result, 1);
    }
}

int grid_for(int64_t n) {
    int64_t blocks = kmx_cdiv(n, 256);
    const int64_t cap = (int64_t)kmx_num_cus() * 8;
    if (blocks > cap) blocks = cap;
    return (int)(blocks < 1 ? 1 : blocks);
}

// Workgroups per row of the centring pass: 16 KB of a row each, 16 384 in all where that is more.
int64_t center_blocks_per_row(int64_t rows, int64_t cols) {
    int64_t b = kmx_cdiv(cols, 256 * 16);
    if (b * rows > 16384) b = kmx_cdiv(16384, rows);
    return b < 1 ? 1 : b;
}

int sum_blocks_per_row(int64_t cols) {
    int64_t b = kmx_cdiv(cols, 256 * 8);
    if (b > SUM_MAX_BLOCKS_PER_ROW) b = SUM_MAX_BLOCKS_PER_ROW;
    return (int)(b < 1 ? 1 : b);
}

// The elements of a transposed tile that fit its LDS (33 KB: four workgroups' tiles and their
// loads are in flight on a compute unit).
template <typename T>
constexpr int TRANSPOSE_LDS = 33792 / (int)sizeof(T);
constexpr int TRANSPOSE_XCDS = 8;

// dst (cols x rows) = transpose of src (rows x cols), through LDS.  Bound by memory.  A tile is
// tall (up to 1 KB of a row of dst) and narrow (about 32 columns): dst's rows start at any
// address, and long runs leave few cache lines that two tiles share.  Tiles are numbered along
// the columns and handed out to the XCDs in contiguous ranges, so the lines that neighbours share
// meet in one L2.  Both sides walk the tile flat, every lane with an element, eight loads in flight
// per lane; an odd pitch spreads the transposed stores over the banks.
// 70 000 x 784 fp32 106 -> 87 us (5.0 TB/s); 300 007 x 100 fp32 82 -> 59 us (4.0 TB/s), both with the
// check, from tiles of 64 x 64 without it.
// CHECK: *not_finite = 1 if an element is a NaN or an infinity (any number of equal stores).
template <typename T, bool CHECK>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ src, T* __restrict__ dst,
                                                        int64_t rows, int64_t cols, int tile_r, int tile_c,
                                                        int64_t tiles_c, int64_t tiles, int64_t per_xcd,
                                                        int32_t* __restrict__ not_finite) {
    __shared__ T tile[TRANSPOSE_LDS<T>];
    const int64_t t = (int64_t)(blockIdx.x % TRANSPOSE_XCDS) * per_xcd + blockIdx.x / TRANSPOSE_XCDS;
    if (t >= tiles) return;
    const int64_t r0 = t / tiles_c * tile_r, c0 = t % tiles_c * tile_c;
    const int nr = rows - r0 < tile_r ? (int)(rows - r0) : tile_r;
    const int nc = cols - c0 < tile_c ? (int)(cols - c0) : tile_c;
    const int pitch = tile_r | 1;
    constexpr int B = 8;
    bool bad = false;
    {
        const T* __restrict__ from = src + (size_t)r0 * cols + c0;
        const int step_r = 256 / nc, step_c = 256 % nc;
        int r = (int)threadIdx.x / nc, c = (int)threadIdx.x % nc;
        for (int e0 = 0; e0 < nr * nc; e0 += 256 * B) {
            T v[B];
            int at[B];
#pragma unroll
            for (int i = 0; i < B; ++i) {
                const int rc = r < nr ? r : nr - 1;  // past the end: a valid element, not kept
                v[i] = from[(size_t)rc * cols + c];
                at[i] = r < nr ? c * pitch + r : -1;
                r += step_r;
                c += step_c;
                if (c >= nc) {
                    c -= nc;
                    ++r;
                }
            }
#pragma unroll
            for (int i = 0; i < B; ++i) {
                if (CHECK) bad |= kmx_not_finite(v[i]);
                if (at[i] >= 0) tile[at[i]] = v[i];
            }
        }
    }
    if (CHECK && bad) *not_finite = 1;
    __syncthreads();
    T* __restrict__ to = dst + (size_t)c0 * rows + r0;
    const int step_c = 256 / nr, step_r = 256 % nr;
    int c = (int)threadIdx.x / nr, r = (int)threadIdx.x % nr;
#pragma unroll 4
    for (int e = threadIdx.x; e < nr * nc; e += 256) {
        to[(size_t)c * rows + r] = tile[c * pitch + r];
        c += step_c;
        r += step_r;
        if (r >= nr) {
            r -= nr;
            ++c;
        }
    }
}

// *not_finite = 1 if one of the n values is a NaN or an infinity.  One read at memory speed;
// VEC: 16 bytes a load (aligned arrays).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void all_finite_kernel(const T* __restrict__ a, int64_t n,
                                                         int32_t* __restrict__ not_finite) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    bool bad = false;
    int64_t done = 0;
    if constexpr (VEC) {
        constexpr int V = 16 / sizeof(T);
        struct alignas(16) Quad { T v[V]; };
        const Quad* __restrict__ q = reinterpret_cast<const Quad*>(a);
        const int64_t nq = n / V;
#pragma unroll 4
        for (int64_t i = id; i < nq; i += stride) {
            const Quad x = q[i];
#pragma unroll
            for (int j = 0; j < V; ++j) bad |= kmx_not_finite(x.v[j]);
        }
        done = nq * V;
    }
    for (int64_t i = done + id; i < n; i += stride) bad |= kmx_not_finite(a[i]);
    if (bad) *not_finite = 1;
}

// Tile of the transposed copy: up to 1 KB of a dst row (2 KB where src has at most 16 columns, or a
// tile would be a few elements per lane), and the columns that then fit the LDS, evenly split.
template <typename T>
void launch_transpose(const void* src, void* dst, int64_t rows, int64_t cols, int32_t* not_finite, hipStream_t s) {
    const int64_t most_r = (cols <= 16 ? 2048 : 1024) / (int64_t)sizeof(T);
    const int tile_r = (int)(rows < most_r ? rows : most_r);
    const int64_t fit_c = TRANSPOSE_LDS<T> / (tile_r | 1);
    const int64_t tiles_c = kmx_cdiv(cols, fit_c);
    const int tile_c = (int)kmx_cdiv(cols, tiles_c);
    const int64_t used_c = kmx_cdiv(cols, tile_c);
    const int64_t tiles = used_c * kmx_cdiv(rows, tile_r), per_xcd = kmx_cdiv(tiles, TRANSPOSE_XCDS);
    const dim3 grid((unsigned)(per_xcd * TRANSPOSE_XCDS));
    if (not_finite)
        hipLaunchKernelGGL((transpose_kernel<T, true>), grid, dim3(256), 0, s, (const T*)src, (T*)dst, rows, cols,
                           tile_r, tile_c, used_c, tiles, per_xcd, not_finite);
    else
        hipLaunchKernelGGL((transpose_kernel<T, false>), grid, dim3(256), 0, s, (const T*)src, (T*)dst, rows, cols,
                           tile_r, tile_c, used_c, tiles, per_xcd, not_finite);
}

int32_t transpose_copy(const void* src, void* dst, int64_t rows, int64_t cols, int32_t* not_finite, int32_t dtype,
                       hipStream_t stream) {
    KMX_REQUIRE_PTR(src);
    KMX_REQUIRE_PTR(dst);
    if (rows <= 0 || cols <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    if (src == dst) return KMX_ERR_BAD_ARGUMENT;
    if (kmx_cdiv(cols, 64) * kmx_cdiv(rows, 64) > INT32_MAX) return KMX_ERR_BAD_SHAPE;
    if (not_finite)
        hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, stream, not_finite, (int64_t)1, 0,
                           (int32_t*)nullptr, 0);
    if (dtype == KMX_F32)
        launch_transpose<float>(src, dst, rows, cols, not_finite, stream);
    else
        launch_transpose<double>(src, dst, rows, cols, not_finite, stream);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

}  // namespace

extern "C" {

size_t kmx_sum_workspace_bytes(int64_t rows, int64_t cols) {
    if (rows <= 0 || cols <= 0) return 0;
    const size_t a = (size_t)rows * SUM_MAX_BLOCKS_PER_ROW * sizeof(double);
    const size_t b = (size_t)cols * SUM_COL_CHUNKS * sizeof(double);
    return kmx_align256(a > b ? a : b);
}

int32_t kmx_sum_rows(const void* in, void* out, int64_t rows, int64_t cols, int32_t square,
                     void* workspace, size_t workspace_bytes, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(in);
    KMX_REQUIRE_PTR(out);
    KMX_REQUIRE_PTR(workspace);
    if (rows <= 0 || cols <= 0 || rows > 65535) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    const int b = sum_blocks_per_row(cols);
    if (workspace_bytes < (size_t)rows * b * sizeof(double)) return KMX_ERR_WORKSPACE;
    hipStream_t stream = (hipStream_t)stream_;
    double* partial = (double*)workspace;
    // Few workgroups (one round of them on the chip): one launch, the last workgroup of a row
    // finishes it (same sums, same order).  The hand-over costs every workgroup two round trips
    // to memory at its end, which a launch of many short workgroups pays for more dearly than
    // for the second launch: 14 rows of 5e6 values took 69 us that way against 45 us.
    static std::atomic<unsigned int> next_slot{0};
    const bool fused = rows <= SUM_TICKET_ROWS && rows * (int64_t)b <= 2 * (int64_t)kmx_num_cus();
    const int slot = fused ? (int)(next_slot.fetch_add(1u) % (unsigned int)SUM_TICKET_SLOTS) : 0;
#define KMX_SUM_ROWS(T)                                                                            \
    do {                                                                                           \
        if (fused) {                                                                               \
            hipLaunchKernelGGL((sum_rows_fused<T>), dim3(b, (unsigned)rows), dim3(256), 0, stream, \
                               (const T*)in, partial, (T*)out, cols, square, slot);                \
        } else {                                                                                   \
            hipLaunchKernelGGL((sum_rows_stage1<T>), dim3(b, (unsigned)rows), dim3(256), 0, stream, \
                               (const T*)in, partial, cols, square);                               \
            hipLaunchKernelGGL((sum_rows_stage2<T>), dim3((unsigned)rows), dim3(256), 0, stream,    \
                               partial, (T*)out, b);                                               \
        }                                                                                          \
    } while (0)
    if (dtype == KMX_F32) KMX_SUM_ROWS(float); else KMX_SUM_ROWS(double);
#undef KMX_SUM_ROWS
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

// ---- kmx_sum_rows without any allocation: the per-workgroup partial sums live in a
// file-scope device array instead of a caller-provided workspace.
}  // extern "C"

namespace {
constexpr int SUM_STATIC_MAX_ROWS = 64;
__device__ __align__(256) double sum_static_scratch[SUM_STATIC_MAX_ROWS * SUM_MAX_BLOCKS_PER_ROW];  // 128 KiB

// Device address of sum_static_scratch on the current device (every GPU holds its own copy of
// the array at its own address; the array's name is only a host-side handle and must never be
// handed to a kernel).  Looked up once per device; no allocation.
constexpr int SUM_STATIC_MAX_DEVICES = 64;
int32_t sum_static_scratch_ptr(double** out) {
    static double* ptrs[SUM_STATIC_MAX_DEVICES] = {};
    static std::mutex lock;
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int32_t)e;
    if (dev < 0 || dev >= SUM_STATIC_MAX_DEVICES) return KMX_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> guard(lock);
    if (ptrs[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(sum_static_scratch));
        if (e != hipSuccess) return (int32_t)e;
        if (p == nullptr) return KMX_ERR_UNSUPPORTED;
        ptrs[dev] = static_cast<double*>(p);
    }
    *out = ptrs[dev];
    return KMX_OK;
}
}  // namespace

extern "C" {

int32_t kmx_sum_rows_static(const void* in, void* out, int64_t rows, int64_t cols, int32_t square,
                            int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(in);
    KMX_REQUIRE_PTR(out);
    if (rows <= 0 || cols <= 0) return KMX_ERR_BAD_SHAPE;
    if (rows > SUM_STATIC_MAX_ROWS) return KMX_ERR_UNSUPPORTED;  // beyond the static scratch
    KMX_REQUIRE_DTYPE(dtype);
    double* partial = nullptr;
    const int32_t rc = sum_static_scratch_ptr(&partial);
    if (rc != KMX_OK) return rc;
    // stage 1 writes every slot stage 2 reads (rows * b of them), so nothing has to start at
    // zero and the previous call's contents do not matter
    return kmx_sum_rows(in, out, rows, cols, square, partial,
                        sizeof(double) * SUM_STATIC_MAX_ROWS * SUM_MAX_BLOCKS_PER_ROW, dtype, stream_);
}

int32_t kmx_sum_cols(const void* in, void* out, int64_t rows, int64_t cols, void* workspace,
                     size_t workspace_bytes, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(in);
    KMX_REQUIRE_PTR(out);
    KMX_REQUIRE_PTR(workspace);
    if (rows <= 0 || cols <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    int64_t chunks = kmx_cdiv(rows, 64);
    if (chunks > SUM_COL_CHUNKS) chunks = SUM_COL_CHUNKS;
    const int64_t rows_per_chunk = kmx_cdiv(rows, chunks);
    chunks = kmx_cdiv(rows, rows_per_chunk);
    if (workspace_bytes < (size_t)chunks * cols * sizeof(double)) return KMX_ERR_WORKSPACE;
    hipStream_t stream = (hipStream_t)stream_;
    double* partial = (double*)workspace;
    const unsigned gx = (unsigned)kmx_cdiv(cols, 256);
    if (dtype == KMX_F32) {
        hipLaunchKernelGGL((sum_cols_stage1<float>), dim3(gx, (unsigned)chunks), dim3(256), 0,
                           stream, (const float*)in, partial, rows, cols, rows_per_chunk);
        hipLaunchKernelGGL((sum_cols_stage2<float>), dim3(gx), dim3(256), 0, stream, partial,
                           (float*)out, cols, (int)chunks);
    } else {
        hipLaunchKernelGGL((sum_cols_stage1<double>), dim3(gx, (unsigned)chunks), dim3(256), 0,
                           stream, (const double*)in, partial, rows, cols, rows_per_chunk);
        hipLaunchKernelGGL((sum_cols_stage2<double>), dim3(gx), dim3(256), 0, stream, partial,
                           (double*)out, cols, (int)chunks);
    }
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_argmin(const void* values, int32_t* out, int64_t n, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(values);
    KMX_REQUIRE_PTR(out);
    if (n <= 0 || n > INT32_MAX) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((argmin_kernel<float>), dim3(1), dim3(1024), 0, stream,
                           (const float*)values, out, n);
    else
        hipLaunchKernelGGL((argmin_kernel<double>), dim3(1), dim3(1024), 0, stream,
                           (const double*)values, out, n);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_half_sq_norms(const void* a_t, void* out, int32_t rows, int32_t cols, int32_t dtype,
                          void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(a_t);
    KMX_REQUIRE_PTR(out);
    if (rows <= 0 || cols <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    const unsigned grid = (unsigned)kmx_cdiv(cols, 256);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((half_sq_norms_kernel<float>), dim3(grid), dim3(256), 0, stream,
                           (const float*)a_t, (float*)out, rows, cols);
    else
        hipLaunchKernelGGL((half_sq_norms_kernel<double>), dim3(grid), dim3(256), 0, stream,
                           (const double*)a_t, (double*)out, rows, cols);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_transpose(const void* src, void* dst, int64_t rows, int64_t cols, int32_t dtype, void* stream) {
    KMX_ENTRY();
    return transpose_copy(src, dst, rows, cols, nullptr, dtype, (hipStream_t)stream);
}

int32_t kmx_transpose_finite(const void* src, void* dst, int64_t rows, int64_t cols, int32_t* not_finite,
                             int32_t dtype, void* stream) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(not_finite);
    return transpose_copy(src, dst, rows, cols, not_finite, dtype, (hipStream_t)stream);
}

int32_t kmx_all_finite(const void* data, int64_t n_items, int32_t* not_finite, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(data);
    KMX_REQUIRE_PTR(not_finite);
    if (n_items <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, stream, not_finite, (int64_t)1, 0, (int32_t*)nullptr, 0);
    // (four loads of 16 bytes per thread, at most eight workgroups a compute unit)
    int64_t blocks = kmx_cdiv(n_items * (int64_t)kmx_dtype_size(dtype), 256 * 64);
    if (blocks > 8 * kmx_num_cus()) blocks = 8 * kmx_num_cus();
    const bool vec = (uintptr_t)data % 16 == 0;
#define KMX_FINITE(T, VEC)                                                                               \
    hipLaunchKernelGGL((all_finite_kernel<T, VEC>), dim3((unsigned)blocks), dim3(256), 0, stream, (const T*)data, \
                       n_items, not_finite)
    if (dtype == KMX_F32) {
        if (vec) KMX_FINITE(float, true); else KMX_FINITE(float, false);
    } else {
        if (vec) KMX_FINITE(double, true); else KMX_FINITE(double, false);
    }
#undef KMX_FINITE
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

// The partial sums of the rows (those of the weights are one row's) or of the centring pass, one after the other:
// not the column sums' scratch of kmx_sum_workspace_bytes, 512 bytes a column.
size_t kmx_center_workspace_bytes(int64_t rows, int64_t cols) {
    if (rows <= 0 || cols <= 0) return 0;
    const int64_t a = sum_blocks_per_row(cols), b = center_blocks_per_row(rows, cols);
    return kmx_align256((size_t)rows * (size_t)(a > b ? a : b) * sizeof(double));
}

int32_t kmx_center_rows(const void* X_t, void* dst, const void* sample_weight, void* mean, void* stats, void* workspace,
                        size_t workspace_bytes, int64_t rows, int64_t cols, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(dst);
    KMX_REQUIRE_PTR(sample_weight);
    KMX_REQUIRE_PTR(mean);
    KMX_REQUIRE_PTR(stats);
    KMX_REQUIRE_PTR(workspace);
    if (rows <= 0 || cols <= 0 || rows > 65535) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    if (workspace_bytes < kmx_center_workspace_bytes(rows, cols)) return KMX_ERR_WORKSPACE;
    hipStream_t stream = (hipStream_t)stream_;
    // (one workspace: the launches follow one another on the stream)
    int32_t rc = kmx_sum_rows(sample_weight, (char*)stats + 2 * kmx_dtype_size(dtype), 1, cols, 0, workspace,
                              workspace_bytes, dtype, stream_);
    if (rc != KMX_OK) return rc;
    rc = kmx_sum_rows(X_t, mean, rows, cols, 0, workspace, workspace_bytes, dtype, stream_);
    if (rc != KMX_OK) return rc;
    const int64_t b = center_blocks_per_row(rows, cols);
    double* partial = (double*)workspace;
#define KMX_CENTER(T)                                                                                                  \
    do {                                                                                                               \
        hipLaunchKernelGGL((center_mean_kernel<T>), dim3(1), dim3(256), 0, stream, (T*)mean, (T*)stats, rows, (T)cols); \
        hipLaunchKernelGGL((center_rows_kernel<T>), dim3((unsigned)b, (unsigned)rows), dim3(256), 0, stream,           \
                           (const T*)X_t, (T*)dst, (const T*)mean, (const T*)stats, partial, cols);                    \
        hipLaunchKernelGGL((center_total_kernel<T>), dim3(1), dim3(1024), 0, stream, partial, b * rows,                \
                           (const T*)sample_weight, (T*)stats);                                                        \
    } while (0)
    if (dtype == KMX_F32) KMX_CENTER(float); else KMX_CENTER(double);
#undef KMX_CENTER
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_broadcast_rows(void* a, const void* v, int64_t rows, int64_t cols, int32_t op,
                           int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(a);
    KMX_REQUIRE_PTR(v);
    if (rows <= 0 || cols <= 0 || rows > 65535) return KMX_ERR_BAD_SHAPE;
    if (op != 0 && op != 1) return KMX_ERR_BAD_ARGUMENT;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    int64_t gx = kmx_cdiv(cols, 256 * 4);
    if (gx > 2048) gx = 2048;
#define KMX_BCAST(T)                                                                            \
    hipLaunchKernelGGL((broadcast_rows_kernel<T>), dim3((unsigned)gx, (unsigned)rows),           \
                       dim3(256), 0, stream, (T*)a, (const T*)v, rows, cols, op)
    if (dtype == KMX_F32) KMX_BCAST(float); else KMX_BCAST(double);
#undef KMX_BCAST
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_broadcast_div_cols(void* a, const void* v, int64_t rows, int64_t cols, int32_t dtype,
                               void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(a);
    KMX_REQUIRE_PTR(v);
    if (rows <= 0 || cols <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    const unsigned grid = (unsigned)kmx_cdiv(cols, 256);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((broadcast_div_cols_kernel<float>), dim3(grid), dim3(256), 0, stream,
                           (float*)a, (const float*)v, rows, cols);
    else
        hipLaunchKernelGGL((broadcast_div_cols_kernel<double>), dim3(grid), dim3(256), 0, stream,
                           (double*)a, (const double*)v, rows, cols);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_divide_by(void* data, int64_t n_items, double divisor, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(data);
    if (n_items <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    const int grid = grid_for(n_items);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((divide_by_kernel<float>), dim3(grid), dim3(256), 0, stream,
                           (float*)data, n_items, (float)divisor);
    else
        hipLaunchKernelGGL((divide_by_kernel<double>), dim3(grid), dim3(256), 0, stream,
                           (double*)data, n_items, divisor);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_fill_zero(void* data, int64_t n_bytes, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(data);
    if (n_bytes < 0) return KMX_ERR_BAD_SHAPE;
    if (n_bytes == 0) return KMX_OK;
    hipStream_t stream = (hipStream_t)stream_;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(n_bytes / 4 + 1)), dim3(256), 0, stream,
                       (unsigned char*)data, n_bytes);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_centroid_shifts(const void* a_t, const void* b_t, void* out, int32_t d, int32_t k,
                            int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(a_t);
    KMX_REQUIRE_PTR(b_t);
    KMX_REQUIRE_PTR(out);
    if (d <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    const unsigned grid = (unsigned)kmx_cdiv(k, 256);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((centroid_shifts_kernel<float>), dim3(grid), dim3(256), 0, stream,
                           (const float*)a_t, (const float*)b_t, (float*)out, d, k);
    else
        hipLaunchKernelGGL((centroid_shifts_kernel<double>), dim3(grid), dim3(256), 0, stream,
                           (const double*)a_t, (const double*)b_t, (double*)out, d, k);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_is_same_clustering(const uint32_t* labels1, const uint32_t* labels2, int32_t* mapping,
                               int32_t* result, int64_t n, int32_t k, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(labels1);
    KMX_REQUIRE_PTR(labels2);
    KMX_REQUIRE_PTR(mapping);
    KMX_REQUIRE_PTR(result);
    if (n <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    hipStream_t stream = (hipStream_t)stream_;
    const int grid = grid_for(n);
    hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, stream, mapping, (int64_t)k, -1,
                       result, 1);
    hipLaunchKernelGGL(build_mapping_kernel, dim3(grid), dim3(256), 0, stream, labels1, labels2,
                       mapping, n);
    hipLaunchKernelGGL(check_mapping_kernel, dim3(grid), dim3(256), 0, stream, labels1, labels2,
                       mapping, result, n);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_count_distinct_clusters(const uint32_t* labels, int32_t* seen, int32_t* result,
                                    int64_t n, int32_t k, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(labels);
    KMX_REQUIRE_PTR(seen);
    KMX_REQUIRE_PTR(result);
    if (n <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    hipStream_t stream = (hipStream_t)stream_;
    hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, stream, seen, (int64_t)k, 0, result,
                       0);
    if (k <= DISTINCT_LDS_CLUSTERS) {
        // (sixteen labels per thread and round; a workgroup per compute unit at most)
        int64_t blocks = kmx_cdiv(n, 256 * 16);
        if (blocks > kmx_num_cus()) blocks = kmx_num_cus();
        hipLaunchKernelGGL(count_distinct_lds_kernel, dim3((unsigned)blocks), dim3(256), (size_t)((k + 3) & ~3), stream,
                           labels, seen, result, n, k);
    } else {
        hipLaunchKernelGGL(count_distinct_kernel, dim3(grid_for(n)), dim3(256), 0, stream, labels, seen, result, n);
    }
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

}  // extern "C"
