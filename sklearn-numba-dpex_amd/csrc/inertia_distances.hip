// Per-sample inertia, euclidean distances and empty-cluster relocation for gfx950.
// Inertia and relocation are HBM-bound passes over X_t: one thread per sample, features read with
// coalesced loads (consecutive lanes = consecutive samples of one feature row).  Distances are taken
// from either layout of X, in fp32 on the fp64 matrix cores.
#include "kmx_common.h"

#include <type_traits>

namespace {

// out[i] = w_i * sum_f (x_fi - c_f,label_i)^2, features accumulated in order.  A thread takes
// four consecutive samples (128-bit loads of every feature row); the centroids are staged in
// LDS when they fit (LDS_CENTROIDS), so that the per-sample gather of the label's centroid
// does not go through the vector memory pipe.
// SUM: nothing is written per sample; the workgroup's total goes to its slot of `partial` in fp64
// (fixed order inside the workgroup, so the result does not depend on timing).  With few samples
// of many features the launch has a second grid dimension and workgroup (x, y) takes the y-th
// stretch of the features only: a thread that walks hundreds of feature rows alone, with a few
// hundred threads on the whole device, is a chain of trips to memory.
template <typename T, bool LDS_CENTROIDS, bool SUM>
__global__ __launch_bounds__(256) void per_sample_inertia_kernel(
    const T* __restrict__ X_t, const T* __restrict__ sample_weight,
    const T* __restrict__ centroids_t, const uint32_t* __restrict__ labels, T* __restrict__ out,
    double* __restrict__ partial, int64_t n, int d, int k) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* cs = reinterpret_cast<T*>(smem_raw);  // the workgroup's feature rows of centroids_t, same layout
    const int f_chunk = (d + (int)gridDim.y - 1) / (int)gridDim.y;
    const int f_begin = (int)blockIdx.y * f_chunk;
    const int f_end = f_begin + f_chunk < d ? f_begin + f_chunk : d;
    if (LDS_CENTROIDS) {
        for (int idx = threadIdx.x; idx < (f_end - f_begin) * k; idx += 256) cs[idx] = centroids_t[(size_t)f_begin * k + idx];
        __syncthreads();
    }
    // (row f of the centroids: cent + f k)
    const T* __restrict__ cent = LDS_CENTROIDS ? cs - (size_t)f_begin * k : centroids_t;
    const int64_t n_groups = (n + 3) >> 2;
    const int64_t stride = (int64_t)gridDim.x * 256;
    double total = 0.0;
    (void)total;
    // Rows in flight: eight where few workgroups wait for memory, the values of a relocation among many features
    // (30 002 x 500 fp64: 161 us with four, 139 with eight; 206 with a branch per row, 144 as single loads); else
    // four (1 000 003 x 100 fp64, sum: 145 us, 150 with eight; 2e6 x 32 fp64, values: 93 and 99).
    constexpr int WALK = SUM || LDS_CENTROIDS ? 4 : 8;
    for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < n_groups; g += stride) {
        const int64_t i0 = g * 4;
        const bool full = i0 + 4 <= n;
        uint32_t c[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r] = (i0 + r < n) ? labels[i0 + r] : 0u;
        T acc[4] = {T(0), T(0), T(0), T(0)};
        // (decided before the walk: a branch per row would have each load waited for before the next)
        const auto walk = [&](auto whole) {
#pragma unroll WALK
            for (int f = f_begin; f < f_end; ++f) {
                T x[4];
                kmx_load4<T>(X_t + (size_t)f * n, i0, n, decltype(whole)::value, x);
                const T* __restrict__ crow = cent + (size_t)f * k;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const T diff = x[r] - crow[c[r]];
                    acc[r] += diff * diff;
                }
            }
        };
        if (full) walk(std::true_type{});
        else walk(std::false_type{});
        if (sample_weight) {
            T w[4];
            kmx_load4<T>(sample_weight, i0, n, full, w);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] *= w[r];
        }
        if constexpr (SUM) {
            // samples past n have x = 0 and label 0: their value is dropped here
#pragma unroll
            for (int r = 0; r < 4; ++r) total += (i0 + r < n) ? (double)acc[r] : 0.0;
        } else {
            kmx_store4<T>(out, i0, n, full, acc);
        }
    }
    if constexpr (SUM) {
        __shared__ double wave_part[4];
        total = kmx_block_sum<double>(total, wave_part);
        if (threadIdx.x == 0) partial[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = total;
    }
}

// The same from the rows of a row-major copy of X and of the packed centroids: 16 lanes per sample and
// 128-bit loads, so that the gathered centroid is whole cache lines too; lanes sum in T, the sample and
// the total in fp64.  Bound by reading X once.  WHOLE: rows of whole 16-byte groups; else the last
// values of a row are loaded one by one.
// per-sample values to `out` (SUM false) or the workgroup's total to `partial`.
template <typename T, bool WHOLE, bool SUM>
__global__ __launch_bounds__(256) void rows_inertia_kernel(
    const T* __restrict__ X_rm, const T* __restrict__ sample_weight, const T* __restrict__ cpack,
    const uint32_t* __restrict__ labels, T* __restrict__ out, double* __restrict__ partial, int64_t n, int d, int dpad) {
    constexpr int W = 16 / (int)sizeof(T);
    using V = typename KmxVec<T, W>::type;
    const int e = threadIdx.x & 15;
    const int64_t per_pass = (int64_t)gridDim.x * 32;  // two samples per group of lanes
    double total = 0.0;
    for (int64_t base = (int64_t)blockIdx.x * 32; base < n; base += per_pass) {
        const int64_t i0 = base + 2 * (threadIdx.x >> 4);
        const T* __restrict__ row[2];
        const T* __restrict__ cen[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t i = i0 + u < n ? i0 + u : n - 1;
            row[u] = X_rm + (size_t)i * d;
            cen[u] = cpack + (size_t)labels[i] * dpad;
        }
        T acc[2] = {T(0), T(0)};
#pragma unroll 2
        for (int f = e * W; f < d; f += 16 * W) {
            T x[2][W], c[2][W];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (WHOLE || f + W <= d) {
                    const V xv = *reinterpret_cast<const V*>(row[u] + f), cv = *reinterpret_cast<const V*>(cen[u] + f);
#pragma unroll
                    for (int j = 0; j < W; ++j) {
                        x[u][j] = xv[j];
                        c[u][j] = cv[j];
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < W; ++j) {
                        x[u][j] = f + j < d ? row[u][f + j] : T(0);
                        c[u][j] = f + j < d ? cen[u][f + j] : T(0);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    const T diff = x[u][j] - c[u][j];
                    acc[u] += diff * diff;
                }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            double v = (double)acc[u];
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
            if (e == 0 && i0 + u < n) {
                if (sample_weight != nullptr) v *= (double)sample_weight[i0 + u];
                if constexpr (SUM) total += v;
                else out[i0 + u] = (T)v;
            }
        }
    }
    if constexpr (SUM) {
        __shared__ double wave_part[4];
        total = kmx_block_sum<double>(total, wave_part);
        if (threadIdx.x == 0) partial[blockIdx.x] = total;
    }
}

// out[0] = sum of the workgroup partials, in order.
template <typename T>
__global__ __launch_bounds__(256) void inertia_total_kernel(const double* __restrict__ partial, int count,
                                                            T* __restrict__ out) {
    __shared__ double wave_part[4];
    double v = 0.0;
    for (int i = threadIdx.x; i < count; i += 256) v += partial[i];
    v = kmx_block_sum<double>(v, wave_part);
    if (threadIdx.x == 0) out[0] = (T)v;
}

// Square root of a non-negative squared distance.  fp32: the hardware approximation (1 ulp)
// refined by one Newton step on the residual, which is within an ulp of the correctly rounded
// root at a third of its cost; tiny arguments, where the approximation loses bits, take the
// library routine.
__device__ __forceinline__ float dist_sqrt(float a) {
    if (a < 1e-30f) return sqrtf(a);
    const float s = __builtin_amdgcn_sqrtf(a);
    const float half_inv = 0.5f * __builtin_amdgcn_rcpf(s);
    return fmaf(fmaf(-s, s, a), half_inv, s);
}
__device__ __forceinline__ double dist_sqrt(double a) { return sqrt(a); }

// Four consecutive values in LDS at a 16-byte boundary.
template <typename T>
__device__ __forceinline__ void lds_load4(const T* p, T (&v)[4]) {
    struct alignas(16) Four { T e[4]; };
    const Four q = *reinterpret_cast<const Four*>(p);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = q.e[r];
}

// distances_t[c, i] = sqrt(sum_f (c_fc - x_fi)^2).  Output bound (k values written per
// sample).  A thread keeps the features of four consecutive samples in registers (d <= DREG; up to
// DREG_EXACT features the kernel is compiled for each d); the workgroup's share of the centroids
// (blockIdx.y: `c_chunk` of them, a multiple of 4) is staged in LDS, and the thread walks it four
// centroids at a time: one 128-bit broadcast read per feature, sixteen independent sums, one
// 128-bit store per centroid row.
// ROWS (exact d): X is (n, d); the thread's samples are 4 d consecutive values, and a NaN or an infinity in
// them sets *not_finite; else (d, n).
template <typename T>
constexpr int DREG_EXACT = sizeof(T) == 4 ? 16 : 8;
template <typename T, int DREG, bool ROWS>
__global__ __launch_bounds__(256) void euclidean_distances_reg_kernel(
    const T* __restrict__ X, const T* __restrict__ centroids_t, T* __restrict__ distances_t,
    int32_t* __restrict__ not_finite, int64_t n, int d_, int k, int c_chunk) {
    static_assert(!ROWS || DREG <= DREG_EXACT<T>, "rows are split at compile time");
    const int d = DREG <= DREG_EXACT<T> ? DREG : d_;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* cs = reinterpret_cast<T*>(smem_raw);  // [d][c_chunk]
    const int c_begin = blockIdx.y * c_chunk;
    for (int idx = threadIdx.x; idx < d * c_chunk; idx += 256) {
        const int f = idx / c_chunk, c = c_begin + idx % c_chunk;
        cs[idx] = c < k ? centroids_t[(size_t)f * k + c] : T(0);
    }
    __syncthreads();
    const int64_t n_groups = (n + 3) >> 2;
    const int64_t stride = (int64_t)gridDim.x * 256;
    bool bad = false;
    for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < n_groups; g += stride) {
        const int64_t i0 = g * 4;
        const bool full = i0 + 4 <= n;
        T x[DREG][4];
        if constexpr (ROWS) {
            T flat[DREG][4];  // 128 bits at a time (fp64: twice)
#pragma unroll
            for (int q = 0; q < DREG; ++q) kmx_load4<T>(X + (size_t)i0 * DREG, 4 * q, (n - i0) * DREG, full, flat[q]);
#pragma unroll
            for (int f = 0; f < DREG; ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x[f][r] = flat[(r * DREG + f) / 4][(r * DREG + f) % 4];
                    bad |= kmx_not_finite(x[f][r]);
                }
        } else {
#pragma unroll
            for (int f = 0; f < DREG; ++f) {
                if (f < d) {
                    kmx_load4<T>(X + (size_t)f * n, i0, n, full, x[f]);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[f][r] = T(0);
                }
            }
        }
        for (int c4 = 0; c4 < c_chunk; c4 += 4) {
            T acc[4][4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][r] = T(0);
#pragma unroll
            for (int f = 0; f < DREG; ++f) {
                if (f < d) {
                    T cv[4];
                    lds_load4<T>(cs + f * c_chunk + c4, cv);  // same address in every lane
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const T diff = cv[j] - x[f][r];
                            acc[j][r] = fma(diff, diff, acc[j][r]);
                        }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = c_begin + c4 + j;
                if (c < k) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[j][r] = dist_sqrt(acc[j][r]);
                    kmx_store4<T>(distances_t + (size_t)c * n, i0, n, full, acc[j]);
                }
            }
        }
    }
    if (ROWS && bad) *not_finite = 1;
}

// fp64, any d: a workgroup owns a tile of DT_S samples x DC centroids, a thread a 4 x (DC / 8) block of
// it; the features are staged DT_K at a time through LDS (feature-major arrays: a stage is a copy of
// rows, 128-bit loads), the next stage's loads in flight during the arithmetic.  Per staged feature a
// thread reads its four samples and its centroids from LDS (the centroid reads are broadcasts) and updates
// its sums with a difference and a fused multiply-add each, features in order: vector-ALU bound.
// DC = 64, or 16 for up to 32 clusters: with 10 clusters a tile of 64 is five sixths padding,
// and the kernel took ten times what reading X takes.
constexpr int DT_S = 128, DT_C = 64, DT_C_FEW = 16, DT_K = 16;
constexpr int DT_V = 2;  // elements per 128-bit vector

// 128-bit vectors per thread of a staged tile of COLS columns (fewer vectors than threads: the
// first threads take one)
template <int COLS>
constexpr int dt_vectors() {
    return (DT_K * (COLS / DT_V) + 255) / 256;
}

template <int COLS>
__device__ __forceinline__ void dt_stage_load(double (*regs)[DT_V], const double* __restrict__ base, int64_t len,
                                              int64_t c0, int d, int f0) {
    constexpr int PER_ROW = COLS / DT_V;     // vectors per staged row
    constexpr int N = dt_vectors<COLS>();    // vectors per thread
    // (the same for the whole workgroup: the loads of a stage that exists whole are straight-line code)
    const bool whole = f0 + DT_K <= d && c0 + COLS <= len;
#pragma unroll
    for (int l = 0; l < N; ++l) {
        const int g = threadIdx.x + 256 * l;
        const int f = f0 + g / PER_ROW;
        const int64_t c = c0 + (int64_t)DT_V * (g % PER_ROW);
        const double* __restrict__ src = base + (size_t)f * (size_t)len + c;
        const bool used = g < DT_K * PER_ROW;  // (known at compile time but for a narrow tile)
        if (whole) {
            if (used) {
                const auto v = *reinterpret_cast<const KmxVec<double, DT_V>::type*>(src);
#pragma unroll
                for (int e = 0; e < DT_V; ++e) regs[l][e] = v[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < DT_V; ++e) regs[l][e] = used && f < d && c + e < len ? src[e] : 0.0;
        }
    }
}

template <int COLS>
__device__ __forceinline__ void dt_stage_store(double (*tile)[COLS], const double (*regs)[DT_V]) {
    constexpr int PER_ROW = COLS / DT_V;
    constexpr int N = dt_vectors<COLS>();
#pragma unroll
    for (int l = 0; l < N; ++l) {
        const int g = threadIdx.x + 256 * l;
        if (g < DT_K * PER_ROW) {
#pragma unroll
            for (int e = 0; e < DT_V; ++e) tile[g / PER_ROW][DT_V * (g % PER_ROW) + e] = regs[l][e];
        }
    }
}

// A stage of the samples from the (n, d) array: thread t takes 16 bytes of rows t / 8 + 32 l, and puts
// them feature by feature into the tile (rows of DT_S + 2: the eight lanes of a sample and the four
// samples beside them fall on all banks).
__device__ __forceinline__ void dt_rows_load(double (*regs)[DT_V], const double* __restrict__ X, int64_t n, int64_t i0,
                                             int d, int f0) {
    constexpr int PER_ROW = DT_K / DT_V, N = DT_S * PER_ROW / 256;
    const bool whole = f0 + DT_K <= d && i0 + DT_S <= n;  // (the same for the whole workgroup)
#pragma unroll
    for (int l = 0; l < N; ++l) {
        const int64_t i = i0 + (threadIdx.x + 256 * l) / PER_ROW;
        const int f = f0 + DT_V * (threadIdx.x % PER_ROW);
        const double* __restrict__ src = X + (size_t)i * d + f;
        if (whole) {
            const auto v = *reinterpret_cast<const KmxVec<double, DT_V>::type*>(src);
#pragma unroll
            for (int e = 0; e < DT_V; ++e) regs[l][e] = v[e];
        } else {
#pragma unroll
            for (int e = 0; e < DT_V; ++e) regs[l][e] = i < n && f + e < d ? src[e] : 0.0;
        }
    }
}
__device__ __forceinline__ bool dt_rows_store(double (*tile)[DT_S + 2], const double (*regs)[DT_V]) {
    constexpr int PER_ROW = DT_K / DT_V, N = DT_S * PER_ROW / 256;
    bool bad = false;
#pragma unroll
    for (int l = 0; l < N; ++l)
#pragma unroll
        for (int e = 0; e < DT_V; ++e) {
            tile[DT_V * (threadIdx.x % PER_ROW) + e][(threadIdx.x + 256 * l) / PER_ROW] = regs[l][e];
            bad |= kmx_not_finite(regs[l][e]);
        }
    return bad;
}

// ROWS: X is (n, d), and a NaN or an infinity in it sets *not_finite; else (d, n).
template <int DC, bool ROWS>
__global__ __launch_bounds__(256) void euclidean_distances_tiled_kernel(
    const double* __restrict__ X, const double* __restrict__ centroids_t, double* __restrict__ distances_t,
    int32_t* __restrict__ not_finite, int64_t n, int d, int k) {
    constexpr int CT = DC / 8;  // centroids per thread
    constexpr int XP = ROWS ? DT_S + 2 : DT_S;
    __shared__ __align__(16) double xs[DT_K][XP];
    __shared__ __align__(16) double cs[DT_K][DC];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int64_t i0 = (int64_t)blockIdx.x * DT_S;
    const int c0 = blockIdx.y * DC;
    double rx[dt_vectors<DT_S>()][DT_V], rc[dt_vectors<DC>()][DT_V];
    bool bad = false;
    double acc[CT][4];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][i] = 0.0;

    auto load_x = [&](const int f0) __attribute__((always_inline)) {
        if constexpr (ROWS) dt_rows_load(rx, X, n, i0, d, f0);
        else dt_stage_load<DT_S>(rx, X, n, i0, d, f0);
    };
    load_x(0);
    dt_stage_load<DC>(rc, centroids_t, k, c0, d, 0);
    const int n_stages = (d + DT_K - 1) / DT_K;
    for (int st = 0; st < n_stages; ++st) {
        __syncthreads();  // the previous stage's reads are over
        if constexpr (ROWS) bad |= dt_rows_store(xs, rx);
        else dt_stage_store<DT_S>(xs, rx);
        dt_stage_store<DC>(cs, rc);
        __syncthreads();
        if (st + 1 < n_stages) {
            load_x((st + 1) * DT_K);
            dt_stage_load<DC>(rc, centroids_t, k, c0, d, (st + 1) * DT_K);
        }
        // (rows past d hold zeros on both sides: their differences add nothing)
#pragma unroll
        for (int kk = 0; kk < DT_K; ++kk) {
            double xv[4], cv[CT];
#pragma unroll
            for (int i = 0; i < 4; ++i) xv[i] = xs[kk][4 * tx + i];
#pragma unroll
            for (int c = 0; c < CT; ++c) cv[c] = cs[kk][CT * ty + c];
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double diff = cv[c] - xv[i];
                    acc[c][i] = fma(diff, diff, acc[c][i]);
                }
        }
    }
    if (ROWS && bad) *not_finite = 1;
    const int64_t i = i0 + 4 * tx;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int cc = c0 + CT * ty + c;
        if (cc >= k) continue;
        double* __restrict__ dst = distances_t + (size_t)cc * (size_t)n + i;
        double v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = dist_sqrt(acc[c][e]);
        kmx_store4<double>(dst - i, i, n, i + 4 <= n, v);
    }
}

// ---------------------------------------------------------------------------- fp32 distances
//
// |x - c|^2 = |x - m|^2 + |c - m|^2 - 2 <x - m, c - m> with every term in fp64 (x and c are fp32, so the differences
// and products carry 53 bits), the inner products on the fp64 matrix cores.  m lies among the centroids, as far as
// DM_M features: coordinate by coordinate the median of five of them, which an outlier among them does not move.
// Where the result is less than about d 2^-27 of what it is the difference of, rounding would show in
// fp32: those pairs are redone in the difference form, feature by feature in fp32, as are pairs that
// involve values beyond 2^62 or infinities: a few one after the other (dm_redo_pairs), many of a wave's (two groups
// a thousand times as far apart as they are wide, an offset beyond DM_M features) all at once (dm_redo_wave), and
// a call takes two to four times as long.  What is left is one rounding of the square to fp32 and one of its root:
// relative error at 300 007 x 100, 64 clusters 3.3e-8 root mean square and 8.9e-8 at most, of d rounded additions
// 8.1e-8 and 4.6e-7.
// Why: the difference form costs two vector instructions per pair and feature (98 us for 300 007 x 100 x 64
// at the chip's rate without packed arithmetic), the fp64 matrix cores take 49 us for the same.  And the
// rows of X are read where they are: a transposed copy of X for this one pass over it took 59 us there.
// A workgroup keeps 16 NCT centroids and walks tiles of 128 samples, DM_K features at a time through LDS (the
// operands of up to DM_K features stay there); the next stage's loads are in flight during the arithmetic.
// A wave: two tiles of 16 samples (lane j: samples 2 j and 2 j + 1, so that results leave in pairs).
// ROWS: X is (n, d), and a stage is kept sample by sample (DM_RP: sixteen lanes and four features on 64
// banks); else (d, n) and feature by feature (DM_CP).
// Nothing of the vector work hides behind these matrix instructions, so the end of a tile counts: square
// root from one reciprocal root, one test of a lane's 32 results instead of one each, norms from LDS.
// Bound by the matrix work and the vector work one after the other (34 TFLOP/s at 300 007 x 100, 64 clusters,
// 44 at 1e5 x 784, 300) and, with few features, by the end of a tile.  Kernel times, us, the transposed copy and
// the differences it replaces / this: 300 007 x 100, 64 clusters 178 / 114; 1e5 x 784, 300 clusters 1 340 / 1 065;
// 1e6 x 20, 16 clusters 90 / 60.  Reading the next step's operands ahead of the
// matrix instructions: 292 -> 321 us at 1e6 x 96, 64 clusters (registers), not done.
constexpr int DM_S = 128, DM_K = 32, DM_RP = DM_K + 2, DM_CP = DM_S + 32, DM_M = 1792;
// pairs of a wave, per centroid tile, beyond which it redoes them all at once, and features at a time then (one after the
// other: about 2.5 us a pair of 100 features; at once: 18 us for one tile of centroids, 65 for four)
constexpr int DM_REDO = 5, DM_R = 8;
typedef double dm_v4d __attribute__((ext_vector_type(4)));

// The median of five values, 0 where it is not finite.
__device__ __forceinline__ double dm_middle(const float (&v)[5]) {
    const float low = fmaxf(fminf(v[0], v[1]), fminf(v[2], v[3]));
    const float high = fminf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
    // (of the four, low and high are the middle ones, in either order)
    const float middle = __builtin_amdgcn_fmed3f(v[4], low, high);
    return kmx_not_finite(middle) ? 0.0 : (double)middle;
}

// The pairs of a wave that `redo` names (bit 8 tile + 2 r + b of lane (g, j): centroid c0 + 16 tile + g + 4 r, sample
// 2 j + b of the wave) in the difference form, features in order.  A few of them: one after the other, a feature per lane,
// 256 features' loads in flight; the lanes' differences are then added up in their order.
template <bool ROWS>
__device__ __forceinline__ void dm_redo_pairs(const float* __restrict__ X, const float* __restrict__ centroids_t,
                                              float* __restrict__ distances_t, unsigned int redo, int64_t i0, int here,
                                              int c0, int64_t n, int d, int k, int lane, int wave) {
    asm volatile("" : "+v"(lane));  // (what follows from it is made here, not kept over the tiles)
    for (unsigned long long lanes = __ballot(redo != 0u); lanes != 0ull; lanes = __ballot(redo != 0u)) {
        const int from = __builtin_ctzll(lanes), u = __builtin_ctz((unsigned int)__builtin_amdgcn_readlane((int)redo, from));
        if (lane == from) redo &= redo - 1u;
        const int c = c0 + 16 * (u >> 3) + (from >> 4) + 4 * ((u >> 1) & 3), si = 32 * wave + 2 * (from & 15) + (u & 1);
        if (c >= k || si >= here) continue;
        float sum = 0.0f;
        for (int f0 = 0; f0 < d; f0 += 256) {
            float diff[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int fi = f0 + 64 * q + lane, f = fi < d ? fi : d - 1;
                diff[q] = 0.0f;
                if (f0 + 64 * q < d) {
                    const float x = ROWS ? X[(size_t)(i0 + si) * d + f] : X[(size_t)f * n + i0 + si];
                    diff[q] = fi < d ? centroids_t[(size_t)f * k + c] - x : 0.0f;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                for (int l = 0; l < 64 && f0 + 64 * q + l < d; l += 16)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(diff[q]), l + e));
                        sum = fmaf(v, v, sum);
                    }
        }
        if (lane == 0) distances_t[(size_t)c * n + i0 + si] = dist_sqrt(sum);
    }
}

// Many of them: all the wave's pairs, DM_R features at a time through `own`, the part of xs that only this wave reads (its
// samples'; rows of 32 floats): [feature][sample], then [feature][g][tile][r] of the centroids.  Bound by its loads'
// latency.  300 007 x 100, 64 clusters in two groups (half of all pairs): 315 us, 1 630 with each lane on its own pairs;
// 121 with none to redo.
template <int NCT, bool ROWS>
__device__ __forceinline__ void dm_redo_wave(const float* __restrict__ X, const float* __restrict__ centroids_t,
                                             float* __restrict__ distances_t, float* own, unsigned int redo, int64_t i0,
                                             int here, int c0, int64_t n, int d, int k, int lane, int wave) {
    asm volatile("" : "+v"(lane));  // (what follows from it is made here, not kept over the tiles)
    constexpr int PITCH = ROWS ? 36 : DM_CP;
    constexpr int NA = NCT > 2 ? 2 : NCT, CW = 16 * NA;  // NA tiles of centroids at a time (registers)
    static_assert(ROWS ? PITCH * (DM_R + DM_R * CW / 32) <= 32 * DM_RP : DM_R + DM_R * CW / 32 <= DM_K, "fits xs");
    const int s0 = 32 * wave, g = lane >> 4, j = lane & 15;
    for (int a0 = 0; a0 < NCT; a0 += NA) {
        const int c00 = c0 + 16 * a0;
        float sum[NA][4][2];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[a][r][0] = sum[a][r][1] = 0.0f;
        for (int f0 = 0; f0 < d; f0 += DM_R) {
            float xv[DM_R / 2], cv[DM_R * CW / 64];
#pragma unroll
            for (int p = 0; p < DM_R / 2; ++p) {
                const int u = lane + 64 * p, fi = f0 + (ROWS ? u % DM_R : u / 32), si = s0 + (ROWS ? u / DM_R : u % 32);
                const int s = si < here ? si : here - 1, f = fi < d ? fi : d - 1;
                xv[p] = ROWS ? X[(size_t)(i0 + s) * d + f] : X[(size_t)f * n + i0 + s];
            }
#pragma unroll
            for (int p = 0; p < DM_R * CW / 64; ++p) {
                const int u = lane + 64 * p, fi = f0 + u / CW, c = c00 + u % CW;
                cv[p] = centroids_t[(size_t)(fi < d ? fi : d - 1) * k + (c < k ? c : k - 1)];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads of the previous stage are over
#pragma unroll
            for (int p = 0; p < DM_R / 2; ++p) {
                const int u = lane + 64 * p;
                own[(ROWS ? u % DM_R : u / 32) * PITCH + (ROWS ? u / DM_R : u % 32)] = xv[p];
            }
#pragma unroll
            for (int p = 0; p < DM_R * CW / 64; ++p) {
                const int u = lane + 64 * p, c = u % CW, at = u / CW * CW + (c & 3) * 4 * NA + (c >> 4) * 4 + (c >> 2 & 3);
                own[(DM_R + at / 32) * PITCH + at % 32] = cv[p];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const int w = d - f0 < DM_R ? d - f0 : DM_R;
            for (int f = 0; f < w; ++f) {
                const float2 x = *reinterpret_cast<const float2*>(own + f * PITCH + 2 * j);
#pragma unroll
                for (int a = 0; a < NA; ++a) {
                    float c[4];
                    const int at = f * CW + g * 4 * NA + 4 * a;
                    lds_load4<float>(own + (DM_R + at / 32) * PITCH + at % 32, c);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float d0 = c[r] - x.x, d1 = c[r] - x.y;
                        sum[a][r][0] = fmaf(d0, d0, sum[a][r][0]);
                        sum[a][r][1] = fmaf(d1, d1, sum[a][r][1]);
                    }
                }
            }
        }
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const int c = c00 + 16 * a + g + 4 * r, si = s0 + 2 * j + b;
                    if ((redo >> (8 * (a0 + a) + 2 * r + b) & 1u) && c < k && si < here)
                        distances_t[(size_t)c * n + i0 + si] = dist_sqrt(sum[a][r][b]);
                }
    }
}

template <int NCT, bool ROWS>
__global__ __launch_bounds__(256, 3) void distances_f32_kernel(
    const float* __restrict__ X, const float* __restrict__ centroids_t, float* __restrict__ distances_t,
    int32_t* __restrict__ not_finite, int64_t n, int d, int k, int c_tiles, int slots) {
    constexpr int PX = DM_S * DM_K / 256;            // values of X per thread and stage
    constexpr int PC = NCT * 64 * (DM_K / 4) / 256;  // centroid values per thread and stage
    __shared__ __align__(16) float xs[ROWS ? DM_S * DM_RP : DM_K * DM_CP];
    __shared__ double cf[DM_K / 4][NCT][64];  // operand fragments
    __shared__ double ms[DM_M + DM_K];        // m
    __shared__ double cn[4][16 * NCT];        // |c - m|^2: the waves' parts, then the sums in row 0
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = lane >> 4, j = lane & 15;
    // workgroup b: die b % 8, centroid tile (b / 8) % c_tiles, and of the die's sample tiles every slots-th:
    // the workgroups that read the same samples run on one die, next to each other in time
    const int c0 = (int)(blockIdx.x / 8 % c_tiles) * 16 * NCT;
    const int64_t s_step = (int64_t)slots * 8, n_tiles = (n + DM_S - 1) / DM_S;
    int64_t tile = (int64_t)(blockIdx.x / 8 / c_tiles) * 8 + blockIdx.x % 8;
    if (tile >= n_tiles) return;

    float rx[PX], rc[PC];
    bool bad = false;
    auto load = [&](const int64_t i0, const int f0, const bool centroids) __attribute__((always_inline)) {
        const int here = n - i0 < DM_S ? (int)(n - i0) : DM_S;  // samples of the tile that exist
        const int w = d - f0 < DM_K ? d - f0 : DM_K;            // features of the stage
        const bool whole = w == DM_K && here == DM_S;
        if constexpr (ROWS) {
            if (whole) {
#pragma unroll
                for (int p = 0; p < PX / 4; ++p) {
                    const int s = (threadIdx.x >> 3) + 32 * p, q = threadIdx.x & 7;
                    const auto v = *reinterpret_cast<const KmxVec<float, 4>::type*>(X + (size_t)(i0 + s) * d + f0 + 4 * q);
#pragma unroll
                    for (int e = 0; e < 4; ++e) rx[4 * p + e] = v[e];
                }
            } else {
                // the values one after the other (of up to DM_K features: whole cache lines); past the end
                // the last sample's, dropped when they are stored
                const int step_s = 256 / w, step_f = 256 - step_s * w;
                int s = (int)threadIdx.x / w, f = (int)threadIdx.x - s * w;
                asm volatile("" : "+v"(s), "+v"(f));  // (recomputed per stage instead of a register per value)
                const float* __restrict__ from = X + (size_t)i0 * d + f0;
#pragma unroll
                for (int p = 0; p < PX; ++p) {
                    if (256 * p < DM_S * w) rx[p] = from[(size_t)(s < here ? s : here - 1) * d + f];  // (uniform)
                    s += step_s;
                    f += step_f;
                    if (f >= w) {
                        f -= w;
                        ++s;
                    }
                }
            }
        } else if (whole) {
#pragma unroll
            for (int p = 0; p < PX / 4; ++p) {
                const int f = (threadIdx.x >> 5) + 8 * p, s = 4 * (threadIdx.x & 31);
                const auto v = *reinterpret_cast<const KmxVec<float, 4>::type*>(X + (size_t)(f0 + f) * n + i0 + s);
#pragma unroll
                for (int e = 0; e < 4; ++e) rx[4 * p + e] = v[e];
            }
        } else {
#pragma unroll
            for (int p = 0; p < PX / 4; ++p) {
                const int f = (threadIdx.x >> 5) + 8 * p, s = 4 * (threadIdx.x & 31);
                const float* __restrict__ row = X + (size_t)(f < w ? f0 + f : d - 1) * n + i0;
#pragma unroll
                for (int e = 0; e < 4; ++e) rx[4 * p + e] = row[s + e < here ? s + e : here - 1];
            }
        }
        // fragment value (step, tile, lane): feature f0 + 4 step + lane / 16 of centroid c0 + 16 tile + lane % 16
        // (a thread's values are all of one centroid)
        if (centroids) {
            int c = c0 + 16 * (wave % NCT) + j;
            asm volatile("" : "+v"(c));
#pragma unroll
            for (int p = 0; p < PC; ++p) {
                const int f = f0 + 4 * ((wave + 4 * p) / NCT) + g;
                rc[p] = centroids_t[(size_t)(f < d ? f : d - 1) * k + (c < k ? c : k - 1)];
            }
        }
    };
    double my_nc = 0.0;
    auto store = [&](const int64_t i0, const int f0, const bool centroids, const bool first) __attribute__((always_inline)) {
        const int here = n - i0 < DM_S ? (int)(n - i0) : DM_S;
        const int w = d - f0 < DM_K ? d - f0 : DM_K;
        if (ROWS && !(w == DM_K && here == DM_S)) {
            const int step_s = 256 / w, step_f = 256 - step_s * w;
            int s = (int)threadIdx.x / w, f = (int)threadIdx.x - s * w;
            asm volatile("" : "+v"(s), "+v"(f));
#pragma unroll
            for (int p = 0; p < PX; ++p) {
                if (256 * p < DM_S * w && s < DM_S) {
                    xs[s * DM_RP + f] = rx[p];
                    bad |= kmx_not_finite(rx[p]);
                }
                s += step_s;
                f += step_f;
                if (f >= w) {
                    f -= w;
                    ++s;
                }
            }
            // (features up to the next step of four: zero, as the fragments are)
            const int fill = -w & 3;
            for (int u = threadIdx.x; u < DM_S * fill; u += 256) xs[u / fill * DM_RP + w + u % fill] = 0.0f;
        } else if constexpr (ROWS) {
#pragma unroll
            for (int p = 0; p < PX / 4; ++p) {
                const int s = (threadIdx.x >> 3) + 32 * p, q = threadIdx.x & 7;
                float2* at = reinterpret_cast<float2*>(xs + s * DM_RP + 4 * q);
                at[0] = make_float2(rx[4 * p], rx[4 * p + 1]);
                at[1] = make_float2(rx[4 * p + 2], rx[4 * p + 3]);
            }
#pragma unroll
            for (int p = 0; p < PX; ++p) bad |= kmx_not_finite(rx[p]);
        } else {
#pragma unroll
            for (int p = 0; p < PX / 4; ++p) {
                const int f = (threadIdx.x >> 5) + 8 * p;
                float4 v = make_float4(rx[4 * p], rx[4 * p + 1], rx[4 * p + 2], rx[4 * p + 3]);
                if (f >= w) v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                *reinterpret_cast<float4*>(xs + f * DM_CP + 4 * (threadIdx.x & 31)) = v;
            }
        }
        if (centroids) {
            int c = c0 + 16 * (wave % NCT) + j;
            asm volatile("" : "+v"(c));
            const double* m_at = ms + (f0 < DM_M ? f0 : DM_M) + g;
#pragma unroll
            for (int p = 0; p < PC; ++p) {
                const int st = (wave + 4 * p) / NCT, f = 4 * st + g;
                double v = (double)rc[p] - m_at[4 * st];
                v = f < w && c < k ? v : 0.0;
                cf[st][wave % NCT][lane] = v;
                if (first) my_nc = fma(v, v, my_nc);
            }
        }
    };

    const bool resident = d <= DM_K;  // the operands of all features stay in LDS
    bool first = true;
    load(tile * DM_S, 0, true);
    // (zero for the features past d, and for the stages past DM_M)
    {
        // m: the median of the last five centroids (kmeans++ takes outliers early; in a row they are two loads)
        constexpr int P = DM_M / 256;
        const int most = d < DM_M ? d : DM_M;
        float v[P][5];
        if (k >= 5) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (256 * p >= most) break;  // (uniform)
                const int f = threadIdx.x + 256 * p;
                const float* __restrict__ row = centroids_t + (size_t)(f < most ? f : most - 1) * k + k - 5;
                const auto q = *reinterpret_cast<const KmxVec<float, 4>::type*>(row);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[p][i] = q[i];
                v[p][4] = row[4];
            }
        } else {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int f = threadIdx.x + 256 * p;
#pragma unroll
                for (int i = 0; i < 5; ++i) v[p][i] = centroids_t[(size_t)(f < most ? f : most - 1) * k + (i < k ? i : k - 1)];
            }
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int f = threadIdx.x + 256 * p;
            if (256 * p < most + DM_K) ms[f] = f < most ? dm_middle(v[p]) : 0.0;
        }
        if (threadIdx.x < DM_K) ms[DM_M + threadIdx.x] = 0.0;
    }
    for (; tile < n_tiles; tile += s_step) {
        const int64_t i0 = tile * DM_S, i_next = (tile + s_step) * DM_S;
        dm_v4d acc[NCT][2];
        double nx[2] = {0.0, 0.0};
#pragma unroll
        for (int a = 0; a < NCT; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = dm_v4d{0.0, 0.0, 0.0, 0.0};
        for (int f0 = 0; f0 < d; f0 += DM_K) {
            const bool last_stage = f0 + DM_K >= d;
            __syncthreads();  // the previous stage's reads are over
            store(i0, f0, first || !resident, first);
            if (first && last_stage) {
                // (the threads of a centroid: four lanes of the waves that hold its tile)
                double v = my_nc;
                v += __shfl_xor(v, 16, 64);
                v += __shfl_xor(v, 32, 64);
                if (g == 0) cn[wave / NCT][16 * (wave % NCT) + j] = v;
            }
            __syncthreads();
            if (!last_stage || tile + s_step < n_tiles)
                load(last_stage ? i_next : i0, last_stage ? 0 : f0 + DM_K, !resident);
            const int steps = (d - f0 < DM_K ? d - f0 + 3 : DM_K) / 4;
            const double* m_here = ms + (f0 < DM_M ? f0 : DM_M) + g;
#pragma unroll 1
            for (int st = 0; st < steps; ++st) {
                const double m = m_here[4 * st];
                double xb[2];
                if constexpr (ROWS) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) xb[b] = (double)xs[(32 * wave + 2 * j + b) * DM_RP + 4 * st + g] - m;
                } else {
                    const float2 v = *reinterpret_cast<const float2*>(xs + (4 * st + g) * DM_CP + 32 * wave + 2 * j);
                    xb[0] = (double)v.x - m;
                    xb[1] = (double)v.y - m;
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) nx[b] = fma(xb[b], xb[b], nx[b]);
#pragma unroll
                for (int a = 0; a < NCT; ++a) {
                    const double av = cf[st][a][lane];
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, xb[b], acc[a][b], 0, 0, 0);
                }
            }
        }
        if (first && NCT < 4) {
            if (threadIdx.x < 16 * NCT) {
                double v = 0.0;
#pragma unroll
                for (int q = 0; q < 4 / NCT; ++q) v += cn[q][threadIdx.x];
                cn[0][threadIdx.x] = v;
            }
            __syncthreads();
        }
        first = false;

        // the four lanes that share a sample
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1)
#pragma unroll
            for (int b = 0; b < 2; ++b) nx[b] += __shfl_xor(nx[b], off, 64);
        // accumulator r of lane (g, j): centroid 16 a + g + 4 r, samples 2 j + b of the wave
        const int here = n - i0 < DM_S ? (int)(n - i0) : DM_S;
        const int sl = 32 * wave + 2 * j;
        // a result's high word less that of what it is the difference of: how many binades it lost (20 bits
        // each); its least over the lane's results, the largest norm and the least result decide at once
        // (norms as unsigned words: infinities and NaN of either sign are the largest)
        auto binades_lost = [](const double sq, const double of) __attribute__((always_inline)) {
            return (int)((unsigned int)__double2hiint(sq) - (unsigned int)__double2hiint(of));
        };
        auto norm_word = [](const double v) __attribute__((always_inline)) { return (unsigned int)__double2hiint(v); };
        int least = 0x7fffffff;
        unsigned int most = max(norm_word(nx[0]), norm_word(nx[1]));
        float low = kmx_inf<float>();
        auto finish = [&](auto whole_tag) __attribute__((always_inline)) {
            constexpr bool whole = decltype(whole_tag)::value;
            float* __restrict__ dst = distances_t + (size_t)(c0 + g) * n + i0 + sl;
            int c = c0 + g;
#pragma unroll
            for (int a = 0; a < NCT; ++a) {
                __builtin_amdgcn_sched_barrier(0);  // (four norms at a time in registers)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double c2 = cn[0][16 * a + g + 4 * r];
                    most = max(most, norm_word(c2));
                    float v[2];
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const double of = nx[b] + c2, sq = fma(-2.0, acc[a][b][r], of);
                        least = min(least, binades_lost(sq, of));
                        const float q = (float)sq;
                        low = fminf(low, q);
                        // root by one reciprocal root and a Newton step on the residual
                        const float y = __builtin_amdgcn_rsqf(q), t = q * y;
                        v[b] = fmaf(fmaf(-t, t, q), 0.5f * y, t);
                    }
                    // (the running extremes now, not as a tree over 32 results kept to the end)
                    asm volatile("" : "+v"(least), "+v"(most), "+v"(low));
                    if (c < k && (whole || sl + 1 < here))
                        *reinterpret_cast<KmxVec<float, 2>::type*>(dst) = KmxVec<float, 2>::type{v[0], v[1]};
                    else if (!whole && c < k && sl < here)
                        dst[0] = v[0];
                    dst += 4 * n;
                    c += 4;
                }
            }
        };
        if (here == DM_S) finish(std::true_type{});  // (uniform)
        else finish(std::false_type{});
        // d 2^-27, in binades; 2^126: no square beyond it overflows; 1e-30: roots and their residuals are normal
        const int lost = (26 - (31 - __builtin_clz(d))) << 20;
        if (__any(least + lost <= 0 || most >= 0x47d00000u || !(low >= 1e-30f))) {
            unsigned int redo = 0u;
            asm volatile("" : "+v"(nx[0]), "+v"(nx[1]) : : "memory");  // (computed again, not kept in registers since above)
#pragma unroll
            for (int a = 0; a < NCT; ++a) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double c2 = cn[0][16 * a + g + 4 * r];
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const double of = nx[b] + c2, sq = fma(-2.0, acc[a][b][r], of);
                        if (!(binades_lost(sq, of) + lost > 0 && of < 0x1p126 && (float)sq >= 1e-30f))
                            redo |= 1u << (8 * a + 2 * r + b);
                    }
                }
            }
            if (kmx_wave_sum<int>(__popc(redo)) > DM_REDO * NCT)
                dm_redo_wave<NCT, ROWS>(X, centroids_t, distances_t, xs + 32 * wave * (ROWS ? DM_RP : 1), redo, i0, here, c0,
                                        n, d, k, lane, wave);
            else
                dm_redo_pairs<ROWS>(X, centroids_t, distances_t, redo, i0, here, c0, n, d, k, lane, wave);
        }
    }
    if (ROWS && bad) *not_finite = 1;
}

// One workgroup per relocated cluster, threads over features.  Several relocations may take
// samples from the same old cluster, hence the atomic subtraction.  sq_dist (or null): nothing is
// moved if the first sample, the farthest, has no distance above zero.
template <typename T>
__global__ __launch_bounds__(256) void relocate_kernel(
    const T* __restrict__ X_t, const T* __restrict__ sample_weight,
    const uint32_t* __restrict__ labels, const int64_t* __restrict__ far_samples,
    const uint32_t* __restrict__ empty_clusters, T* __restrict__ per_sample_inertia,
    T* __restrict__ sums_t, T* __restrict__ sizes, const T* __restrict__ sq_dist, int64_t n, int d, int k) {
    const int r = blockIdx.x;
    if (sq_dist != nullptr && !(sq_dist[far_samples[0]] > T(0))) return;
    const uint32_t cluster = empty_clusters[r];
    const int64_t sample = far_samples[r];
    const uint32_t old = labels[sample];
    const T w = sample_weight[sample];
    for (int f = threadIdx.x; f < d; f += 256) {
        const T addend = X_t[(size_t)f * n + sample] * w;
        kmx_atomic_add(sums_t + (size_t)f * k + old, -addend);
        sums_t[(size_t)f * k + cluster] = addend;
    }
    if (threadIdx.x == 0) {
        if (per_sample_inertia) per_sample_inertia[sample] = T(0);
        kmx_atomic_add(sizes + old, -w);
        sizes[cluster] = w;
    }
}

int stream_grid(int64_t n);
// fp64 partial sums a launch of the summing kernel may write: eight per compute unit, or one per
// workgroup of its first grid dimension where that is more
int64_t inertia_partial_slots(int64_t n) {
    const int64_t a = (int64_t)kmx_num_cus() * 8, b = stream_grid(kmx_cdiv(n, 4));
    return a > b ? a : b;
}

int stream_grid(int64_t n) {
    int64_t blocks = kmx_cdiv(n, 256);
    const int64_t cap = (int64_t)kmx_num_cus() * 8;
    if (blocks > cap) blocks = cap;
    return (int)(blocks < 1 ? 1 : blocks);
}

}  // namespace

int32_t kmx_inertia_total_launch(const double* partial, int count, void* out, int32_t dtype, hipStream_t stream) {
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((inertia_total_kernel<float>), dim3(1), dim3(256), 0, stream, partial, count, (float*)out);
    else
        hipLaunchKernelGGL((inertia_total_kernel<double>), dim3(1), dim3(256), 0, stream, partial, count, (double*)out);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

namespace {
__global__ void clear_word_kernel(int32_t* word) {
    if (threadIdx.x == 0) *word = 0;
}

// The register kernel for d features: DREG = 16 (any d up to it) or DREG = d.  Its centroid range is split over
// blockIdx.y until there are about six workgroups per compute unit (a thread's walk over the centroids
// is one dependent chain).
template <typename T, int DREG, bool ROWS>
int32_t launch_distances_reg(const void* X, const void* centroids_t, void* distances_t, int32_t* not_finite, int64_t n,
                             int d, int k, hipStream_t stream) {
    if constexpr (DREG <= DREG_EXACT<T> && DREG > 1) {
        if (d < DREG)
            return launch_distances_reg<T, DREG - 1, ROWS>(X, centroids_t, distances_t, not_finite, n, d, k, stream);
    }
    const int64_t wgx = stream_grid(kmx_cdiv(n, 4));
    int64_t gy = kmx_cdiv((int64_t)kmx_num_cus() * 6, wgx);
    if (gy > kmx_cdiv(k, 16)) gy = kmx_cdiv(k, 16);
    if (gy < 1) gy = 1;
    int c_chunk = (int)(4 * kmx_cdiv(kmx_cdiv(k, gy), 4));
    const int most = (int)(64 * 1024 / (d * sizeof(T))) & ~3;  // (the share within 64 KB of LDS)
    if (c_chunk > most) c_chunk = most;
    gy = kmx_cdiv(k, c_chunk);
    if (gy > 65535) return KMX_ERR_BAD_SHAPE;
    hipLaunchKernelGGL((euclidean_distances_reg_kernel<T, DREG, ROWS>), dim3((unsigned)wgx, (unsigned)gy), dim3(256),
                       (size_t)d * c_chunk * sizeof(T), stream, (const T*)X, (const T*)centroids_t, (T*)distances_t,
                       not_finite, n, d, k, c_chunk);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

template <bool ROWS>
int32_t launch_distances_f32(const void* X, const void* centroids_t, void* distances_t, int32_t* not_finite, int64_t n,
                             int d, int k, hipStream_t stream) {
    // few features: the differences are fewer instructions than what the end of a tile takes on the matrix cores
    // (transform of 1e6 x d by k clusters, us, matrix cores / registers: d 3 k 5 87 / 57, d 8 k 64 127 / 112,
    // d 9 k 64 133 / 113, d 9 k 5 94 / 64, and the copy and differences both took 79, 136, 142, 87 before)
    if (d <= DREG_EXACT<float>)
        return launch_distances_reg<float, DREG_EXACT<float>, ROWS>(X, centroids_t, distances_t, not_finite, n, d, k, stream);
    const int nct = k <= 16 ? 1 : k <= 32 ? 2 : 4;
    const int64_t c_tiles = kmx_cdiv(k, 16 * nct), groups = kmx_cdiv(kmx_cdiv(n, DM_S), 8);
    // as many workgroups as run at once, each on one centroid tile
    int64_t slots = (int64_t)3 * kmx_num_cus() / (8 * c_tiles);
    if (slots < 1) slots = 1;
    if (slots > groups) slots = groups;
    if (c_tiles * slots > INT32_MAX / 8) return KMX_ERR_BAD_SHAPE;
#define KMX_DIST_F32(NCT)                                                                                         \
    hipLaunchKernelGGL((distances_f32_kernel<NCT, ROWS>), dim3((unsigned)(8 * c_tiles * slots)), dim3(256), 0,    \
                       stream, (const float*)X, (const float*)centroids_t, (float*)distances_t, not_finite, n, d, \
                       k, (int)c_tiles, (int)slots)
    if (nct == 1) KMX_DIST_F32(1); else if (nct == 2) KMX_DIST_F32(2); else KMX_DIST_F32(4);
#undef KMX_DIST_F32
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

template <bool ROWS>
int32_t launch_distances_f64(const void* X, const void* centroids_t, void* distances_t, int32_t* not_finite, int64_t n,
                             int d, int k, hipStream_t stream) {
    if (d <= DREG_EXACT<double>)
        return launch_distances_reg<double, DREG_EXACT<double>, ROWS>(X, centroids_t, distances_t, not_finite, n, d, k, stream);
    if constexpr (!ROWS) {
        if (d <= 16) return launch_distances_reg<double, 16, ROWS>(X, centroids_t, distances_t, not_finite, n, d, k, stream);
    }
    const int dc = k <= 2 * DT_C_FEW ? DT_C_FEW : DT_C;
    const dim3 grid((unsigned)kmx_cdiv(n, DT_S), (unsigned)kmx_cdiv(k, dc));
#define KMX_DIST_TILED(DC)                                                                                          \
    hipLaunchKernelGGL((euclidean_distances_tiled_kernel<DC, ROWS>), grid, dim3(256), 0, stream,            \
                       (const double*)X, (const double*)centroids_t, (double*)distances_t, not_finite, n, d, k)
    if (dc == DT_C_FEW) KMX_DIST_TILED(DT_C_FEW); else KMX_DIST_TILED(DT_C);
#undef KMX_DIST_TILED
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}
}  // namespace

extern "C" {

static int32_t inertia_launch(const void* X_t, const void* sample_weight, const void* centroids_t,
                              const uint32_t* labels, void* out, double* partial, int64_t n, int32_t d, int32_t k,
                              int32_t dtype, hipStream_t stream) {
    const bool sum = partial != nullptr;
    const int grid = stream_grid(kmx_cdiv(n, 4));
    const size_t es = kmx_dtype_size(dtype);
    // the sum over few samples of many features: the features split over the second grid dimension
    // until there are about four workgroups per compute unit (and at least 16 features each)
    int gy = 1;
    if (sum) {
        gy = (int)kmx_cdiv((int64_t)kmx_num_cus() * 4, grid);
        if (gy > d / 16) gy = d / 16;
        if ((int64_t)gy * grid > inertia_partial_slots(n)) gy = (int)(inertia_partial_slots(n) / grid);
        if (gy < 1) gy = 1;
    }
    const int f_chunk = (int)kmx_cdiv(d, gy);
    const size_t lds = (size_t)f_chunk * k * es;
    const bool in_lds = lds <= 48 * 1024;
#define KMX_INERTIA(T, L, S)                                                                       \
    hipLaunchKernelGGL((per_sample_inertia_kernel<T, L, S>), dim3(grid, gy), dim3(256), (L) ? lds : 0,  \
                       stream, (const T*)X_t, (const T*)sample_weight, (const T*)centroids_t,      \
                       labels, (S) ? nullptr : (T*)out, partial, n, d, k)
#define KMX_INERTIA_T(T)                                                        \
    do {                                                                        \
        if (in_lds && sum) KMX_INERTIA(T, true, true);                          \
        else if (in_lds) KMX_INERTIA(T, true, false);                           \
        else if (sum) KMX_INERTIA(T, false, true);                              \
        else KMX_INERTIA(T, false, false);                                      \
    } while (0)
    if (dtype == KMX_F32) KMX_INERTIA_T(float); else KMX_INERTIA_T(double);
#undef KMX_INERTIA_T
#undef KMX_INERTIA
    if (sum) {
        if (dtype == KMX_F32)
            hipLaunchKernelGGL((inertia_total_kernel<float>), dim3(1), dim3(256), 0, stream, partial, grid * gy, (float*)out);
        else
            hipLaunchKernelGGL((inertia_total_kernel<double>), dim3(1), dim3(256), 0, stream, partial, grid * gy, (double*)out);
    }
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_per_sample_inertia(const void* X_t, const void* sample_weight, const void* centroids_t,
                               const uint32_t* labels, void* out, int64_t n, int32_t d, int32_t k,
                               int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(centroids_t);
    KMX_REQUIRE_PTR(labels);
    KMX_REQUIRE_PTR(out);
    if (n <= 0 || d <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    return inertia_launch(X_t, sample_weight, centroids_t, labels, out, nullptr, n, d, k, dtype, (hipStream_t)stream_);
}

size_t kmx_inertia_workspace_bytes(int64_t n) {
    if (n <= 0) return 0;
    return kmx_align256((size_t)inertia_partial_slots(n) * sizeof(double));
}

int32_t kmx_inertia(const void* X_t, const void* sample_weight, const void* centroids_t, const uint32_t* labels,
                    void* out_total, void* workspace, size_t workspace_bytes, int64_t n, int32_t d, int32_t k,
                    int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(centroids_t);
    KMX_REQUIRE_PTR(labels);
    KMX_REQUIRE_PTR(out_total);
    KMX_REQUIRE_PTR(workspace);
    if (n <= 0 || d <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    if (workspace_bytes < kmx_inertia_workspace_bytes(n)) return KMX_ERR_WORKSPACE;
    return inertia_launch(X_t, sample_weight, centroids_t, labels, out_total, (double*)workspace, n, d, k, dtype,
                          (hipStream_t)stream_);
}

}  // extern "C"

// (the feature-major kernel keeps its stretch of the centroids in LDS if that takes up to 48 KB)
bool kmx_inertia_in_lds(int64_t n, int d, int k, int dtype) {
    const int grid = stream_grid(kmx_cdiv(n, 4));
    int64_t gy = kmx_cdiv((int64_t)kmx_num_cus() * 4, grid);
    if (gy > d / 16) gy = d / 16;
    if (gy < 1) gy = 1;
    return (size_t)kmx_cdiv(d, gy) * k * kmx_dtype_size(dtype) <= 48 * 1024;
}

int32_t kmx_inertia_rows(const void* X_rowmajor, const void* sample_weight, const void* cpack, const uint32_t* labels,
                         void* out, double* workspace, int64_t n, int d, int dpad, int dtype, hipStream_t stream) {
    int64_t grid = kmx_cdiv(n, 32);
    const int64_t cap = workspace != nullptr ? inertia_partial_slots(n) : 65536;
    if (grid > 8 * (int64_t)kmx_num_cus()) grid = 8 * (int64_t)kmx_num_cus();
    if (grid > cap) grid = cap;
    const size_t es = kmx_dtype_size(dtype);
    const bool whole = (size_t)d * es % 16 == 0;
#define KMX_ROWS_INERTIA(T, V, S)                                                                                     \
    hipLaunchKernelGGL((rows_inertia_kernel<T, V, S>), dim3((unsigned)grid), dim3(256), 0, stream, (const T*)X_rowmajor, \
                       (const T*)sample_weight, (const T*)cpack, labels, (S) ? nullptr : (T*)out, workspace, n, d, dpad)
#define KMX_ROWS_INERTIA_T(T)                                                  \
    do {                                                                       \
        if (whole && workspace) KMX_ROWS_INERTIA(T, true, true);                 \
        else if (whole) KMX_ROWS_INERTIA(T, true, false);                        \
        else if (workspace) KMX_ROWS_INERTIA(T, false, true);                  \
        else KMX_ROWS_INERTIA(T, false, false);                                \
    } while (0)
    if (dtype == KMX_F32) KMX_ROWS_INERTIA_T(float); else KMX_ROWS_INERTIA_T(double);
#undef KMX_ROWS_INERTIA_T
#undef KMX_ROWS_INERTIA
    if (workspace != nullptr) return kmx_inertia_total_launch(workspace, (int)grid, out, dtype, stream);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

extern "C" {

int32_t kmx_euclidean_distances(const void* X_t, const void* centroids_t, void* distances_t,
                                int64_t n, int32_t d, int32_t k, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(centroids_t);
    KMX_REQUIRE_PTR(distances_t);
    if (n <= 0 || d <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    return dtype == KMX_F32 ? launch_distances_f32<false>(X_t, centroids_t, distances_t, nullptr, n, d, k, stream)
                            : launch_distances_f64<false>(X_t, centroids_t, distances_t, nullptr, n, d, k, stream);
}

int32_t kmx_euclidean_distances_rows(const void* X, const void* centroids_t, void* distances_t, int32_t* not_finite,
                                     int64_t n, int32_t d, int32_t k, int32_t dtype, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X);
    KMX_REQUIRE_PTR(centroids_t);
    KMX_REQUIRE_PTR(distances_t);
    KMX_REQUIRE_PTR(not_finite);
    if (n <= 0 || d <= 0 || k <= 0) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    hipStream_t stream = (hipStream_t)stream_;
    hipLaunchKernelGGL(clear_word_kernel, dim3(1), dim3(64), 0, stream, not_finite);
    return dtype == KMX_F32 ? launch_distances_f32<true>(X, centroids_t, distances_t, not_finite, n, d, k, stream)
                            : launch_distances_f64<true>(X, centroids_t, distances_t, not_finite, n, d, k, stream);
}

static int32_t relocate(const void* X_t, const void* sample_weight, const uint32_t* labels, const int64_t* far_samples,
                        const uint32_t* empty_clusters, int32_t n_relocated, void* per_sample_inertia, void* sums_t,
                        void* cluster_sizes, const void* sq_dist, int64_t n, int32_t d, int32_t k, int32_t dtype,
                        void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(sample_weight);
    KMX_REQUIRE_PTR(labels);
    KMX_REQUIRE_PTR(far_samples);
    KMX_REQUIRE_PTR(empty_clusters);
    KMX_REQUIRE_PTR(sums_t);
    KMX_REQUIRE_PTR(cluster_sizes);
    if (n <= 0 || d <= 0 || k <= 0 || n_relocated < 0 || n_relocated > k) return KMX_ERR_BAD_SHAPE;
    KMX_REQUIRE_DTYPE(dtype);
    if (n_relocated == 0) return KMX_OK;
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((relocate_kernel<float>), dim3(n_relocated), dim3(256), 0, stream,
                           (const float*)X_t, (const float*)sample_weight, labels, far_samples,
                           empty_clusters, (float*)per_sample_inertia, (float*)sums_t,
                           (float*)cluster_sizes, (const float*)sq_dist, n, d, k);
    else
        hipLaunchKernelGGL((relocate_kernel<double>), dim3(n_relocated), dim3(256), 0, stream,
                           (const double*)X_t, (const double*)sample_weight, labels, far_samples,
                           empty_clusters, (double*)per_sample_inertia, (double*)sums_t,
                           (double*)cluster_sizes, (const double*)sq_dist, n, d, k);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_relocate_empty_clusters(const void* X_t, const void* sample_weight,
                                    const uint32_t* labels, const int64_t* far_samples,
                                    const uint32_t* empty_clusters, int32_t n_relocated,
                                    void* per_sample_inertia, void* sums_t, void* cluster_sizes,
                                    int64_t n, int32_t d, int32_t k, int32_t dtype, void* stream) {
    return relocate(X_t, sample_weight, labels, far_samples, empty_clusters, n_relocated, per_sample_inertia, sums_t,
                    cluster_sizes, nullptr, n, d, k, dtype, stream);
}

int32_t kmx_relocate_empty_clusters_if(const void* X_t, const void* sample_weight, const uint32_t* labels,
                                       const int64_t* far_samples, const uint32_t* empty_clusters, int32_t n_relocated,
                                       const void* sq_dist, void* sums_t, void* cluster_sizes, int64_t n, int32_t d,
                                       int32_t k, int32_t dtype, void* stream) {
    KMX_REQUIRE_PTR(sq_dist);
    return relocate(X_t, sample_weight, labels, far_samples, empty_clusters, n_relocated, nullptr, sums_t, cluster_sizes,
                    sq_dist, n, d, k, dtype, stream);
}

}  // extern "C"
