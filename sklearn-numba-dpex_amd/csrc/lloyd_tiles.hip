// Labels of a Lloyd run from a half-precision copy of X that stays on the device for the run, for
// samples of more features than the fused steps keep on chip (fp32 and fp64).
//
// Once per run X is rounded to fp16 (scaled by a power of two) and laid out as the matrix
// instructions read it: tiles of 32 samples x 16 features, 1 KB each, lane (j, h) of a wave
// holding features 8 h .. 8 h + 7 of sample j.  An iteration then reads 2 bytes per value (a
// quarter of fp64) in whole kilobytes, converts nothing, and needs ONE v_mfma_f32_32x32x16_f16
// per 32 centroids x 32 samples x 16 features.
//
// The scores of the rounded data only screen the labels; a certificate says which of them are
// those of the exact data.  With x = x' + e_x and c = c' + e_c (primes: rounded) distances move by
// at most |e_x| + |e_c|, whatever the scores' size, so the nearest rounded centroid b is the
// nearest one if every other j has D'_j - D'_b > 2 eps, eps = |e_x| + max |e_c|.  |e_x| is not
// bounded but KNOWN, from the copy.  In scores s = <x', c'> - 0.5 |c'|^2 (D'^2 = |x'|^2 - 2 s), each
// with an error of at most delta from the fp32 accumulation, that is
//     s_b - s_j > 2 delta + 2 eps sqrt(|x'|^2 - 2 s_b + 2 delta) + 2 eps^2.
// (An error bound on the scores themselves would grow with |x| |c| instead of with the distance
// to the nearest centroid and certify far fewer samples.)  Samples without a certificate are
// listed together with the score below which no centroid can be theirs; a second kernel looks
// up the few centroids above it and takes their distances in fp64 from the exact rows.  A sample with
// more such centroids than that kernel holds goes through the tiled product of lloyd_gemm.hip.  If more than
// an eighth of the samples are listed, all samples do, and the run takes its labels from X again
// soon after (kmx_lloyd_run): the copy cannot tell such data apart, one feature being much wider than the
// others for instance.  1e6 x 100 with one feature 1e5 times wider, ten iterations, before this copy / with it
// alone / with the way back: fp32, 300 clusters 18.4 / 28.3 / 17.7 ms; fp64, 100 clusters 8.8 / 14.6 / 9.0.
//
// The labels that a run ends with are those that kmx_assign_labels gives for its centroids, which for
// fp32 inputs is the arg-max of fp32 scores: there the thresholds also leave room for the errors E of two
// such scores (MATCH in the code below; E = prod_rho (|x| C + C^2 / 2), C = max |c|).  A score gap of 2 E is
// a gap of 4 E between squared distances, and D_j^2 - D_b^2 >= (D'_j - eps)^2 - (D'_b + eps)^2 asks of the
// scores s a further 2 E (D'_b + 2 eps) / (D'_b + eps).  Candidates closer than that are decided by the
// scores themselves, from the instruction that the product uses, pair by pair on a diagonal.
//
// Measured, labels of one iteration: 1e6 x 256 fp32, 1 024 clusters 1.60 -> 0.54 ms (three fp16 products
// per pair and the listed samples in fp32 before), 1e6 x 100 fp64, 100 clusters 0.54 -> 0.10 ms (fp64 products
// before).  Bound by the matrix cores for many clusters (1.07e15 operations per second, where a large
// library product of this type reaches 1.25e15 on the same machine), by reading the copy for few (3.3 TB/s).
#include "lloyd_layout.h"

#include <type_traits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v8d __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int TILE_D_MAX = 256;      // samples' fragments live in registers: 16 steps of 16 features
constexpr int GRP = 8;               // accumulator registers per arg-max group
constexpr float ULP = 1.1920929e-7f; // 2^-23
constexpr float HALF_MIN = 6.1035156e-5f;  // 2^-14: smaller magnitudes are rounded to zero (no fp16 subnormals)

struct TileArea {
    int S;              // steps of 16 features
    int n_blocks;       // blocks of 32 centroids
    int64_t n_tiles;    // tiles of 32 samples (even)
    size_t off_xt, off_norm, off_err, off_ct, off_hneg, off_cmax, off_half, off_list, off_thr, off_rest, off_least, off_sums, sums_bytes, total;
};

inline TileArea tile_area(int64_t n, int d, int k, int words = 0) {  // (words of the kept sums, at the end)
    TileArea a;
    a.S = (d + 15) / 16;
    a.n_blocks = (k + 31) / 32;
    a.n_tiles = 2 * kmx_cdiv(n, 64);
    a.off_xt = kmx_align256(KMX_TH_WORDS * sizeof(unsigned int));
    a.off_norm = a.off_xt + (size_t)a.n_tiles * a.S * 1024;
    a.off_err = a.off_norm + kmx_align256((size_t)a.n_tiles * 32 * sizeof(float));
    a.off_ct = a.off_err + kmx_align256((size_t)a.n_tiles * 32 * sizeof(float));
    a.off_hneg = a.off_ct + (size_t)a.n_blocks * a.S * 1024;
    a.off_cmax = a.off_hneg + kmx_align256((size_t)a.n_blocks * 32 * sizeof(float));
    a.off_half = a.off_cmax + kmx_align256((size_t)a.n_blocks * sizeof(float2));
    a.off_list = a.off_half + kmx_align256((size_t)k * sizeof(double));
    a.off_thr = a.off_list + kmx_align256((size_t)n * sizeof(int));
    a.off_rest = a.off_thr + kmx_align256((size_t)n * sizeof(float));
    a.off_least = a.off_rest + kmx_align256((size_t)n * sizeof(int));
    a.off_sums = a.off_least + kmx_align256((size_t)(d + 1) * sizeof(unsigned int));
    a.sums_bytes = kmx_align256((size_t)(d + 1) * k * 8);
    a.total = a.off_sums + words * a.sums_bytes;
    return a;
}

__device__ __forceinline__ _Float16 to_half(float v) {
    return fabsf(v) < HALF_MIN ? (_Float16)0.0f : (_Float16)v;
}

// The scale: a power of two that brings the largest centroid coordinate into [2^10, 2^11), which
// leaves samples 32 times further out inside fp16 (beyond it they become infinite and get no
// certificate), but not the largest coordinate of 256 samples below 1: initial
// centroids far from all samples would round the samples away for the whole run, though the first
// relocation removes them (1e6 x 100 fp64, 100 clusters of which 3 start at 1e8: 27.5 -> 5.2 ms for
// ten iterations).  One workgroup.
// The exponent that brings m into [2^at, 2^(at + 1)), within what a float holds after scaling either
// way; none: lower than any.
constexpr int NO_EXPONENT = -1000;
__device__ __forceinline__ int scale_exponent(float m, int at) {
    if (!(m > 0.0f && m < kmx_inf<float>())) return NO_EXPONENT;
    const int e = at - ilogbf(m);
    return e > 100 ? 100 : e < -100 ? -100 : e;
}

// (`high`, `low`: the largest magnitudes a thread has seen of what goes to 2^10 and of what stays above 1)
__device__ __forceinline__ void tiles_write_scale(float high, float low, float (*m_s)[16], unsigned int* __restrict__ header) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        high = fmaxf(high, __shfl_xor(high, off, 64));
        low = fmaxf(low, __shfl_xor(low, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        m_s[0][threadIdx.x >> 6] = high;
        m_s[1][threadIdx.x >> 6] = low;
    }
    __syncthreads();
    if (threadIdx.x < KMX_TH_WORDS) header[threadIdx.x] = 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; ++i) {
            high = fmaxf(high, m_s[0][i]);
            low = fmaxf(low, m_s[1][i]);
        }
        const int eh = scale_exponent(high, 10), el = scale_exponent(low, 0), e = eh > el ? eh : el;
        header[KMX_TH_SCALE] = __float_as_uint(e == NO_EXPONENT ? 1.0f : ldexpf(1.0f, e));
    }
}

// largest magnitude in this thread's share of 256 samples: spread evenly over X, or STRETCHES: 64 in a row
// at four places (whole cache lines: 1e6 x 256, where a line per value takes 145 us, 10)
template <typename T, bool STRETCHES>
__device__ __forceinline__ float sampled_max(const T* __restrict__ X_t, int64_t n, int d) {
    const int t = threadIdx.x & 255;
    int64_t i = STRETCHES ? (int64_t)(t >> 6) * n / 4 + (t & 63) : (int64_t)t * n / 256;
    i = i < n ? i : n - 1;
    float m = 0.0f;
    for (int f0 = threadIdx.x >> 8; f0 < d; f0 += 4 * 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = fabsf((float)X_t[(size_t)(f0 + 4 * u < d ? f0 + 4 * u : f0) * n + i]);
#pragma unroll
        for (int u = 0; u < 16; ++u) m = fmaxf(m, v[u]);
    }
    return m;
}

template <typename T>
__global__ __launch_bounds__(1024) void tiles_scale_kernel(const T* __restrict__ centroids_t, const T* __restrict__ X_t,
                                                           unsigned int* __restrict__ header, unsigned int* __restrict__ least,
                                                           int items, int64_t n, int d) {
    __shared__ float m_s[2][16];
    float m = 0.0f;
    if ((int)threadIdx.x <= d) least[threadIdx.x] = 0u;  // (d <= 256; for the pass that follows)
    for (int i0 = threadIdx.x; i0 < items; i0 += 16 * 1024) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = i0 + u * 1024 < items ? fabsf((float)centroids_t[i0 + u * 1024]) : 0.0f;
#pragma unroll
        for (int u = 0; u < 16; ++u) m = fmaxf(m, v[u]);
    }
    tiles_write_scale(m, sampled_max<T, true>(X_t, n, d), m_s, header);
}

// The same where there are no centroids yet: from the samples alone.  One workgroup.
template <typename T>
__global__ __launch_bounds__(1024) void tiles_sample_scale_kernel(const T* __restrict__ X_t, unsigned int* __restrict__ header,
                                                                  int64_t n, int d) {
    __shared__ float m_s[2][16];
    tiles_write_scale(sampled_max<T, false>(X_t, n, d), 0.0f, m_s, header);
}

// The tiles, |x'|^2 and |e_x| per sample, the row-major copy of X and (absmax not null) the bits of
// max |x| per feature, the smallest |x| per feature and |w| (kmx_least_word) and whether all are finite, in one pass:
// 128 samples per workgroup and pass, 32 features at a time through LDS.  Bound by memory: (2 + 2 sizeof(T)) bytes
// per value.  A row's extremes meet over its lanes only where one of them exceeds what the workgroup has seen: of the few
// tiles that a workgroup takes about the first two.
template <typename T>
__global__ __launch_bounds__(256) void tiles_prepare_kernel(const T* __restrict__ X_t, T* __restrict__ X_rm,
                                                            const T* __restrict__ sample_weight, uint4* __restrict__ xt,
                                                            float* __restrict__ norm, float* __restrict__ err,
                                                            unsigned int* __restrict__ header,
                                                            unsigned int* __restrict__ absmax, unsigned int* __restrict__ least,
                                                            int64_t n, int d, int S, int64_t n_pad) {
    constexpr int NS = 128, NF = 32;
    constexpr int W = 16 / (int)sizeof(T);      // samples per 128-bit load
    constexpr int TPR = NS / W;                 // threads per row of 128 samples
    constexpr int RPP = 256 / TPR;              // rows per pass
    __shared__ T tile[NF][NS + 1];
    __shared__ float part[2][2][NS];
    __shared__ uint2 extremes[TILE_D_MAX];  // bits of the largest, flipped word of the smallest
    __shared__ unsigned int w_min;
    for (int f = threadIdx.x; f < TILE_D_MAX; f += 256) extremes[f] = make_uint2(0u, 0u);
    if (threadIdx.x == 0) w_min = 0u;
    const float xs = __uint_as_float(header[KMX_TH_SCALE]);
    const int s = threadIdx.x & (NS - 1), g2 = threadIdx.x >> 7;   // sample, pair of groups of 8 features
    float odd = 0.0f;  // (NaN once a value is NaN or infinite; the maxima leave NaN out)
    unsigned int w_least = ~0u;
    for (int64_t i0 = (int64_t)blockIdx.x * NS; i0 < n_pad; i0 += (int64_t)gridDim.x * NS) {
        float sq = 0.0f, e2 = 0.0f;
        if (absmax != nullptr && g2 == 0 && i0 + s < n) {
            const T w = sample_weight[i0 + s];
            w_least = min(w_least, kmx_least_word(w));
            odd = fmaf((float)w, 0.0f, odd);
        }
        for (int f0 = 0; f0 < 16 * S; f0 += NF) {
            {
                const int col = (threadIdx.x % TPR) * W, row0 = threadIdx.x / TPR;
                const int64_t i = i0 + col;
                T v[NF / RPP][W];
                // (the same for the whole workgroup: the loads of a stage that exists whole are straight-line code)
                const bool whole = f0 + NF <= d && i0 + NS <= n;
#pragma unroll
                for (int p = 0; p < NF / RPP; ++p) {
                    const int f = f0 + row0 + p * RPP;
                    const T* __restrict__ src = X_t + (size_t)f * n + i;
                    if (whole) {
                        const auto q = *reinterpret_cast<const typename KmxVec<T, W>::type*>(src);
#pragma unroll
                        for (int e = 0; e < W; ++e) v[p][e] = q[e];
                    } else {
#pragma unroll
                        for (int e = 0; e < W; ++e) v[p][e] = f < d && i + e < n ? src[e] : T(0);
                    }
                }
                __syncthreads();  // (the previous stage's reads are over)
                if (absmax != nullptr) {
#pragma unroll
                    for (int p = 0; p < NF / RPP; ++p) {
                        const int f = f0 + row0 + p * RPP;  // (below TILE_D_MAX)
                        float m = 0.0f;
                        unsigned int low = ~0u;
#pragma unroll
                        for (int e = 0; e < W; ++e) {
                            m = fmaxf(m, fabsf((float)v[p][e]));
                            low = min(low, kmx_least_word(v[p][e]));
                        }
                        const uint2 seen = extremes[f];
                        if (__any(__float_as_uint(m) > seen.x || ~low > seen.y)) {
#pragma unroll
                            for (int off = 1; off < TPR; off <<= 1) {
                                m = fmaxf(m, __shfl_xor(m, off, 64));
                                low = min(low, (unsigned int)__shfl_xor((int)low, off, 64));
                            }
                            if (col == 0) {
                                atomicMax(&extremes[f].x, __float_as_uint(m));
                                atomicMax(&extremes[f].y, ~low);
                            }
                        }
                    }
                }
#pragma unroll
                for (int p = 0; p < NF / RPP; ++p)
#pragma unroll
                    for (int e = 0; e < W; ++e) tile[row0 + p * RPP][col + e] = v[p][e];
            }
            __syncthreads();
            const int64_t i = i0 + s;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int g = 2 * g2 + q;
                if (f0 + 8 * g < 16 * S) {
                    v8h hv;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float v = (float)tile[8 * g + e][s] * xs;
                        const _Float16 hb = to_half(v);
                        const float hf = (float)hb;
                        hv[e] = hb;
                        sq = fmaf(hf, hf, sq);
                        const float r = v - hf;
                        e2 = fmaf(r, r, e2);
                        odd = fmaf(v, 0.0f, odd);
                    }
                    // step (f0 + 8 g) / 16, half h = g & 1
                    const int st = f0 / 16 + (g >> 1);
                    if (i < n_pad) xt[((size_t)(i >> 5) * S + st) * 64 + (g & 1) * 32 + (i & 31)] = __builtin_bit_cast(uint4, hv);
                }
            }
            if (X_rm != nullptr) {
                const int nf = d - f0 < NF ? d - f0 : NF;
                for (int e = threadIdx.x; e < NS * NF; e += 256) {
                    const int f = e % NF, ss = e / NF;
                    if (f < nf && i0 + ss < n) X_rm[(size_t)(i0 + ss) * d + f0 + f] = tile[f][ss];
                }
            }
        }
        part[0][g2][s] = sq;
        part[1][g2][s] = e2;
        __syncthreads();
        if (threadIdx.x < NS && i0 + s < n_pad) {
            const float tot = part[0][0][s] + part[0][1][s];
            norm[i0 + s] = tot;
            // (rounded up: the sum's own roundings, and for fp64 the rounding to fp32 before the split)
            const float lost = sqrtf(part[1][0][s] + part[1][1][s]) * 1.0001f;
            err[i0 + s] = sizeof(T) == 8 ? lost + 6.1e-8f * sqrtf(tot) * 1.001f : lost;
        }
    }
    if (absmax != nullptr) {
        __syncthreads();
        for (int f = threadIdx.x; f < d; f += 256) {
            atomicMax(absmax + f, extremes[f].x);
            atomicMax(least + f, extremes[f].y);
        }
        if (w_least != ~0u) atomicMax(&w_min, ~w_least);
        if (odd != 0.0f) header[KMX_TH_ODD] = 1u;  // (true for NaN)
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(least + d, w_min);
    }
}

// The centroids of a labelling: their tiles (32 centroids x 16 features, laid out like those of
// the samples), -0.5 |c'|^2 (-inf past the last one), and per block of 32 the maxima of 0.5 |c'|^2 and
// |e_c|.  A workgroup per block; its sixteen waves
// take a step each (four took four trips to memory: 11 us, now 6).  The first one clears the counts.
constexpr int CENT_WAVES = 16;
template <typename T>
__global__ __launch_bounds__(64 * CENT_WAVES) void tiles_centroids_kernel(const T* __restrict__ centroids_t, uint4* __restrict__ ct,
                                                              float* __restrict__ hneg, float2* __restrict__ cmax,
                                                              unsigned int* __restrict__ header,
                                                              const kmx_lloyd_status* __restrict__ status,
                                                              const unsigned int* __restrict__ absmax,
                                                              const unsigned int* __restrict__ least, int d, int k, int S, int span) {
    if (status != nullptr && status->state != KMX_RUNNING) return;
    __shared__ double part[2][CENT_WAVES][64];
    const float xs = __uint_as_float(header[KMX_TH_SCALE]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 32 + (lane & 31), h = lane >> 5;
    double sq = 0.0, e2 = 0.0;
    for (int st = wave; st < S; st += CENT_WAVES) {
        v8h hv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int f = 16 * st + 8 * h + e;
            const double v = (c < k && f < d) ? (double)centroids_t[(size_t)f * k + c] * (double)xs : 0.0;
            const _Float16 hb = to_half((float)v);
            hv[e] = hb;
            const double hf = (double)(float)hb;
            sq += hf * hf;
            e2 += (v - hf) * (v - hf);
        }
        ct[((size_t)blockIdx.x * S + st) * 64 + lane] = __builtin_bit_cast(uint4, hv);
    }
    part[0][wave][lane] = sq;
    part[1][wave][lane] = e2;
    __syncthreads();
    if (threadIdx.x < 64) {
        float hm = 0.0f, em = 0.0f;
        if (threadIdx.x < 32) {
            double s = 0.0, q = 0.0;
            for (int w = 0; w < (S < CENT_WAVES ? S : CENT_WAVES); ++w) {
                s += part[0][w][lane] + part[0][w][lane + 32];
                q += part[1][w][lane] + part[1][w][lane + 32];
            }
            const float hv = (float)(0.5 * s);
            hneg[c] = c < k ? -hv : -kmx_inf<float>();
            if (c < k) {
                // (NaN or infinite centroids: an infinite bound, no certificates)
                hm = hv < kmx_inf<float>() ? hv : kmx_inf<float>();
                em = (float)(sqrt(q) * 1.00001);
                em = em < kmx_inf<float>() ? em : kmx_inf<float>();
            }
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
            hm = fmaxf(hm, __shfl_xor(hm, off, 64));
            em = fmaxf(em, __shfl_xor(em, off, 64));
        }
        if (threadIdx.x == 0) {
            cmax[blockIdx.x] = make_float2(hm, em);
            if (blockIdx.x == 0) {
                header[KMX_TH_LISTED] = 0u;
                header[KMX_TH_REST] = 0u;
                header[KMX_TH_MOVED] = 0u;
                header[KMX_TH_ENTRIES] = 0u;
            }
        }
    }
    // (an iteration: whether the sums have fixed point, and whether those kept from the one before can be corrected)
    if (blockIdx.x == 0 && absmax != nullptr) {
        bool fixed = header[KMX_TH_ODD] == 0u;
        for (int f = threadIdx.x; f <= d; f += 64 * CENT_WAVES) fixed &= kmx_kept_fixed<T>(absmax, least, d, f, span);
        const bool all = __syncthreads_and(fixed ? 1 : 0) != 0;
        if (threadIdx.x == 0) {
            header[KMX_TH_FIXED] = all ? 1u : 0u;
            header[KMX_TH_KEEP] = all && status->n_iter > 0 && header[KMX_TH_SUMS] == (unsigned int)status->n_iter ? 1u : 0u;
        }
    }
}

// LDS reads the compiler does not count: it would wait for every direct-to-LDS copy in flight
// before each of them.  The values are valid after lds_wait<N> (N later reads still in flight), which
// takes them as operands.
template <int OFFSET>
__device__ __forceinline__ v4f lds_read16(unsigned int addr) {
    v4f v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFFSET));
    return v;
}
template <int N>
__device__ __forceinline__ void lds_wait(v4f& a, v4f& b, v4f& c, v4f& d) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : "n"(N));
}

// Blocks of centroid tiles in each of the three LDS buffers of STREAM mode (S kilobytes a block)
constexpr int stream_blocks(int S) { return S >= 8 ? 2 : S >= 4 ? 4 : 8; }

// over all blocks of centroids: max 0.5 |c'|^2 and max |e_c| (uniform)
__device__ __forceinline__ float2 reduce_block_max(const float2* __restrict__ block_max, int n_blocks) {
    float2 v = make_float2(0.0f, 0.0f);
    for (int b = threadIdx.x & 63; b < n_blocks; b += 64) {
        const float2 m = block_max[b];
        v.x = fmaxf(v.x, m.x);
        v.y = fmaxf(v.y, m.y);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v.x = fmaxf(v.x, __shfl_xor(v.x, off, 64));
        v.y = fmaxf(v.y, __shfl_xor(v.y, off, 64));
    }
    v.x = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v.x)));
    v.y = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v.y)));
    return v;
}

constexpr int PEND = 128;  // entries a wave gathers before it adds them to the list

// NCOL: tiles of 32 samples per wave.  STREAM: the centroid tiles do not fit the LDS and travel
// through three buffers of stream_blocks(S) blocks, shared by the eight waves; otherwise they are
// copied once and the waves go their own ways.
template <int S, int NCOL, bool STREAM>
__global__ __launch_bounds__(512, 2) void tiles_label_kernel(
    const uint4* __restrict__ xt, const float* __restrict__ norm, const float* __restrict__ err,
    const uint4* __restrict__ ct, const float* __restrict__ hneg, const float2* __restrict__ block_max,
    unsigned int* __restrict__ header, const kmx_lloyd_status* __restrict__ status, uint32_t* __restrict__ labels,
    const uint32_t* __restrict__ labels_prev, int* __restrict__ list, float* __restrict__ list_thr, int64_t n, int n_blocks,
    float prod_rho) {
    if (status != nullptr && status->state != KMX_RUNNING) return;
    extern __shared__ __align__(16) unsigned char tiles_lds[];
    constexpr int CB = STREAM ? stream_blocks(S) : 1;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, j = lane & 31;
    // -0.5 |c'|^2 of every centroid first, then the centroid tiles
    float* hneg_s = reinterpret_cast<float*>(tiles_lds);
    const int hneg_bytes = (n_blocks * 32 * 4 + 1023) & ~1023;
    uint4* ct_s = reinterpret_cast<uint4*>(tiles_lds + hneg_bytes);
    // Samples without a certificate, gathered by every wave until there are enough for one addition to
    // the counter of the list: with one per group of samples that has any, the additions to that
    // one word were the kernel (138 us instead of 60 at 1e6 x 100).
    __shared__ int pend_i[8][PEND];
    __shared__ float pend_thr[8][PEND];
    int pending = 0;  // (the same in all lanes)
    __shared__ unsigned int moved_block;
    if (threadIdx.x == 0) moved_block = 0u;
    unsigned int moved = 0u;
    auto flush = [&]() __attribute__((always_inline)) {
        unsigned int base = 0;
        if (lane == 0) base = atomicAdd(header + KMX_TH_LISTED, (unsigned int)pending);
        base = (unsigned int)__builtin_amdgcn_readfirstlane((int)base);
        for (int e = lane; e < pending; e += 64) {
            list[base + e] = pend_i[wave][e];
            list_thr[base + e] = pend_thr[wave][e];
        }
        pending = 0;
    };
    for (int c = threadIdx.x; c < n_blocks * 32; c += 512) hneg_s[c] = hneg[c];
    const unsigned int hneg_addr = (unsigned int)(uintptr_t)hneg_s + (unsigned int)(16 * h);
    const unsigned int ct_addr = (unsigned int)(uintptr_t)ct_s + (unsigned int)lane * 16u;
    // one kilobyte per wave and instruction, straight into LDS
    auto copy_tiles = [&](const uint4* src, int first_kb, int n_kb) {
        for (int q = wave; q < n_kb; q += 8)
            __builtin_amdgcn_global_load_lds(src + (size_t)q * 64 + lane,
                                             (__attribute__((address_space(3))) void*)(ct_s + (size_t)(first_kb + q) * 64), 16, 0, 0);
    };
    if constexpr (!STREAM) copy_tiles(ct, 0, n_blocks * S);

    const float2 most = reduce_block_max(block_max, n_blocks);
    const float hmax = most.x, emax = most.y;
    const float cmax = sqrtf(2.0f * hmax) * 1.0001f;
    const float rho = ULP * (17.0f * (float)S + 4.0f);
    float pos_inf = kmx_inf<float>();
    asm volatile("" : "+s"(pos_inf));  // (keeps the first maximum of a group an instruction the compiler sees as such)
    const float neg_inf = -kmx_inf<float>();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    const int64_t n_groups = (n + 32 * NCOL - 1) / (32 * NCOL);  // columns of samples of a wave
    const int n_chunks = STREAM ? (n_blocks + CB - 1) / CB : 1;
    // STREAM: the waves of a workgroup stay together (idle ones past the end take part in the barriers)
    const int64_t rounds_end = STREAM ? (n_groups + 7) / 8 * 8 : n_groups;
    for (int64_t grp = (int64_t)blockIdx.x * 8 + wave; grp < rounds_end; grp += (int64_t)gridDim.x * 8) {
        const bool live_group = grp < n_groups;
        const int64_t grp_r = live_group ? grp : n_groups - 1;
        v8h x[NCOL][S];
#pragma unroll
        for (int cl = 0; cl < NCOL; ++cl) {
            const uint4* __restrict__ src = xt + (size_t)(grp_r * NCOL + cl) * S * 64 + lane;
#pragma unroll
            for (int s = 0; s < S; ++s) x[cl][s] = __builtin_bit_cast(v8h, src[s * 64]);
        }
        // Running arg-max of each column of samples: best score, second best group, and the eight
        // registers of the winning group (kept as they are; the position inside is looked up once
        // per tile).  Plain variables: a struct or an array of them ends up in memory.
        float best0 = neg_inf, best1 = neg_inf, second0 = neg_inf, second1 = neg_inf;
        unsigned int code0 = 0, code1 = 0;
        double w00, w01, w02, w03, w10, w11, w12, w13;
        asm volatile("" : "=v"(w00), "=v"(w01), "=v"(w02), "=v"(w03));
        asm volatile("" : "=v"(w10), "=v"(w11), "=v"(w12), "=v"(w13));

        // arg-max by groups of eight registers, with the second largest of the group maxima
        auto argmax = [&](const v16f& sc, float& best, float& second, unsigned int& code, double& w0, double& w1, double& w2,
                          double& w3, const int b) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const unsigned int cd = (unsigned int)(2 * b + g);  // wave-uniform
                float m = __builtin_amdgcn_fmed3f(sc[g * GRP], sc[g * GRP + 1], pos_inf);
#pragma unroll
                for (int r = 2; r + 1 < GRP; r += 2)
                    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(m), "v"(sc[g * GRP + r]), "v"(sc[g * GRP + r + 1]));
                asm("v_med3_f32 %0, %1, %2, %3" : "=v"(second) : "v"(best), "v"(second), "v"(m));
                if (m > best) {  // strict: the earlier group keeps a tie
                    best = m;
                    code = cd;
                    const v8d ad = __builtin_bit_cast(v8d, sc);
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w0) : "v"(ad[g * 4]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w1) : "v"(ad[g * 4 + 1]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w2) : "v"(ad[g * 4 + 2]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w3) : "v"(ad[g * 4 + 3]));
                }
            }
        };

        // one block of 32 centroids: accumulator register r of half h is centroid 8 (r / 4) + 4 h + r % 4
        auto block = [&](const int b, const unsigned int a_addr) __attribute__((always_inline)) {
            const unsigned int hb = hneg_addr + (unsigned int)b * 128u;
            v4f hq[4] = {lds_read16<0>(hb), lds_read16<32>(hb), lds_read16<64>(hb), lds_read16<96>(hb)};
            constexpr int G = (S + 3) / 4;
            v4f a[2][4];
            auto issue = [&](auto g_tag) __attribute__((always_inline)) {
                constexpr int g = decltype(g_tag)::value;
                a[g & 1][0] = lds_read16<(4 * g + 0) * 1024>(a_addr);
                if constexpr (4 * g + 1 < S) a[g & 1][1] = lds_read16<(4 * g + 1) * 1024>(a_addr);
                if constexpr (4 * g + 2 < S) a[g & 1][2] = lds_read16<(4 * g + 2) * 1024>(a_addr);
                if constexpr (4 * g + 3 < S) a[g & 1][3] = lds_read16<(4 * g + 3) * 1024>(a_addr);
            };
            v16f acc[NCOL];
            issue(std::integral_constant<int, 0>{});
            auto step = [&](auto g_tag) __attribute__((always_inline)) {
                constexpr int g = decltype(g_tag)::value;
                constexpr int N_NEXT = g + 1 < G ? (S - 4 * (g + 1) < 4 ? S - 4 * (g + 1) : 4) : 0;
                if constexpr (g + 1 < G) issue(std::integral_constant<int, g + 1>{});
                if constexpr (g == 0) {
                    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(hq[0]), "+v"(hq[1]), "+v"(hq[2]), "+v"(hq[3]) : "n"(N_NEXT));
                }
                lds_wait<N_NEXT>(a[g & 1][0], a[g & 1][1], a[g & 1][2], a[g & 1][3]);
                if constexpr (g == 0) {
#pragma unroll
                    for (int cl = 0; cl < NCOL; ++cl)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            acc[cl][e] = hq[0][e];
                            acc[cl][4 + e] = hq[1][e];
                            acc[cl][8 + e] = hq[2][e];
                            acc[cl][12 + e] = hq[3][e];
                        }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (4 * g + u < S) {
                        const v8h av = __builtin_bit_cast(v8h, a[g & 1][u]);
#pragma unroll
                        for (int cl = 0; cl < NCOL; ++cl)
                            acc[cl] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, x[cl][4 * g + u], acc[cl], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);
            };
            step(std::integral_constant<int, 0>{});
            if constexpr (G > 1) step(std::integral_constant<int, 1>{});
            if constexpr (G > 2) step(std::integral_constant<int, 2>{});
            if constexpr (G > 3) step(std::integral_constant<int, 3>{});
            argmax(acc[0], best0, second0, code0, w00, w01, w02, w03, b);
            if constexpr (NCOL > 1) argmax(acc[1], best1, second1, code1, w10, w11, w12, w13, b);
        };

        if constexpr (STREAM) {
            auto issue_chunk = [&](int ch) {
                const int left = n_blocks - ch * CB;
                copy_tiles(ct + (size_t)ch * CB * S * 64, (ch % 3) * CB * S, (left < CB ? left : CB) * S);
            };
            // every wave is done with the buffers of the previous round
            __syncthreads();
            issue_chunk(0);
            if (n_chunks > 1) issue_chunk(1);
            for (int ch = 0; ch < n_chunks; ++ch) {
                // A wave's copies of chunk ch are complete when at most those of chunk ch + 1 are in
                // flight (at most CB * S / 8 of them per wave: all full chunks but the last)
                if (ch + 2 < n_chunks)
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CB * S / 8) : "memory");
                else
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                asm volatile("s_barrier" ::: "memory");
                if (ch + 2 < n_chunks) issue_chunk(ch + 2);
                const int left = n_blocks - ch * CB;
                const int nb = left < CB ? left : CB;
                unsigned int addr = ct_addr + (unsigned int)((ch % 3) * CB * S) * 1024u;
                for (int b = 0; b < nb; ++b, addr += S * 1024u) block(ch * CB + b, addr);
            }
        } else {
            unsigned int addr = ct_addr;
            for (int b = 0; b < n_blocks; ++b, addr += S * 1024u) block(b, addr);
        }

        auto finish = [&](const float best, const float second, const unsigned int code, const double w0, const double w1,
                          const double w2, const double w3, const int cl) __attribute__((always_inline)) {
            float sv[GRP];
            {
                const float2 p0 = __builtin_bit_cast(float2, w0), p1 = __builtin_bit_cast(float2, w1);
                const float2 p2 = __builtin_bit_cast(float2, w2), p3 = __builtin_bit_cast(float2, w3);
                sv[0] = p0.x; sv[1] = p0.y; sv[2] = p1.x; sv[3] = p1.y;
                sv[4] = p2.x; sv[5] = p2.y; sv[6] = p3.x; sv[7] = p3.y;
            }
            unsigned int pos = GRP - 1, n_eq = 0;
            float sec = second;
#pragma unroll
            for (int r = GRP - 1; r >= 0; --r) {
                const bool eq = sv[r] == best;
                pos = eq ? (unsigned int)r : pos;
                n_eq += eq ? 1u : 0u;
                const float rest = eq ? neg_inf : sv[r];
                sec = rest > sec ? rest : sec;
            }
            sec = n_eq > 1u ? best : sec;
            const unsigned int reg = (code & 1u) * GRP + pos;
            int c = (int)(32 * (code >> 1) + 8 * (reg >> 2) + 4 * h + (reg & 3u));
            float bb = best;
            {
                const float ov = __shfl_xor(best, 32, 64);
                const float o2 = __shfl_xor(sec, 32, 64);
                const int oc = __shfl_xor(c, 32, 64);
                const float t2 = sec > o2 ? sec : o2;
                const float lower = ov < best ? ov : best;
                sec = lower > t2 ? lower : t2;
                if (ov > bb || (ov == bb && oc < c)) {
                    c = oc;
                    bb = ov;
                }
            }
            const int64_t i = (grp_r * NCOL + cl) * 32 + j;
            const bool mine = live_group && h == 0 && i < n;
            const float nx2 = mine ? norm[i] : 0.0f, ex = mine ? err[i] : 0.0f;
            const uint32_t was = mine && labels_prev != nullptr ? labels_prev[i] : 0u;
            const float delta = rho * fmaf(sqrtf(nx2) * 1.0001f, cmax, hmax);
            const float eps = (ex + emax) * 1.0001f;
            const float d2 = fmaxf(nx2 * 1.00005f - 2.0f * bb + 2.0f * delta, 0.0f);
            float thr = (2.0f * delta + 2.0f * eps * (sqrtf(d2) + eps)) * 1.0001f;
            if (prod_rho > 0.0f) {  // MATCH
                const float cfull = cmax + emax;
                const float e_prod = prod_rho * fmaf(sqrtf(nx2) * 1.0001f + ex, cfull, 0.5f * cfull * cfull);
                const float near = sqrtf(fmaxf(nx2 * 0.99995f - 2.0f * bb - 2.0f * delta, 0.0f));
                const float ratio = near + eps > 0.0f ? (near + 2.0f * eps) / (near + eps) : 2.0f;
                thr += 2.0f * e_prod * ratio * 1.0001f;
            }
            // (a NaN anywhere makes the sample uncertain)
            const bool unsure = mine && !(bb - sec > thr);
            const unsigned long long um = __ballot(unsure);
            if (um) {
                if (unsure) {
                    const int at = pending + __popcll(um & ((1ull << lane) - 1ull));
                    pend_i[wave][at] = (int)i;
                    pend_thr[wave][at] = bb - thr - ULP * fabsf(bb);  // (rounded down)
                }
                pending += __popcll(um);
                if (pending > PEND - 32) flush();
            }
            if (mine && !unsure) {
                labels[i] = (uint32_t)c;
                moved += was != (uint32_t)c ? 1u : 0u;
            }
        };
        finish(best0, second0, code0, w00, w01, w02, w03, 0);
        if constexpr (NCOL > 1) finish(best1, second1, code1, w10, w11, w12, w13, 1);
    }
    if (pending > 0) flush();
    if (labels_prev != nullptr) {
        if (moved != 0u) atomicAdd(&moved_block, moved);
        __syncthreads();
        if (threadIdx.x == 0 && moved_block != 0u) atomicAdd(header + KMX_TH_MOVED, moved_block);
    }
}

// The listed samples: the centroids whose score reaches the sample's threshold are looked up again
// on the matrix cores (32 samples per workgroup, the tiles gathered by sample, the blocks of
// centroids dealt out to the four waves, the next block's tiles in flight), then their squared distances
// are taken in fp64 from the exact rows, eight lanes per sample; the lowest index wins a tie.  Bound
// by trips to memory: a few percent of the samples are listed in the usual run.
// MATCH (fp32 inputs): candidates whose squared distances are not 4 E apart are decided by the scores of
// the product: pair p of a sample and a candidate is row and column p of 32 x 32 blocks of
// v_mfma_f32_32x32x2_f32, features in order from -0.5 |c|^2 (`half_norms`), of which the diagonal counts.
constexpr int CAND = 8;
template <typename T, int S, bool MATCH>
__global__ __launch_bounds__(256) void tiles_resolve_kernel(
    const T* __restrict__ X_rm, const T* __restrict__ cpack, const uint4* __restrict__ xt, const uint4* __restrict__ ct,
    const float* __restrict__ hneg, unsigned int* __restrict__ header, kmx_lloyd_status* __restrict__ status,
    uint32_t* __restrict__ labels, const int* __restrict__ list, const float* __restrict__ list_thr, int* __restrict__ rest,
    int64_t n, int d, int dpad, int k, int n_blocks, const float2* __restrict__ block_max,
    const float* __restrict__ half_norms, float prod_rho, unsigned int* __restrict__ listed_out) {
    static_assert(!MATCH || sizeof(T) == 4, "fp64 inputs: labels by fp64 distances");
    if (status != nullptr && status->state != KMX_RUNNING) return;
    __shared__ int cand_n[32];
    __shared__ int cand[32][CAND];
    __shared__ int n_pairs;                                     // MATCH: pairs to be decided by scores
    __shared__ uint16_t pair_s[MATCH ? 32 * CAND : 1];          // sample * CAND + candidate
    __shared__ float score_s[MATCH ? 32 : 1][CAND];
    __shared__ bool close_s[32];
    double c_most = 0.0;  // max |c|, unscaled
    if constexpr (MATCH) {
        const float2 most = reduce_block_max(block_max, n_blocks);
        c_most = (sqrt(2.0 * (double)most.x) * 1.0001 + (double)most.y) / (double)__uint_as_float(header[KMX_TH_SCALE]);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, j = lane & 31;
    const int64_t n_listed = (int64_t)header[KMX_TH_LISTED];
    if (listed_out != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *listed_out = (unsigned int)n_listed;
    if (n_listed > (n >> 3)) {  // the tiled product takes all samples
        if (status != nullptr && blockIdx.x == 0 && threadIdx.x == 0 && status->uncertified_iter == 0)
            status->uncertified_iter = status->n_iter + 1;
        return;
    }
    for (int64_t t0 = (int64_t)blockIdx.x * 32; t0 < n_listed; t0 += (int64_t)gridDim.x * 32) {
        const int64_t slot = t0 + j;
        const bool live = slot < n_listed;
        const int i = list[live ? slot : t0];
        const float thr = live ? list_thr[slot] : kmx_inf<float>();
        if (threadIdx.x < 32) {
            cand_n[j] = live ? 0 : CAND + 1;
            close_s[j] = false;
        }
        if (MATCH && threadIdx.x == 0) n_pairs = 0;
        __syncthreads();
        if (wave < n_blocks) {
            const uint4* __restrict__ xs = xt + (size_t)(i >> 5) * S * 64 + h * 32 + (i & 31);
            v8h x[S];
#pragma unroll
            for (int s = 0; s < S; ++s) x[s] = __builtin_bit_cast(v8h, xs[s * 64]);
            uint4 a[S];
            v16f start;
            auto fetch = [&](const int b) __attribute__((always_inline)) {
                const uint4* __restrict__ as = ct + (size_t)b * S * 64 + lane;
#pragma unroll
                for (int s = 0; s < S; ++s) a[s] = as[s * 64];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(hneg + 32 * b + 8 * q + 4 * h);
                    start[4 * q] = v.x;
                    start[4 * q + 1] = v.y;
                    start[4 * q + 2] = v.z;
                    start[4 * q + 3] = v.w;
                }
            };
            fetch(wave);
            for (int b = wave; b < n_blocks; b += 4) {
                v16f acc = start;
#pragma unroll
                for (int s = 0; s < S; ++s)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[s]), x[s], acc, 0, 0, 0);
                if (b + 4 < n_blocks) fetch(b + 4);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int c = 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (live && c < k && !(acc[r] < thr)) {
                        const int at = atomicAdd(&cand_n[j], 1);
                        if (at < CAND) cand[j][at] = c;
                    }
                }
            }
        }
        __syncthreads();
        const int e = lane & 7, js = 8 * wave + (lane >> 3);  // eight lanes per sample
        const int nc = cand_n[js];
        const int64_t sl = t0 + js;
        const bool here = sl < n_listed;
        const int is = list[here ? sl : t0];
        const bool fine = here && nc >= 1 && nc <= CAND;
        double best = __builtin_huge_val(), next = __builtin_huge_val(), x_sq = 0.0;
        int arg = 0x7fffffff;
        const T* __restrict__ row = X_rm + (size_t)is * d;
        int most = fine ? nc : 0;
#pragma unroll
        for (int off = 8; off < 64; off <<= 1) {
            const int o = __shfl_xor(most, off, 64);
            most = o > most ? o : most;
        }
        for (int m = 0; m < most; m += 2) {
            const int ca = cand[js][fine && m < nc ? m : 0], cb = cand[js][fine && m + 1 < nc ? m + 1 : 0];
            const T* __restrict__ ra = cpack + (size_t)(fine ? ca : 0) * dpad;
            const T* __restrict__ rb = cpack + (size_t)(fine ? cb : 0) * dpad;
            double sa = 0.0, sb = 0.0;
#pragma unroll 8
            for (int f = e; f < d; f += 8) {
                const double xv = (double)row[f];
                if (MATCH && m == 0) x_sq = fma(xv, xv, x_sq);
                const double da = xv - (double)ra[f], db = xv - (double)rb[f];
                sa = fma(da, da, sa);
                sb = fma(db, db, sb);
            }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) {
                sa += __shfl_xor(sa, off, 64);
                sb += __shfl_xor(sb, off, 64);
            }
            if (fine && m < nc) {
                next = fmin(next, fmax(sa, best));
                if (sa < best || (sa == best && ca < arg)) {
                    best = sa;
                    arg = ca;
                }
            }
            if (fine && m + 1 < nc) {
                next = fmin(next, fmax(sb, best));
                if (sb < best || (sb == best && cb < arg)) {
                    best = sb;
                    arg = cb;
                }
            }
        }
        bool close = false;
        if constexpr (MATCH) {
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) x_sq += __shfl_xor(x_sq, off, 64);
            const double e_prod = (double)prod_rho * (sqrt(x_sq) + 0.5 * c_most) * c_most;
            close = fine && nc > 1 && !(next - best > 4.001 * e_prod + (d + 8) * 2.3e-16 * (next + best));
            if (close && e == 0) {
                const int at = atomicAdd(&n_pairs, nc);
                for (int m = 0; m < nc; ++m) pair_s[at + m] = (uint16_t)(js * CAND + m);
                close_s[js] = true;
            }
        }
        if (e == 0 && here && !close) {
            // (no candidate at all, or a distance that is not a number: left to the tiled product too)
            if (fine && arg < k)
                labels[is] = (uint32_t)arg;
            else
                rest[atomicAdd(header + KMX_TH_REST, 1u)] = is;
        }
        __syncthreads();
        if constexpr (MATCH) {
            for (int b = wave; 32 * b < n_pairs; b += 4) {
                const int p = 32 * b + j;
                const int pair = pair_s[p < n_pairs ? p : 0], c = cand[pair / CAND][pair % CAND];
                const float* __restrict__ xr = X_rm + (size_t)list[t0 + pair / CAND] * d;
                const float* __restrict__ cr = cpack + (size_t)c * dpad;
                const float start = -half_norms[c];
                v16f acc;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] = start;
                for (int f0 = 0; f0 < d; f0 += 16) {
                    float xv[8], cv[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int f = f0 + 2 * u + h;
                        xv[u] = f < d ? xr[f] : 0.0f;
                        cv[u] = f < d ? cr[f] : 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(cv[u], xv[u], acc, 0, 0, 0);
                }
                // the diagonal: row j is register 4 (j / 8) + j % 4 of half (j / 4) % 2
                float v = acc[0];
#pragma unroll
                for (int r = 1; r < 16; ++r) v = r == 4 * (j >> 3) + (j & 3) ? acc[r] : v;
                if (p < n_pairs && h == ((j >> 2) & 1)) score_s[pair / CAND][pair % CAND] = v;
            }
            __syncthreads();
            if (threadIdx.x < 32 && close_s[j]) {
                float top = -kmx_inf<float>();
                int lab = 0x7fffffff;
                bool finite = true;
                for (int m = 0; m < cand_n[j]; ++m) {
                    const float v = score_s[j][m];
                    finite &= fabsf(v) < kmx_inf<float>();
                    if (v > top || (v == top && cand[j][m] < lab)) {
                        top = v;
                        lab = cand[j][m];
                    }
                }
                const int ic = list[t0 + j];
                if (finite) labels[ic] = (uint32_t)lab;
                else rest[atomicAdd(header + KMX_TH_REST, 1u)] = ic;
            }
            __syncthreads();
        }
    }
}

template <int S, int NCOL, bool STREAM>
int32_t launch_labels(const TileArea& a, char* area, const kmx_lloyd_status* status, uint32_t* labels,
                      const uint32_t* labels_prev, int64_t n, float prod_rho, hipStream_t stream) {
    const size_t hneg_bytes = ((size_t)a.n_blocks * 128 + 1023) & ~(size_t)1023;
    const size_t lds = hneg_bytes + (STREAM ? (size_t)3 * stream_blocks(S) * S * 1024 : (size_t)a.n_blocks * S * 1024);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&tiles_label_kernel<S, NCOL, STREAM>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int32_t)e;
    }
    int64_t grid = kmx_cdiv(n, 8 * 32 * NCOL);
    if (grid > kmx_num_cus()) grid = kmx_num_cus();
    hipLaunchKernelGGL((tiles_label_kernel<S, NCOL, STREAM>), dim3((unsigned)grid), dim3(512), lds, stream,
                       (const uint4*)(area + a.off_xt), (const float*)(area + a.off_norm), (const float*)(area + a.off_err),
                       (const uint4*)(area + a.off_ct), (const float*)(area + a.off_hneg),
                       (const float2*)(area + a.off_cmax), (unsigned int*)area, status, labels, labels_prev,
                       (int*)(area + a.off_list), (float*)(area + a.off_thr), n, a.n_blocks, prod_rho);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

constexpr size_t TILES_LDS_MAX = 148 * 1024;  // (beside the 8 KB of the waves' list entries)

template <int S>
int32_t launch_labels_s(const TileArea& a, char* area, const kmx_lloyd_status* status, uint32_t* labels,
                        const uint32_t* labels_prev, int64_t n, float prod_rho, hipStream_t stream) {
    const size_t resident = (((size_t)a.n_blocks * 128 + 1023) & ~(size_t)1023) + (size_t)a.n_blocks * S * 1024;
    const bool in_lds = resident <= TILES_LDS_MAX;
    // two columns per wave (a centroid fragment read from LDS serves two products) unless that leaves
    // compute units without a wave
    const bool two = n >= (int64_t)64 * 8 * kmx_num_cus() / 2;
    if (in_lds)
        return two ? launch_labels<S, 2, false>(a, area, status, labels, labels_prev, n, prod_rho, stream)
                   : launch_labels<S, 1, false>(a, area, status, labels, labels_prev, n, prod_rho, stream);
    return two ? launch_labels<S, 2, true>(a, area, status, labels, labels_prev, n, prod_rho, stream)
               : launch_labels<S, 1, true>(a, area, status, labels, labels_prev, n, prod_rho, stream);
}

}  // namespace

bool kmx_tiles_fit(int64_t n, int d, int k) {
    // (the half norms of all centroids stay in LDS beside the buffers of the centroid tiles)
    return d <= TILE_D_MAX && n <= INT32_MAX - 64 && k <= 8192;
}

size_t kmx_tiles_bytes(int64_t n, int d, int k, int words) { return tile_area(n, d, k, words).total; }

static void tiles_copy(const void* X_t, void* X_rowmajor, const void* w, char* area, unsigned int* absmax, unsigned int* least,
                       int64_t n, int d, int dtype, hipStream_t stream) {
    const TileArea a = tile_area(n, d, 0);  // (the samples' part depends on n and d alone)
    unsigned int* header = (unsigned int*)area;
    const int64_t n_pad = a.n_tiles * 32;
    int64_t grid = kmx_cdiv(n_pad, 128);
    const int64_t cap = (int64_t)(dtype == KMX_F32 ? 8 : 4) * kmx_num_cus();
    if (grid > cap) grid = cap;
#define KMX_TILES_COPY(T)                                                                                                 \
    do {                                                                                                                  \
        hipLaunchKernelGGL((tiles_prepare_kernel<T>), dim3((unsigned)grid), dim3(256), 0, stream, (const T*)X_t,          \
                           (T*)X_rowmajor, (const T*)w, (uint4*)(area + a.off_xt), (float*)(area + a.off_norm),           \
                           (float*)(area + a.off_err), header, absmax, least, n, d, a.S, n_pad);                          \
    } while (0)
    if (dtype == KMX_F32) KMX_TILES_COPY(float); else KMX_TILES_COPY(double);
#undef KMX_TILES_COPY
}

// Scale, tiles and norms of X, and its row-major copy; `centroids_t`: the initial centroids.
int32_t kmx_tiles_prepare(const void* X_t, void* X_rowmajor, const void* w, const void* centroids_t, char* area,
                          unsigned int* absmax, int64_t n, int d, int k, int dtype, hipStream_t stream) {
    unsigned int* header = (unsigned int*)area;
    unsigned int* least = (unsigned int*)(area + tile_area(n, d, k).off_least);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((tiles_scale_kernel<float>), dim3(1), dim3(1024), 0, stream, (const float*)centroids_t,
                           (const float*)X_t, header, least, d * k, n, d);
    else
        hipLaunchKernelGGL((tiles_scale_kernel<double>), dim3(1), dim3(1024), 0, stream, (const double*)centroids_t,
                           (const double*)X_t, header, least, d * k, n, d);
    tiles_copy(X_t, X_rowmajor, w, area, absmax, least, n, d, dtype, stream);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

// The same without centroids (kmeans++, kmeanspp.hip): the area ends where the centroid tiles would begin.
size_t kmx_tiles_samples_bytes(int64_t n, int d) { return tile_area(n, d, 0).off_ct; }

int32_t kmx_tiles_prepare_samples(const void* X_t, void* X_rowmajor, char* area, int64_t n, int d, int dtype,
                                  hipStream_t stream) {
    unsigned int* header = (unsigned int*)area;
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((tiles_sample_scale_kernel<float>), dim3(1), dim3(1024), 0, stream, (const float*)X_t, header, n, d);
    else
        hipLaunchKernelGGL((tiles_sample_scale_kernel<double>), dim3(1), dim3(1024), 0, stream, (const double*)X_t, header, n, d);
    tiles_copy(X_t, X_rowmajor, nullptr, area, nullptr, nullptr, n, d, dtype, stream);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

KmxTiles kmx_tiles_view(char* area, int64_t n, int d) {
    const TileArea a = tile_area(n, d, 0);
    return {(const uint4*)(area + a.off_xt), (const float*)(area + a.off_norm), (const float*)(area + a.off_err),
            (const float*)area + KMX_TH_SCALE, a.S};
}

KmxKept kmx_tiles_kept(char* area, const unsigned int* absmax, int64_t n, int d, int k, int words) {
    const TileArea a = tile_area(n, d, k, words);
    KmxKept kept;
    kept.header = (unsigned int*)area;
    kept.absmax = absmax;
    kept.n = n;
    kept.words = words;
    for (int i = 0; i < words; ++i) kept.sums[i] = (unsigned long long*)(area + a.off_sums + i * a.sums_bytes);
    // (the lists of a labelling, which is over when the sums begin)
    kept.entry = (uint32_t*)(area + a.off_list);
    kept.entry_cluster = (uint32_t*)(area + a.off_thr);
    return kept;
}

char* kmx_tiles_half_norms(char* area, int64_t n, int d, int k) { return area + tile_area(n, d, k).off_half; }

// Labels of all samples for `centroids_t` (their packed copy `cpack` and half norms as the workspace
// holds them).  `status` null: labels whatever the state, those of kmx_assign_labels, whose half norms
// `half_norms` are then.  listed_out (or null): the number of samples without a certificate.  An iteration whose
// sums are kept hands over the labels before, the bits of max |x| per feature and max |w| (else null) and kmx_kept_span.
int32_t kmx_tiles_labels(const void* X_t, const void* X_rowmajor, const void* centroids_t, const void* cpack,
                         const void* half_norms, char* area, kmx_lloyd_status* status, uint32_t* labels, int64_t n,
                         int d, int dpad, int k, int dtype, hipStream_t stream, unsigned int* listed_out,
                         const uint32_t* labels_prev, const unsigned int* absmax, int span) {
    const TileArea a = tile_area(n, d, k);
    unsigned int* header = (unsigned int*)area;
    uint4* ct = (uint4*)(area + a.off_ct);
    float* hneg = (float*)(area + a.off_hneg);
    float2* cmax = (float2*)(area + a.off_cmax);
    const unsigned int* least = (const unsigned int*)(area + a.off_least);
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((tiles_centroids_kernel<float>), dim3((unsigned)a.n_blocks), dim3(64 * CENT_WAVES), 0, stream,
                           (const float*)centroids_t, ct, hneg, cmax, header, status, absmax, least, d, k, a.S, span);
    else
        hipLaunchKernelGGL((tiles_centroids_kernel<double>), dim3((unsigned)a.n_blocks), dim3(64 * CENT_WAVES), 0, stream,
                           (const double*)centroids_t, ct, hneg, cmax, header, status, absmax, least, d, k, a.S, span);
    // (an fp32 score: d + 1 roundings of partial sums, as many of the half norm)
    const bool match = status == nullptr && dtype == KMX_F32;
    const float prod_rho = match ? ULP * (float)(d + 8) : 0.0f;
    int32_t rc = KMX_ERR_UNSUPPORTED;
    switch (a.S) {
#define KMX_TILES_CASE(S_) case S_: rc = launch_labels_s<S_>(a, area, status, labels, labels_prev, n, prod_rho, stream); break
        KMX_TILES_CASE(1); KMX_TILES_CASE(2); KMX_TILES_CASE(3); KMX_TILES_CASE(4);
        KMX_TILES_CASE(5); KMX_TILES_CASE(6); KMX_TILES_CASE(7); KMX_TILES_CASE(8);
        KMX_TILES_CASE(9); KMX_TILES_CASE(10); KMX_TILES_CASE(11); KMX_TILES_CASE(12);
        KMX_TILES_CASE(13); KMX_TILES_CASE(14); KMX_TILES_CASE(15); KMX_TILES_CASE(16);
#undef KMX_TILES_CASE
    }
    if (rc != KMX_OK) return rc;
    int* list = (int*)(area + a.off_list);
    float* thr = (float*)(area + a.off_thr);
    int* rest = (int*)(area + a.off_rest);
    int64_t grid = kmx_cdiv(n, 32);
    if (grid > 4 * (int64_t)kmx_num_cus()) grid = 4 * (int64_t)kmx_num_cus();
#define KMX_TILES_RESOLVE(T, S_, M_)                                                                                     \
    hipLaunchKernelGGL((tiles_resolve_kernel<T, S_, M_>), dim3((unsigned)grid), dim3(256), 0, stream, (const T*)X_rowmajor,   \
                       (const T*)cpack, (const uint4*)(area + a.off_xt), ct, hneg, header, status, labels, list, thr,    \
                       rest, n, d, dpad, k, a.n_blocks, cmax, (const float*)half_norms, prod_rho, listed_out)
    switch (a.S) {
#define KMX_TILES_CASE(S_)                                                                         \
    case S_:                                                                                       \
        if (match) KMX_TILES_RESOLVE(float, S_, true);                                             \
        else if (dtype == KMX_F32) KMX_TILES_RESOLVE(float, S_, false);                            \
        else KMX_TILES_RESOLVE(double, S_, false);                                                 \
        break
        KMX_TILES_CASE(1); KMX_TILES_CASE(2); KMX_TILES_CASE(3); KMX_TILES_CASE(4);
        KMX_TILES_CASE(5); KMX_TILES_CASE(6); KMX_TILES_CASE(7); KMX_TILES_CASE(8);
        KMX_TILES_CASE(9); KMX_TILES_CASE(10); KMX_TILES_CASE(11); KMX_TILES_CASE(12);
        KMX_TILES_CASE(13); KMX_TILES_CASE(14); KMX_TILES_CASE(15); KMX_TILES_CASE(16);
#undef KMX_TILES_CASE
    }
#undef KMX_TILES_RESOLVE
    KMX_LAUNCH_CHECK();
    return kmx_lloyd_gemm_labels_listed(X_t, centroids_t, half_norms, labels, status, rest, header + KMX_TH_REST, n, d, k, dtype,
                                        stream, header + KMX_TH_LISTED, (n >> 3) + 1);
}
