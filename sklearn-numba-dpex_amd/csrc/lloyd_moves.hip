// Sums per cluster of a run whose labels come from the half-precision copy (lloyd_tiles.hip): kept from one
// iteration to the next and corrected for the samples that moved.
//
// A rebuild reads every row of X, by cluster: the samples are sorted by label, and every stretch of the order is
// added up in registers, one atomic per feature, stretch and cluster.  Few labels change after the first
// iterations (1e6 x 256, 1 024 clusters within 3.5 standard deviations: 28, 7, 2 and 0.5 % in the second
// to fifth), so an iteration sorts only the samples that moved, twice each, taken off the old cluster and added to
// the new one.  That has to be exact, so the sums are integers: term = round(x w 2^q) in 64 bits, and for fp64 the
// rest round((x w - term 2^-q) 2^p) in another 64, which leaves out 2^-80 of the largest term; sums
// and corrections of the same labels are then the same bits in any order, and the
// sum that an iteration divides has one rounding (fp64 additions in an order of their own before).
//
// Values that are not finite, and those of a feature whose largest fp32 does not hold, have no such terms.  They are
// added up as they are, in sums of their own that join in the end, and a run with any among its data rebuilds every
// iteration (of fp64 features below fp32's smallest only where there are no others: beside those they are good to 2^-240).
//
// Bound by the read of rows (a rebuild: 4.8 TB/s) or by a chain of trips to memory (corrections).  moves_sum_kernel, every
// iteration a rebuild before: 1e6 x 256 fp32, 1 024 clusters 216 us, now 215 / 112 / 45 / 27 / 22 in the first five
// iterations; 1e6 x 100 fp64, 100 clusters 177, now 180 / 165 / 47 / 27.  Runs 5 801 -> 5 220, 2 152 -> 1 920 us.
#include "lloyd_layout.h"
#include "lloyd_screen.h"

#include <type_traits>

namespace {

constexpr int COUNT_TILE = 2048;  // samples per workgroup and pass of the count
constexpr int COUNT_LDS_K = 4096; // clusters whose counts are gathered in LDS first
constexpr int CHUNK = 1024;       // positions per workgroup of a rebuild
constexpr int CHUNK_MIN = 16;     // and at least of a correction
constexpr uint32_t OFF = 0x80000000u;  // an entry that is taken off its cluster

// Whether the sums of this iteration are corrected: those of the iteration before are there, and what the
// label kernels know of changed labels (samples without a certificate counted as changed) leaves less to read
// than all rows.  The same in every kernel between the labels and the sums.
__device__ __forceinline__ bool sums_corrected(const unsigned int* __restrict__ header, int64_t n) {
    const int64_t listed = (int64_t)header[KMX_TH_LISTED], moved = (int64_t)header[KMX_TH_MOVED] + listed;
    return header[KMX_TH_KEEP] != 0u && listed <= (n >> 3) && 5 * moved <= 2 * n;
}

__device__ __forceinline__ double read_lane(double v, int src) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src), __builtin_amdgcn_readlane(__double2loint(v), src));
}

// Samples per cluster and every sample's rank among them (rebuild), or the same of the entries of the samples
// that moved, which are written here (correction); the number of changed labels.
__global__ __launch_bounds__(256) void moves_count_kernel(const uint32_t* __restrict__ labels,
                                                          const uint32_t* __restrict__ labels_prev, KmxKept kept,
                                                          int* __restrict__ counts, int* __restrict__ ranks,
                                                          kmx_lloyd_status* __restrict__ status, int64_t n, int k) {
    if (status->state != KMX_RUNNING) return;
    __shared__ int cnt[COUNT_LDS_K];
    __shared__ unsigned int changed_block, entries_s, base_s;
    const bool corrected = sums_corrected(kept.header, n);
    const bool in_lds = k <= COUNT_LDS_K;
    if (threadIdx.x == 0) changed_block = 0;
    unsigned int changed = 0;
    const int64_t n_tiles = (n + COUNT_TILE - 1) / COUNT_TILE;
    constexpr int U = COUNT_TILE / 256;
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t i0 = tile * COUNT_TILE + threadIdx.x;
        uint32_t lab[U], was[U];
        int rank_new[U], rank_old[U];
        unsigned int take = 0u;  // bit u: the sample is counted
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + 256 * u;
            lab[u] = i < n ? labels[i] : 0u;
            was[u] = i < n ? labels_prev[i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool here = i0 + 256 * u < n, differs = here && was[u] != lab[u];
            changed += differs ? 1u : 0u;
            take |= (corrected ? differs : here) ? 1u << u : 0u;
        }
        if (threadIdx.x == 0) entries_s = 0u;
        if (in_lds)
            for (int c = threadIdx.x; c < k; c += 256) cnt[c] = 0;
        __syncthreads();
        unsigned int slot = 0u;
        if (corrected && take != 0u) slot = atomicAdd(&entries_s, 2u * (unsigned int)__popc(take));
        int* __restrict__ const at = in_lds ? cnt : counts;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if ((take >> u) & 1u) {
                rank_new[u] = atomicAdd(&at[lab[u]], 1);
                if (corrected) rank_old[u] = atomicAdd(&at[was[u]], 1);
            }
        __syncthreads();
        if (in_lds) {
            // one global atomic per cluster present in the tile
            for (int c = threadIdx.x; c < k; c += 256) {
                const int v = cnt[c];
                if (v != 0) cnt[c] = atomicAdd(&counts[c], v);
            }
        }
        if (corrected && threadIdx.x == 0 && entries_s != 0u) base_s = atomicAdd(kept.header + KMX_TH_ENTRIES, entries_s);
        __syncthreads();
        slot += corrected ? base_s : 0u;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if ((take >> u) & 1u) {
                const int64_t i = i0 + 256 * u;
                const int add = in_lds ? cnt[lab[u]] : 0;
                if (corrected) {
                    kept.entry[slot] = (uint32_t)i;
                    kept.entry_cluster[slot] = lab[u];
                    ranks[slot] = add + rank_new[u];
                    kept.entry[slot + 1] = (uint32_t)i | OFF;
                    kept.entry_cluster[slot + 1] = was[u];
                    ranks[slot + 1] = (in_lds ? cnt[was[u]] : 0) + rank_old[u];
                    slot += 2u;
                } else {
                    ranks[i] = add + rank_new[u];
                }
            }
        __syncthreads();
    }
    if (changed) atomicAdd(&changed_block, changed);
    __syncthreads();
    if (threadIdx.x == 0 && changed_block) atomicAdd(&status->n_changed, changed_block);
}

// The order: samples (rebuild; the kept sums are cleared) or entries by cluster.
__global__ __launch_bounds__(256) void moves_scatter_kernel(const uint32_t* __restrict__ labels, KmxKept kept,
                                                            const int* __restrict__ offsets, const int* __restrict__ ranks,
                                                            uint32_t* __restrict__ order, int64_t n, int items, bool two,
                                                            const kmx_lloyd_status* __restrict__ status) {
    // (an iteration behind the end of the run: its labels may never have been written)
    if (status->state != KMX_RUNNING) return;
    const int64_t stride = (int64_t)gridDim.x * 256, first = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (sums_corrected(kept.header, n)) {
        const int64_t entries = (int64_t)kept.header[KMX_TH_ENTRIES];
        for (int64_t e = first; e < entries; e += stride) order[offsets[kept.entry_cluster[e]] + ranks[e]] = kept.entry[e];
        return;
    }
    for (int64_t i = first; i < n; i += stride) order[offsets[labels[i]] + ranks[i]] = (uint32_t)i;
    for (int64_t i = first; i < items; i += stride) {
        kept.hi[i] = 0ull;
        kept.odd[i] = 0.0;
        if (two) kept.lo[i] = 0ull;
    }
}

// LPR lanes take a row, 16 bytes each (RPW = 64 / LPR rows per wave and load); the features past LPR * V on the second
// grid dimension.  A workgroup per stretch of the order, its four waves the rows in turn.  Clears counts
// for the next iteration.
template <typename T, int LPR>
__global__ __launch_bounds__(256) void moves_sum_kernel(const T* __restrict__ X_rm, const T* __restrict__ sample_weight,
                                                        const uint32_t* __restrict__ order, const int* __restrict__ offsets,
                                                        int* __restrict__ counts, KmxKept kept,
                                                        const kmx_lloyd_status* __restrict__ status, int64_t n, int d, int k) {
    if (status->state != KMX_RUNNING) return;
    constexpr bool TWO = sizeof(T) == 8;
    constexpr int V = 16 / (int)sizeof(T), RPW = 64 / LPR, FB = LPR * V, U = 4;  // (eight rows in flight: 272 for 216 us, half the waves)
    using Vec = typename KmxVec<T, V>::type;
    __shared__ unsigned long long red_hi[4][FB + 1], red_lo[TWO ? 4 : 1][TWO ? FB + 1 : 1];
    __shared__ int c_first;
    const bool corrected = sums_corrected(kept.header, n);
    const bool finite = kept.header[KMX_TH_FINITE] != 0u;
    const int total = offsets[k];
    int chunk = CHUNK;
    if (corrected) {
        chunk = (total + (int)gridDim.x - 1) / (int)gridDim.x;
        chunk = chunk > CHUNK_MIN ? chunk : CHUNK_MIN;
    }
    const int64_t P0_64 = (int64_t)blockIdx.x * chunk;
    if (blockIdx.y == 0)
        for (int c = blockIdx.x * 256 + threadIdx.x; c < k; c += gridDim.x * 256) counts[c] = 0;
    if (P0_64 >= total) return;
    const int P0 = (int)P0_64, P1 = total - P0 < chunk ? total : P0 + chunk;
    if (threadIdx.x == 0) c_first = k;
    __syncthreads();
    // the (non-empty) cluster that holds position P0
    for (int c = threadIdx.x; c < k; c += 256)
        if (offsets[c] <= P0 && P0 < offsets[c + 1]) c_first = c;
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane / LPR, fb = (int)blockIdx.y * FB;
    const int f0 = fb + (lane % LPR) * V;
    // the lane's load starts at feature fl, moved back for the lane whose features do not all exist (what it
    // reads twice, and what lanes past the row's end read, is dropped below)
    const int fl = f0 + V <= d ? f0 : d - V;
    const bool lane_on = f0 < d;
    const int rest = kmx_kept_rest(n);
    double m_hi[V], m_lo[V];
    auto out_of_range = [&](const int f) __attribute__((always_inline)) {
        const unsigned int bits = kept.absmax[f];
        return kmx_not_finite(__uint_as_float(bits)) || (TWO && bits == 0u);
    };
    const bool w_as_is = out_of_range(d);
    unsigned int as_is = 0u;  // bit j: the values of the lane's feature j are added up as they are
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int q = kmx_kept_exponent(kept.absmax, n, d, fl + j);
        if (w_as_is || out_of_range(fl + j)) as_is |= 1u << j;
        m_hi[j] = fix_magic(q);
        m_lo[j] = fix_magic(q + rest);
    }
    const int q_w = kmx_kept_exponent(kept.absmax, n, d, d);
    const double mw_hi = fix_magic(q_w), mw_lo = fix_magic(q_w + rest);
    const T* __restrict__ col = X_rm + fl;

    auto stretch = [&](auto finite_tag, const int p0, const int p1, const int c) __attribute__((always_inline)) {
        constexpr bool FINITE = decltype(finite_tag)::value;
        unsigned long long hi[V], lo[V], w_hi = 0ull, w_lo = 0ull;
#pragma unroll
        for (int j = 0; j < V; ++j) hi[j] = lo[j] = 0ull;
        // each lane fetches one entry and its weight (a coalesced load and a gather per 64 entries), one group ahead of
        // the rows; lanes past the end hold the last one, weight 0
        auto fetch = [&](const int base, int& idx_out, T& w_out) __attribute__((always_inline)) {
            const int pl = base + lane;
            const uint32_t entry = order[pl < p1 ? pl : p1 - 1];
            idx_out = (int)(entry & ~OFF);
            const T raw_w = sample_weight[idx_out];
            w_out = pl < p1 ? ((entry & OFF) ? -raw_w : raw_w) : T(0);
        };
        int my_idx, next_idx = 0;
        T my_w, next_w = T(0);
        fetch(p0, my_idx, my_w);
        for (int base = p0; base < p1; base += 64) {
            if (base + 64 < p1) fetch(base + 64, next_idx, next_w);
            const int n_here = p1 - base < 64 ? p1 - base : 64;
            for (int r0 = wave * RPW; r0 < n_here; r0 += 4 * RPW * U) {
                Vec xv[U];
                double wv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int src = r0 + 4 * RPW * u + sub;
                    const int idx = RPW == 1 ? __builtin_amdgcn_readlane(my_idx, src & 63) : __shfl(my_idx, src & 63, 64);
                    // (by all lanes, whichever of them have a row)
                    const double w_at = RPW == 1 ? read_lane((double)my_w, src & 63) : (double)__shfl(my_w, src & 63, 64);
                    wv[u] = src < n_here ? w_at : 0.0;
                    xv[u] = *reinterpret_cast<const Vec*>(col + (size_t)idx * (size_t)d);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool there = r0 + 4 * RPW * u + sub < n_here;
                    if (!(fabs(wv[u]) < kmx_inf<double>())) {
                        // (a weight that is not finite: its terms as they are; from the next iteration on FINITE is false)
                        if (lane_on) {
                            kept.header[KMX_TH_ODD] = 1u;
#pragma unroll
                            for (int j = 0; j < V; ++j)
                                if (fl + j >= f0) kmx_atomic_add(kept.odd + (size_t)(fl + j) * k + c, (double)xv[u][j] * wv[u]);
                            if (f0 == 0) kmx_atomic_add(kept.odd + (size_t)d * k + c, wv[u]);
                        }
                        continue;
                    }
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        const double x = (double)xv[u][j];
                        if (!FINITE && (((as_is >> j) & 1u) != 0u || !(fabs(x) < kmx_inf<double>()))) {
                            if (lane_on && fl + j >= f0 && there && x != 0.0) kmx_atomic_add(kept.odd + (size_t)(fl + j) * k + c, x * wv[u]);
                            continue;
                        }
                        const double t = fma(x, wv[u], m_hi[j]);
                        hi[j] += to_fixed_q(t, m_hi[j]);
                        if constexpr (TWO) lo[j] += to_fixed_q(fma(x, wv[u], m_hi[j] - t) + m_lo[j], m_lo[j]);
                    }
                    if (!FINITE && w_as_is) {
                        if (lane_on && f0 == 0 && there) kmx_atomic_add(kept.odd + (size_t)d * k + c, wv[u]);
                        continue;
                    }
                    const double t = wv[u] + mw_hi;
                    w_hi += to_fixed_q(t, mw_hi);
                    if constexpr (TWO) w_lo += to_fixed_q((wv[u] + (mw_hi - t)) + mw_lo, mw_lo);
                }
            }
            my_idx = next_idx;
            my_w = next_w;
        }
        // the rows of a wave, then the waves in LDS; one global atomic per feature and stretch
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) {
#pragma unroll
            for (int j = 0; j < V; ++j) {
                hi[j] += (unsigned long long)__shfl_xor((long long)hi[j], off, 64);
                if constexpr (TWO) lo[j] += (unsigned long long)__shfl_xor((long long)lo[j], off, 64);
            }
            w_hi += (unsigned long long)__shfl_xor((long long)w_hi, off, 64);
            if constexpr (TWO) w_lo += (unsigned long long)__shfl_xor((long long)w_lo, off, 64);
        }
        if (sub == 0 && lane_on) {
#pragma unroll
            for (int j = 0; j < V; ++j)
                if (fl + j >= f0) {
                    red_hi[wave][fl + j - fb] = hi[j];
                    if constexpr (TWO) red_lo[wave][fl + j - fb] = lo[j];
                }
        }
        if (lane == 0) {
            red_hi[wave][FB] = w_hi;
            if constexpr (TWO) red_lo[wave][FB] = w_lo;
        }
        __syncthreads();
        const int here = d - fb < FB ? d - fb : FB;  // features of this part of the grid
        for (int s = threadIdx.x; s <= here; s += 256) {
            const bool weight = s == here;
            if (weight && blockIdx.y != 0) continue;
            const int slot = weight ? FB : s;
            const size_t at = (size_t)(weight ? d : fb + s) * k + c;
            const unsigned long long th = red_hi[0][slot] + red_hi[1][slot] + red_hi[2][slot] + red_hi[3][slot];
            if (th != 0ull) atomicAdd(kept.hi + at, th);
            if constexpr (TWO) {
                const unsigned long long tl = red_lo[0][slot] + red_lo[1][slot] + red_lo[2][slot] + red_lo[3][slot];
                if (tl != 0ull) atomicAdd(kept.lo + at, tl);
            }
        }
        __syncthreads();
    };

    int c = c_first, pos = P0;
    while (pos < P1 && c < k) {
        const int c_end = offsets[c + 1];  // wave-uniform
        const int p1 = c_end < P1 ? c_end : P1;
        if (p1 > pos) {
            if (finite) stretch(std::true_type{}, pos, p1, c);
            else stretch(std::false_type{}, pos, p1, c);
            pos = p1;
        }
        ++c;
    }
}

template <typename T>
int32_t launch_sums(const void* X_rm, const void* w, const uint32_t* order, const int* offsets, int* counts, const KmxKept& kept,
                    const kmx_lloyd_status* status, int64_t n, int d, int k, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    // workgroups: a chunk each, or about four per compute unit where there are fewer chunks
    const unsigned gx = (unsigned)kmx_cdiv(n, CHUNK);
#define KMX_MOVES_SUM(LPR_)                                                                                                  \
    hipLaunchKernelGGL((moves_sum_kernel<T, LPR_>), dim3(gx, (unsigned)kmx_cdiv(d, LPR_ * V)), dim3(256), 0, stream, (const T*)X_rm, \
                       (const T*)w, order, offsets, counts, kept, status, n, d, k)
    if (d <= 16 * V) KMX_MOVES_SUM(16);
    else if (d <= 32 * V) KMX_MOVES_SUM(32);
    else KMX_MOVES_SUM(64);
#undef KMX_MOVES_SUM
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

}  // namespace

// After kmx_tiles_labels: the kept sums are those of `labels`, and status->n_changed.  `bucket`: kmx_bucket_bytes, whose
// first k words (the counts) are zero on entry and on return.
int32_t kmx_lloyd_kept_sums(const void* X_rowmajor, const void* w, const uint32_t* labels_prev, const uint32_t* labels,
                            const KmxKept& kept, kmx_lloyd_status* status, char* bucket, int64_t n, int d, int k,
                            int32_t dtype, hipStream_t stream) {
    int* counts = reinterpret_cast<int*>(bucket);
    int* offsets = counts + k;
    uint32_t* order = reinterpret_cast<uint32_t*>(offsets + (k + 1));
    int* ranks = reinterpret_cast<int*>(order) + n;
    int64_t cg = kmx_cdiv(n, COUNT_TILE);
    if (cg > (int64_t)8 * kmx_num_cus()) cg = (int64_t)8 * kmx_num_cus();
    hipLaunchKernelGGL(moves_count_kernel, dim3((unsigned)cg), dim3(256), 0, stream, labels, labels_prev, kept, counts, ranks,
                       status, n, k);
    KMX_LAUNCH_CHECK();
    const int32_t rc = kmx_bucket_offsets(counts, offsets, status, k, stream);
    if (rc != KMX_OK) return rc;
    int64_t sg = kmx_cdiv(n, 256 * 4);
    if (sg > 2048) sg = 2048;
    hipLaunchKernelGGL(moves_scatter_kernel, dim3((unsigned)sg), dim3(256), 0, stream, labels, kept, offsets, ranks, order, n,
                       (d + 1) * k, dtype == KMX_F64, status);
    KMX_LAUNCH_CHECK();
    return dtype == KMX_F32 ? launch_sums<float>(X_rowmajor, w, order, offsets, counts, kept, status, n, d, k, stream)
                            : launch_sums<double>(X_rowmajor, w, order, offsets, counts, kept, status, n, d, k, stream);
}
