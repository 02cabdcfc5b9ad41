// Sums per cluster of a run whose labels come from the half-precision copy (lloyd_tiles.hip): kept from one
// iteration to the next and corrected for the samples that moved.
//
// A rebuild reads every row of X, by cluster: the samples are sorted by label, and every stretch of the order is
// added up in registers, one atomic per feature, stretch and cluster.  Few labels change after the first
// iterations (1e6 x 256, 1 024 clusters within 3.5 standard deviations: 28, 7, 2 and 0.5 % in the second
// to fifth), so an iteration sorts only the samples that moved, twice each, taken off the old cluster and added to
// the new one.  That has to come to the same sums, so these are integers: round(x w 2^q) in 64 bits, what that leaves out,
// 2^p as fine, in another 64 and, in fp64, the rest of that in a third; sums and corrections of the same labels are then
// the same bits in any order.
//
// Such a term is rounded at a place that the largest of its feature sets, 80 binary places below it for 1e6 samples in
// fp32 and 119 in fp64.  So this is for data whose smallest |x| |w| but zero keep their digits (kmx_kept_fixed: 2^-54 and 2^-64
// of the largest; the smallest of 1e9 normal values is 2^-33 of the largest, an outlier of 1e11 among values of
// about 1 leaves them their digits).  Other runs, and those with NaN, infinities or fp64 values beyond fp32's range, add up in fp64 and
// rebuild every iteration, as all did before.  The wide fp32 step's own sums are fixed point of one word, whatever the
// range: so are these.
//
// Bound by the read of rows (a rebuild: 4.8 TB/s) or by a chain of trips to memory (corrections).  moves_sum_kernel, every
// iteration a rebuild before: 1e6 x 256 fp32, 1 024 clusters 216 us, now 211 / 114 / 45 / 29 / 24 in the first five
// iterations; 1e6 x 100 fp64, 100 clusters 177, now 181 / 170 / 59 / 38.  Runs by this step alone 6 106 -> 5 390, 2 168 -> 1 926 us.
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

__device__ __forceinline__ float read_lane(float v, int src) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src)); }
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
                                                            uint32_t* __restrict__ order, int64_t n, int items,
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
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < kept.words) kept.sums[j][i] = 0ull;
    }
}

// LPR lanes take a row, 16 bytes each (RPW = 64 / LPR rows per wave and load); the features past LPR * V on the second
// grid dimension.  A workgroup per stretch of the order, its four waves the rows in turn.  Clears counts
// for the next iteration.
template <typename T, int LPR, int WORDS>
__global__ __launch_bounds__(256, 4) void moves_sum_kernel(const T* __restrict__ X_rm, const T* __restrict__ sample_weight,
                                                        const uint32_t* __restrict__ order, const int* __restrict__ offsets,
                                                        int* __restrict__ counts, KmxKept kept,
                                                        const kmx_lloyd_status* __restrict__ status, int64_t n, int d, int k) {
    if (status->state != KMX_RUNNING) return;
    constexpr int V = 16 / (int)sizeof(T), RPW = 64 / LPR, FB = LPR * V, U = 4;  // (eight rows in flight: 272 for 216 us, half the waves)
    using Vec = typename KmxVec<T, V>::type;
    constexpr int REG = WORDS > 1 ? WORDS - 1 : 1;  // words of a feature in registers; the last one is in LDS
    __shared__ unsigned long long red[REG][4][FB], red_w[WORDS][4], last[FB];
    __shared__ int c_first;
    const bool corrected = sums_corrected(kept.header, n);
    const bool fixed = kept.header[KMX_TH_FIXED] != 0u;
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
    if (WORDS > 1)
        for (int s = threadIdx.x; s < FB; s += 256) last[s] = 0ull;
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
    double magic[V], magic_w = 0.0;  // of the first word
#pragma unroll
    for (int j = 0; j < V; ++j) magic[j] = fixed ? fix_magic(kmx_kept_exponent(kept.absmax, n, d, fl + j)) : 0.0;
    if (fixed) magic_w = fix_magic(kmx_kept_exponent(kept.absmax, n, d, d));
    // (its binary point `rest` places further down per word)
    auto magic_of = [&](const double first, const int word) __attribute__((always_inline)) {
        return __hiloint2double(__double2hiint(first) - ((word * rest) << 20), 0);
    };
    const T* __restrict__ col = X_rm + fl;

    auto stretch = [&](auto fixed_tag, const int p0, const int p1, const int c) __attribute__((always_inline)) {
        constexpr bool FIXED = decltype(fixed_tag)::value;
        unsigned long long sum[REG][V], w_sum[WORDS];
        double plain[V], w_plain = 0.0;
#pragma unroll
        for (int i = 0; i < WORDS; ++i) w_sum[i] = 0ull;
#pragma unroll
        for (int i = 0; i < REG; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j) sum[i][j] = 0ull;
#pragma unroll
        for (int j = 0; j < V; ++j) plain[j] = 0.0;
        // Terms x w: what a word leaves out, which has no error in fp32 and 2^-54 of itself in fp64, goes to the next; to the
        // last one only of a term that the others hold to less than 24 (fp32) or 55 digits, one in ten thousand of
        // normal values and next to none.  Those are read again and added to LDS: with the last word of all terms, in
        // registers, the first iteration's sums took 235 us instead of 182 (1e6 x 100, 100 clusters fp64) and 8 us more in
        // all iterations of 1e6 x 100, 128 clusters fp32 (one word 112, so 121).
        const unsigned long long digits = 1ull << (WORDS == 3 ? 55 - rest : 24);  // (in units of the first word)
        auto small = [&](const unsigned long long term) __attribute__((always_inline)) {  // |term| < digits
            return term + (digits - 1ull) < 2ull * digits - 1ull;
        };
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
            // (the weights: each lane the one that it holds, a wave every fourth group; beside the rows they cost half as
            // much again as two fp64 features)
            if ((((base - p0) >> 6) & 3) == wave) {
                if constexpr (FIXED) {
                    double left = (double)my_w;
#pragma unroll
                    for (int i = 0; i < WORDS; ++i) {
                        const double m = magic_of(magic_w, i), t = left + m;
                        w_sum[i] += to_fixed_q(t, m);
                        left -= t - m;
                    }
                } else {
                    w_plain += (double)my_w;
                }
            }
            const int n_here = p1 - base < 64 ? p1 - base : 64;
            for (int r0 = wave * RPW; r0 < n_here; r0 += 4 * RPW * U) {
                Vec xv[U];
                T wv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int src = r0 + 4 * RPW * u + sub;
                    const int idx = RPW == 1 ? __builtin_amdgcn_readlane(my_idx, src & 63) : __shfl(my_idx, src & 63, 64);
                    // (by all lanes, whichever of them have a row)
                    const T w_at = RPW == 1 ? read_lane(my_w, src & 63) : __shfl(my_w, src & 63, 64);
                    wv[u] = src < n_here ? w_at : T(0);
                    xv[u] = *reinterpret_cast<const Vec*>(col + (size_t)idx * (size_t)d);
                }
                unsigned int redo = 0u;  // bit u: some term of row u needs the last word (the same in all lanes)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if constexpr (FIXED) {
                        bool more = false;
#pragma unroll
                        for (int j = 0; j < V; ++j) {
                            const double x = (double)xv[u][j], w = (double)wv[u], first = magic[j], t = fma(x, w, first);
                            const unsigned long long term = to_fixed_q(t, first);
                            sum[0][j] += term;
                            if constexpr (WORDS == 3) {
                                const double m = magic_of(first, 1);
                                sum[1][j] += to_fixed_q(fma(x, w, first - t) + m, m);
                            }
                            if constexpr (WORDS > 1) more |= small(term) && x != 0.0;
                        }
                        if (WORDS > 1 && __any(more && wv[u] != T(0))) redo |= 1u << u;
                    } else if (r0 + 4 * RPW * u + sub < n_here) {  // (what is read twice may be infinite)
#pragma unroll
                        for (int j = 0; j < V; ++j) plain[j] = fma((double)xv[u][j], (double)wv[u], plain[j]);
                    }
                }
                while (FIXED && WORDS > 1 && redo != 0u) {
                    const int u = __builtin_ctz(redo), src = r0 + 4 * RPW * u + sub;
                    redo &= redo - 1u;
                    const int idx = __shfl(my_idx, src & 63, 64);
                    const T w_at = __shfl(my_w, src & 63, 64);
                    const double w = src < n_here ? (double)w_at : 0.0;
                    const Vec row = *reinterpret_cast<const Vec*>(col + (size_t)idx * (size_t)d);
                    int down = rest;
                    asm volatile("" : "+s"(down));  // (what is made of it stays in here)
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        const double x = (double)row[j], first = magic[j], t = fma(x, w, first);
                        double left = fma(x, w, first - t);
                        if constexpr (WORDS == 3) {
                            const double m = magic_of(first, 1);
                            left -= (left + m) - m;
                        }
                        const double m = __hiloint2double(__double2hiint(first) - (((WORDS - 1) * down) << 20), 0);
                        if (lane_on && fl + j >= f0 && small(to_fixed_q(t, first)) && left != 0.0)
                            atomicAdd(&last[fl + j - fb], to_fixed_q(left + m, m));
                    }
                }
            }
            my_idx = next_idx;
            my_w = next_w;
        }
        if constexpr (!FIXED) {
            // (their bits take the way of the first word)
#pragma unroll
            for (int off = LPR; off < 64; off <<= 1) {
#pragma unroll
                for (int j = 0; j < V; ++j) plain[j] += __shfl_xor(plain[j], off, 64);
            }
            w_plain = kmx_wave_sum(w_plain);
#pragma unroll
            for (int j = 0; j < V; ++j) sum[0][j] = (unsigned long long)__double_as_longlong(plain[j]);
            w_sum[0] = (unsigned long long)__double_as_longlong(w_plain);
        }
        // the rows of a wave, then the waves in LDS; one global atomic per feature and stretch
        constexpr int USED = FIXED ? REG : 1;
#pragma unroll
        for (int i = 0; i < USED; ++i) {
            if constexpr (FIXED) {
#pragma unroll
                for (int off = LPR; off < 64; off <<= 1)
#pragma unroll
                    for (int j = 0; j < V; ++j) sum[i][j] += (unsigned long long)__shfl_xor((long long)sum[i][j], off, 64);
            }
            if (sub == 0 && lane_on) {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (fl + j >= f0) red[i][wave][fl + j - fb] = sum[i][j];
            }
        }
#pragma unroll
        for (int i = 0; i < (FIXED ? WORDS : 1); ++i) {
            if (FIXED && __any(w_sum[i] != 0ull)) w_sum[i] = kmx_wave_sum(w_sum[i]);
            if (lane == 0) red_w[i][wave] = w_sum[i];
        }
        __syncthreads();
        const int here = d - fb < FB ? d - fb : FB;  // features of this part of the grid
        auto of = [&](const unsigned long long v) __attribute__((always_inline)) { return __longlong_as_double((long long)v); };
        for (int s = threadIdx.x; s < here; s += 256) {
            const size_t at = (size_t)(fb + s) * k + c;
            if constexpr (FIXED) {
#pragma unroll
                for (int i = 0; i < REG; ++i) {
                    const unsigned long long tot = red[i][0][s] + red[i][1][s] + red[i][2][s] + red[i][3][s];
                    if (tot != 0ull) atomicAdd(kept.sums[i] + at, tot);
                }
                if constexpr (WORDS > 1) {
                    const unsigned long long tot = last[s];
                    if (tot != 0ull) {
                        atomicAdd(kept.sums[WORDS - 1] + at, tot);
                        last[s] = 0ull;
                    }
                }
            } else {
                const double tot = (of(red[0][0][s]) + of(red[0][1][s])) + (of(red[0][2][s]) + of(red[0][3][s]));
                if (tot != 0.0) kmx_atomic_add(reinterpret_cast<double*>(kept.sums[0]) + at, tot);
            }
        }
        if (blockIdx.y == 0 && wave == 3 && lane < (FIXED ? WORDS : 1)) {
            const size_t at = (size_t)d * k + c;
            const unsigned long long* part = red_w[lane];
            if constexpr (FIXED) {
                const unsigned long long tot = part[0] + part[1] + part[2] + part[3];
                if (tot != 0ull) atomicAdd((lane == 0 ? kept.sums[0] : lane == 1 ? kept.sums[1] : kept.sums[2]) + at, tot);
            } else {
                const double tot = (of(part[0]) + of(part[1])) + (of(part[2]) + of(part[3]));
                if (tot != 0.0) kmx_atomic_add(reinterpret_cast<double*>(kept.sums[0]) + at, tot);
            }
        }
        __syncthreads();
    };

    int c = c_first, pos = P0;
    while (pos < P1 && c < k) {
        const int c_end = offsets[c + 1];  // wave-uniform
        const int p1 = c_end < P1 ? c_end : P1;
        if (p1 > pos) {
            if (fixed) stretch(std::true_type{}, pos, p1, c);
            else stretch(std::false_type{}, pos, p1, c);
            pos = p1;
        }
        ++c;
    }
}

template <typename T, int WORDS>
int32_t launch_sums(const void* X_rm, const void* w, const uint32_t* order, const int* offsets, int* counts, const KmxKept& kept,
                    const kmx_lloyd_status* status, int64_t n, int d, int k, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    // workgroups: a chunk each, or about four per compute unit where there are fewer chunks
    const unsigned gx = (unsigned)kmx_cdiv(n, CHUNK);
#define KMX_MOVES_SUM(LPR_)                                                                                                  \
    hipLaunchKernelGGL((moves_sum_kernel<T, LPR_, WORDS>), dim3(gx, (unsigned)kmx_cdiv(d, LPR_ * V)), dim3(256), 0, stream, (const T*)X_rm, \
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
                       (d + 1) * k, status);
    KMX_LAUNCH_CHECK();
#define KMX_SUMS(T, WORDS_) \
    return launch_sums<T, WORDS_>(X_rowmajor, w, order, offsets, counts, kept, status, n, d, k, stream)
    if (dtype == KMX_F64) KMX_SUMS(double, 3);
    if (kept.words == 1) KMX_SUMS(float, 1);
    KMX_SUMS(float, 2);
#undef KMX_SUMS
}
