// Iterations of the screened fused steps (lloyd_mfma_screen.hip) that look only at the samples whose label
// can have changed.
//
// Once few labels change, most samples are nearer to their centroid than to any other one by more than
// the centroids have moved since (the triangle inequality; G. Hamerly, "Making k-means even faster", SIAM
// Data Mining 2010).  A sample's word holds how much nearer, rounded down, plus the drift that its
// label had seen by then; an iteration compares it with the drift by now and evaluates the sample only if it
// is not above it:
//   drift[c] += |c_new - c_old| + max over the others of |j_new - j_old|,
//   label unchanged if margin + drift[label] at evaluation > drift[label] now.
// The word of a sample that is passed over is read and not written: 4 bytes per sample instead of a row,
// its norm and two labels.
//
// Labels and sums are bit for bit those of the screened step.  There a label is that of the exact arg-max
// where the screen certifies it and of a fused multiply-add chain in feature order from -0.5 |c|^2
// elsewhere, and whatever the screen certifies that chain would find too.  Here a sample that is looked at goes
// the same way, screen first, and one is passed over only while the exact scores of its centroid and of any
// other are further apart than two errors E of the chain: with r of the margin left and D the distance to the
// own centroid those scores are at least r D + r^2 / 2 apart, and D is still at least D0 - (margin - r); the word
// leaves out as much of the margin as makes that exceed 2 E, with E for the largest centroid that means of the
// data can be.  Scores, margins and drift are those of scaled values (the largest coordinate in [2^12, 2^13)): squares of
// the data themselves leave fp32 from 1e-19 and 1e19 on, with the bounds made of them.  The sums are fixed point: a
// sample that moves is taken off its old cluster and added to the new one, exactly.
//
// bounds_kernel<ENTER> is an iteration over all samples that also writes the words and, in fp32, the rows of X side
// by side (samples here and there read feature by feature cost a 64-byte sector per value);
// bounds_kernel<!ENTER> is an iteration behind it: the words are read, the samples to look at gathered in a queue
// of the workgroup, and its waves screen the queue by 32.  The few samples that the screen cannot tell, or that
// move, are read from X_t.
//
// Bound by trips to memory and barriers, one after the other: 5e6 x 14 fp32 with 127 clusters, 4 to 7 % looked at, 46 to
// 54 us, of which the centroids' preparation takes 7, the words 7, the screen 7, the chain 3, the end of the
// iteration 14 (a screened step 104 to 112, the iteration that enters 192: 680 MB); 2e6 x 32 fp64 with 64 clusters, 10 %
// looked at, 48 to 56 (134, 195).  Runs of 20 and 12 iterations by this step alone: 2 431 -> 2 069 us, 2 653 -> 2 385 (with
// relocations and the iterations behind them).
#include "lloyd_layout.h"
#include "lloyd_screen.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v8d __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

constexpr int LABEL_BITS = 11;
constexpr uint32_t LABEL_MASK = (1u << LABEL_BITS) - 1u;  // the label's bits of a word, in place of the margin's last ones
constexpr int UNIT = 128;                 // samples of a wave's load of words
constexpr int GROUP = 10;                 // loads that are asked for together, a group ahead (four: 8 us more at 5e6 samples)
constexpr int TILE = 32;                  // samples that a wave screens together
constexpr size_t LDS_MAX = 156 * 1024;
constexpr int QUEUE_MAX = 24576, UNSURE_MAX = 640, MOVED_MAX = 512;

constexpr int bounds_waves(int esize, int nk) { return esize == 8 && nk > 2 ? 8 : 16; }

// Workgroups: one per compute unit, or fewer with a load of words for each wave.
constexpr int64_t bounds_grid(int64_t n, int waves, int cus) {
    const int64_t g = (n + (int64_t)UNIT * waves - 1) / ((int64_t)UNIT * waves);
    return g < cus ? g : cus;
}
// Whether the number of a sample within its workgroup's units, past the last of them included (the waves
// take the same number of units), fits an entry of the queue beside its label.  A partition of the GPU has fewer compute
// units, and more samples for each.
constexpr bool bounds_entries_fit(int64_t n, int waves, int cus) {
    const int64_t units = (n + UNIT - 1) / UNIT, per_step = bounds_grid(n, waves, cus) * waves;
    return (units + per_step - 1) / per_step * waves * UNIT <= (int64_t)1 << (32 - LABEL_BITS);
}
static_assert(bounds_entries_fit(((int64_t)1 << 29) - 1, 16, 256) && bounds_entries_fit((int64_t)1 << 29, 8, 256));
static_assert(!bounds_entries_fit(((int64_t)1 << 29) + 1, 16, 256));
static_assert(bounds_entries_fit((int64_t)1 << 26, 16, 32) && !bounds_entries_fit(((int64_t)1 << 26) + 1, 16, 32));
static_assert(bounds_entries_fit(1, 16, 1) && !bounds_entries_fit(((int64_t)1 << 21) + 1, 8, 1));

struct BoundsLds {
    size_t off_hi, off_lo, off_hneg, off_frag, off_half, off_drift, off_part, off_moved, off_unsure, off_queue, total;
    int kp, q_cap;
};
__host__ __device__ inline BoundsLds bounds_lds(int d, int k, int nk, int esize) {
    BoundsLds s;
    s.kp = (k + 31) & ~31;
    const size_t acc = (size_t)(d + 1) * k * 8;  // (feature-major, like the sums in memory; the end of the iteration reuses it)
    s.off_hi = (acc + 15) & ~(size_t)15;
    s.off_lo = s.off_hi + (size_t)s.kp * 16 * nk * 2;
    s.off_hneg = s.off_lo + (size_t)s.kp * 16 * nk * 2;
    s.off_frag = s.off_hneg + (size_t)s.kp * 4;
    s.off_half = s.off_frag + (size_t)s.kp * 16 * nk * esize;
    s.off_drift = s.off_half + (size_t)s.kp * esize;
    s.off_part = s.off_drift + (size_t)3 * s.kp * 4;
    s.off_moved = s.off_part + (size_t)s.kp * 2 * nk * 4;
    s.off_unsure = s.off_moved + (size_t)MOVED_MAX * 8;
    s.off_queue = s.off_unsure + (size_t)UNSURE_MAX * 6;
    const size_t room = s.off_queue < LDS_MAX ? (LDS_MAX - s.off_queue) / 4 : 0;
    s.q_cap = (int)(room < (size_t)QUEUE_MAX ? room : (size_t)QUEUE_MAX) & ~63;
    s.total = s.off_queue + (size_t)s.q_cap * 4;
    return s;
}

// Drift of every label (two copies: an iteration reads one and writes the other), words, rows.
struct BoundsArea {
    int ds;  // elements between rows
    size_t off_drift, off_words, off_rows, total;
};
inline BoundsArea bounds_area(int64_t n, int d, int k) {
    BoundsArea a;
    a.ds = (d + 7) & ~7;
    a.off_drift = 0;
    a.off_words = kmx_align256((size_t)2 * k * sizeof(float));
    a.off_rows = a.off_words + kmx_align256((size_t)kmx_cdiv(n, UNIT) * UNIT * sizeof(uint32_t));
    a.total = a.off_rows + kmx_align256((size_t)n * a.ds * sizeof(float));
    return a;
}

// What a chain of d fused multiply-adds from the half norm (d more) can be off by is chain_ulp (d + 8)
// (|x| R + R^2), R the largest centroid norm, and chain_tiny (d + 8) where products underflow: in fp32 those of the
// values themselves, not of scaled ones.
template <typename T>
constexpr float chain_ulp() { return sizeof(T) == 8 ? 2.3e-16f : 1.2e-7f; }
template <typename T>
__device__ __forceinline__ float chain_tiny(const float xs) { return sizeof(T) == 8 ? 2e-36f : fmaxf(2e-36f * xs * xs, 2e-36f); }

__device__ __forceinline__ float chain_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double chain_fma(double a, double b, double c) { return fma(a, b, c); }

// The margin of a sample, rounded down (zero: look at it next time, whatever the drift).  x_sq = |x|^2 to within
// rel, best and second scores to within e_score, e_chain: E above, all of scaled values.
__device__ __forceinline__ float margin_of(const float x_sq, const float best, const float second, const float rel,
                                           const float e_score, const float e_chain) {
    const float spread = rel * x_sq + 2.01f * e_score;
    const float sq = x_sq - 2.0f * best;
    const float own_most = sqrtf(fmaxf(sq + spread, 0.0f)) * 1.000001f;
    const float own_least = sqrtf(fmaxf(sq - spread, 0.0f)) * 0.999999f;
    const float next_least = sqrtf(fmaxf(x_sq - 2.0f * second - spread, 0.0f)) * 0.999999f;
    const float margin = next_least - own_most;
    if (!(margin > 0.0f)) return 0.0f;
    float keep = 2.01f * sqrtf(e_chain);
    const float base = own_least - margin;
    if (base > 0.0f) keep = fminf(keep, 2.02f * e_chain / base);
    const float out = (margin - keep) * 0.999999f;
    return out > 0.0f ? out : 0.0f;
}

template <typename TX, int NK, bool ENTER>
__global__ __launch_bounds__(64 * bounds_waves((int)sizeof(TX), NK)) void bounds_kernel(
    const TX* __restrict__ X_t, float* __restrict__ rows, const TX* __restrict__ sample_weight,
    const TX* __restrict__ centroids_t, const TX* __restrict__ before_t, uint32_t* __restrict__ labels_a,
    uint32_t* __restrict__ labels_b, uint32_t* __restrict__ words, const float* __restrict__ drift_in,
    float* __restrict__ drift_out, kmx_lloyd_status* __restrict__ status, const unsigned int* __restrict__ absmax,
    const int* __restrict__ q_exp, unsigned long long* __restrict__ gsum, int64_t n, int d, int k, int ds, const LloydTail<TX> tail) {
    constexpr bool F64 = sizeof(TX) == 8;
    constexpr int WAVES = bounds_waves((int)sizeof(TX), NK), THREADS = 64 * WAVES;
    extern __shared__ __align__(16) unsigned char bounds_raw[];
    const BoundsLds lay = bounds_lds(d, k, NK, (int)sizeof(TX));
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(bounds_raw);   // [d + 1][k]
    v8h* hi_s = reinterpret_cast<v8h*>(bounds_raw + lay.off_hi);                   // the screen's centroids, two fp16 parts
    v8h* lo_s = reinterpret_cast<v8h*>(bounds_raw + lay.off_lo);
    float* hneg_s = reinterpret_cast<float*>(bounds_raw + lay.off_hneg);           // -0.5 |c|^2, scaled; -inf past k
    TX* frag = reinterpret_cast<TX*>(bounds_raw + lay.off_frag);                   // the chain's centroids
    TX* half_s = reinterpret_cast<TX*>(bounds_raw + lay.off_half);                 // -0.5 |c|^2, -inf past k
    float* drift_s = reinterpret_cast<float*>(bounds_raw + lay.off_drift);         // drift by now
    float* step_s = drift_s + lay.kp;                                              // |c_new - c_old|, scaled
    float* norm_s = step_s + lay.kp;                                               // |c|, scaled, rounded up
    float* part_s = reinterpret_cast<float*>(bounds_raw + lay.off_part);           // its square, by eight features
    uint32_t* moved = reinterpret_cast<uint32_t*>(bounds_raw + lay.off_moved);     // [MOVED_MAX][2]: sample; old and new label
    uint32_t* u_index = reinterpret_cast<uint32_t*>(bounds_raw + lay.off_unsure);  // samples without a certificate
    uint16_t* u_label = reinterpret_cast<uint16_t*>(u_index + UNSURE_MAX);
    // samples to look at: number within the workgroup's units (bounds_entries_fit), then the label
    uint32_t* queue = reinterpret_cast<uint32_t*>(bounds_raw + lay.off_queue);
    __shared__ unsigned int queued, unsure_count, moved_count, changed_s;
    __shared__ int q_s[65];
    const int kp = lay.kp, q_cap = lay.q_cap;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, j = lane & 31;

    // Everything that the kernel starts from is asked for before anything is waited for, the state of the run included.
    const int state = __hip_atomic_load(&status->state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const unsigned int delta_word = __hip_atomic_load(&tail.clear_word[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    // the first words are on their way while the centroids are prepared
    const int64_t n_units = (n + UNIT - 1) / UNIT;
    const int64_t n_steps = (n_units + (int64_t)gridDim.x * WAVES - 1) / ((int64_t)gridDim.x * WAVES);  // the same for every wave
    auto unit_of = [&](const int64_t step) { return (int64_t)blockIdx.x + (step * WAVES + wave) * gridDim.x; };
    v2u ahead[GROUP];
    auto fetch = [&](const int64_t step) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < GROUP; ++g) {
            const int64_t u = unit_of(step + g);
            ahead[g] = v2u{0u, 0u};
            if (u < n_units) ahead[g] = *reinterpret_cast<const v2u*>(words + u * UNIT + lane * 2);
        }
    };
    if constexpr (!ENTER) fetch(0);

    const unsigned int my_absmax = lane < d ? absmax[lane] : 0u;  // (d <= 64)
    const int my_q = (int)threadIdx.x <= d ? q_exp[threadIdx.x] : 0;
    // eight features of a centroid per thread and pass
    TX now[8], was[8];
    auto centroid_of = [&](const int i) __attribute__((always_inline)) {
        const int c = i % kp, g = i / kp;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int f = 8 * g + e;
            const bool there = i < kp * 2 * NK && c < k && f < d;
            now[e] = there ? centroids_t[(size_t)f * k + c] : TX(0);
            was[e] = there && !ENTER ? before_t[(size_t)f * k + c] : TX(0);
        }
    };
    centroid_of((int)threadIdx.x);
    const float my_drift = !ENTER && (int)threadIdx.x < k ? drift_in[threadIdx.x] : 0.0f;
    if (state != KMX_RUNNING) return;
    const bool full_mode = delta_word == 0u;  // the sums are rebuilt, not corrected

    if ((int)threadIdx.x <= d) q_s[threadIdx.x] = my_q;
    if (threadIdx.x == 0) queued = unsure_count = moved_count = changed_s = 0u;
    for (int i = threadIdx.x; i < (d + 1) * k; i += THREADS) acc[i] = 0ull;
    // The largest coordinate sets the scale (a centroid beyond it overflows, and costs certificates only); the box
    // they span bounds the norm of any mean of the data.
    float x_most = __uint_as_float(my_absmax);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x_most = fmaxf(x_most, __shfl_xor(x_most, off, 64));
    const float xs = __uint_as_float((unsigned int)__builtin_amdgcn_readfirstlane((int)__float_as_uint(screen_scale(x_most))));
    float box = __uint_as_float(my_absmax) * xs;
    box *= box;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) box += __shfl_xor(box, off, 64);
    box = sqrtf(box) * 1.0002f;
    // Centroid (f, c) of the chain: fp32 v_mfma_f32_32x32x2, lane (c % 32, f % 2), pair f / 2, four pairs side by
    // side; fp64 v_mfma_f64_16x16x4, lane (c % 16, f % 4), step f / 4, two steps side by side.
    auto place = [&](const int f, const int c) __attribute__((always_inline)) {
        if constexpr (F64)
            return (((c >> 4) * (2 * NK) + (f >> 3)) * 64 + (f & 3) * 16 + (c & 15)) * 2 + ((f >> 2) & 1);
        else
            return (((c >> 5) * (2 * NK) + (f >> 3)) * 64 + (f & 1) * 32 + (c & 31)) * 4 + ((f >> 1) & 3);
    };
    for (int i = threadIdx.x; i < kp * 2 * NK; i += THREADS) {
        if (i >= THREADS) centroid_of(i);
        const int c = i % kp, g = i / kp;
        TX df = TX(0);
        v8h hi, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const TX diff = (now[e] - was[e]) * (TX)xs;
            df = chain_fma(diff, diff, df);
            frag[place(8 * g + e, c)] = now[e];
            const float v = (float)now[e] * xs;
            const _Float16 hb = (_Float16)v;
            hi[e] = hb;
            lo[e] = (_Float16)(v - (float)hb);
        }
        hi_s[((c >> 5) * NK + (g >> 1)) * 64 + (g & 1) * 32 + (c & 31)] = hi;
        lo_s[((c >> 5) * NK + (g >> 1)) * 64 + (g & 1) * 32 + (c & 31)] = lo;
        if (!ENTER) part_s[i] = (float)(df * (TX)1.00001) * 1.000001f;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < kp; c += THREADS) {
        TX sq = TX(0), sq_scaled = TX(0);
        float df = 0.0f;
#pragma unroll 1
        for (int g = 0; g < 2 * NK; ++g) {
            TX v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = frag[place(8 * g + e, c)];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sq = chain_fma(v[e], v[e], sq);  // (fused as in the other steps: near ties hang on it)
                const TX vs = v[e] * (TX)xs;
                sq_scaled = chain_fma(vs, vs, sq_scaled);
            }
            if (!ENTER) df += part_s[g * kp + c];
        }
        half_s[c] = c < k ? -(sq / TX(2)) : -kmx_inf<TX>();
        hneg_s[c] = c < k ? -((float)sq_scaled / 2.0f) : -kmx_inf<float>();
        norm_s[c] = sqrtf((float)sq_scaled * 1.000001f) * 1.000001f;
        step_s[c] = !ENTER && c < k ? sqrtf(df) * 1.00001f + 1e-17f : 0.0f;  // (squares that underflow: 1e-21 of the data)
    }
    __syncthreads();
    // The largest norm and the two largest steps, by every wave for itself (as bits: a NaN is the largest).
    unsigned int norm_top = 0u, top = 0u, next = 0u;
    int at = -1;
#pragma unroll 1
    for (int c = lane; c < k; c += 64) {
        const unsigned int b = __float_as_uint(step_s[c]);
        norm_top = max(norm_top, __float_as_uint(norm_s[c]));
        next = b > top ? top : (b > next ? b : next);
        at = b > top ? c : at;
        top = b > top ? b : top;
    }
#pragma unroll 1
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned int ot = (unsigned int)__shfl_xor((int)top, off, 64), on = (unsigned int)__shfl_xor((int)next, off, 64);
        const int oa = __shfl_xor(at, off, 64);
        norm_top = max(norm_top, (unsigned int)__shfl_xor((int)norm_top, off, 64));
        const bool take = ot > top || (ot == top && oa > at);
        next = max(min(top, ot), max(next, on));
        at = take ? oa : at;
        top = take ? ot : top;
    }
    const float norm_most = __uint_as_float(norm_top);
    const bool inside = norm_most <= box;  // (else: centroids from elsewhere; all samples are looked at)
    const float r_max = inside ? box : norm_most;
    for (int c = threadIdx.x; c < k; c += THREADS) {
        const float before = c < THREADS ? my_drift : drift_in[c];
        const float v = ENTER ? 0.0f : (before + (step_s[c] + __uint_as_float(c == at ? next : top))) * 1.000001f;
        drift_s[c] = v;
        if (blockIdx.x == 0) drift_out[c] = v;
    }
    __syncthreads();

    // bounds of a score's error: of the chain now and later, of the screen (E of lloyd_mfma_screen.hip)
    const float n_round = (float)(d + 8), rel = n_round * 1.2e-7f;
    const float chain_0 = n_round * chain_tiny<TX>(xs);
    const float cmax = norm_most, hmax = 0.5f * cmax * cmax;
    const float round_term = SCR_ERR_ROUND * 51.0f * (float)NK, abs_term = SCR_ERR_ABS * sqrtf((float)d);
    const float scr_x = 1.001f * ((F64 ? SCR_ERR_SPLIT_F64 : SCR_ERR_SPLIT) + round_term) * cmax + abs_term;
    const float scr_0 = 1.001f * (round_term + (F64 ? SCR_ERR_HNEG_F64 : 0.0f)) * hmax + abs_term * cmax;
    const float neg_inf = -kmx_inf<float>();
    float pos_inf = kmx_inf<float>();
    asm volatile("" : "+s"(pos_inf));  // (keeps the first maximum of a group an instruction the compiler sees as such)
    unsigned int changed = 0u, looked = 0u;

    auto add_term = [&](const int f, const double v, const uint32_t to, const uint32_t from) __attribute__((always_inline)) {
        const unsigned long long term = to_fixed_q(v, fix_magic(q_s[f]));
        atomicAdd(acc + (size_t)f * k + to, term);
        if (!full_mode) atomicSub(acc + (size_t)f * k + from, term);
    };
    // the term of value f of a sample (f = d: of its weight): x * w is exact in fp64 for fp32 inputs, one rounding to
    // a multiple of 2^-q
    auto add_value = [&](const int f, const double x, const double wd, const uint32_t to, const uint32_t from)
                         __attribute__((always_inline)) {
        const double magic = fix_magic(q_s[f]);
        add_term(f, f < d ? fma(x, wd, magic) : wd + magic, to, from);
    };
    // A sample's new label and word, by its owner lane.  A sample that the sums have to hear of goes on a list, the
    // values of which are fetched together in the end.
    auto settle = [&](const uint32_t idx, const uint32_t old_label, const uint32_t label, const float margin)
                      __attribute__((always_inline)) {
        const float v = (margin + drift_s[label]) * 0.9999998f;
        words[idx] = (margin > 0.0f ? (__float_as_uint(v) & ~LABEL_MASK) : 0u) | label;
        const bool differs = label != old_label;
        if (differs) labels_a[idx] = label;
        if (ENTER || differs) labels_b[idx] = label;
        changed += differs ? 1u : 0u;
        if (full_mode || differs) {
            const unsigned int slot = atomicAdd(&moved_count, 1u);
            if (slot < (unsigned int)MOVED_MAX) {
                moved[2 * slot] = idx;
                moved[2 * slot + 1] = old_label | label << 16;
            } else {
                const double wd = (double)sample_weight[idx];
                for (int f = 0; f < d; ++f) add_value(f, (double)X_t[(size_t)f * n + idx], wd, label, old_label);
                add_value(d, 0.0, wd, label, old_label);
            }
        }
    };
    auto value_of = [&](const uint32_t idx, const int f) __attribute__((always_inline)) {
        if constexpr (ENTER || F64) return X_t[(size_t)f * n + idx];
        else return rows[(size_t)idx * ds + f];
    };

    // Up to 32 samples (lane (j, h): sample j) by the chain.  Their margins are within its errors: none.
    auto chain = [&](const bool valid, const uint32_t idx, const uint32_t old_label) __attribute__((always_inline)) {
        if constexpr (!F64) {
            float x[8 * NK];  // feature 2 p + h
#pragma unroll
            for (int p = 0; p < 8 * NK; ++p) x[p] = value_of(idx, 2 * p + h < d ? 2 * p + h : 0);
#pragma unroll
            for (int p = 0; p < 8 * NK; ++p) x[p] = 2 * p + h < d ? x[p] : 0.0f;
            float best = neg_inf;
            int arg = 0x7fffffff;
            for (int cb = 0; cb < kp / 32; ++cb) {
                v16f s;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f v = *reinterpret_cast<const v4f*>(half_s + 32 * cb + 8 * q + 4 * h);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * q + e] = v[e];
                }
                const v4f* __restrict__ fr = reinterpret_cast<const v4f*>(frag) + (size_t)cb * (2 * NK) * 64 + lane;
#pragma unroll
                for (int p4 = 0; p4 < 2 * NK; ++p4) {
                    const v4f a = fr[p4 * 64];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (8 * p4 + 2 * e < d) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], x[4 * p4 + e], s, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {  // centroid 32 cb + 8 (r / 4) + 4 h + r % 4: increasing inside a lane
                    const bool up = s[r] > best;
                    arg = up ? 32 * cb + 8 * (r >> 2) + 4 * h + (r & 3) : arg;
                    best = up ? s[r] : best;
                }
            }
            const float ob = __shfl_xor(best, 32, 64);
            const int oc = __shfl_xor(arg, 32, 64);
            if (ob > best || (ob == best && oc < arg)) {
                best = ob;
                arg = oc;
            }
            if (arg == 0x7fffffff) arg = 0;  // no score compares: the reference's running arg-min keeps 0
            if (valid && h == 0) settle(idx, old_label, (uint32_t)arg, 0.0f);
        } else {
            constexpr int NS = 4 * NK;  // steps of four features; lane (g, m): feature 4 s + g of samples m and 16 + m
            const int g = lane >> 4, m = lane & 15;
            uint32_t idx2[2], old2[2];
            bool valid2[2];
            double x[2][NS];
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                idx2[col] = (uint32_t)__shfl((int)idx, 16 * col + m, 64);
                old2[col] = (uint32_t)__shfl((int)old_label, 16 * col + m, 64);
                valid2[col] = __shfl((int)valid, 16 * col + m, 64) != 0;
#pragma unroll
                for (int s = 0; s < NS; ++s) x[col][s] = (double)value_of(idx2[col], 4 * s + g < d ? 4 * s + g : 0);
            }
            double best[2];
            int arg[2];
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                best[col] = -kmx_inf<double>();
                arg[col] = 0x7fffffff;
#pragma unroll
                for (int s = 0; s < NS; ++s) x[col][s] = 4 * s + g < d ? x[col][s] : 0.0;
            }
            for (int cb = 0; cb < kp / 16; ++cb) {
                const TX* hp = half_s + 16 * cb + g;
                const v4d start = {(double)hp[0], (double)hp[4], (double)hp[8], (double)hp[12]};
                v4d s[2] = {start, start};
                const v2d* __restrict__ fr = reinterpret_cast<const v2d*>(frag) + (size_t)cb * (2 * NK) * 64 + lane;
#pragma unroll
                for (int s2 = 0; s2 < 2 * NK; ++s2) {
                    const v2d a = fr[s2 * 64];
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int col = 0; col < 2; ++col)
                            s[col] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], x[col][2 * s2 + e], s[col], 0, 0, 0);
                }
#pragma unroll
                for (int col = 0; col < 2; ++col)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {  // centroid 16 cb + g + 4 r: increasing inside a lane
                        const double v = s[col][r];
                        const bool up = v > best[col];
                        arg[col] = up ? 16 * cb + g + 4 * r : arg[col];
                        best[col] = up ? v : best[col];
                    }
            }
#pragma unroll
            for (int col = 0; col < 2; ++col) {
#pragma unroll
                for (int off = 16; off <= 32; off <<= 1) {
                    const double ob = __shfl_xor(best[col], off, 64);
                    const int oc = __shfl_xor(arg[col], off, 64);
                    if (ob > best[col] || (ob == best[col] && oc < arg[col])) {
                        best[col] = ob;
                        arg[col] = oc;
                    }
                }
                if (arg[col] == 0x7fffffff) arg[col] = 0;  // no score compares: the reference's running arg-min keeps 0
                if (valid2[col] && g == 0) settle(idx2[col], old2[col], (uint32_t)arg[col], 0.0f);
            }
        }
    };

    // 32 samples through the screen: x[s][e] = feature 16 s + 8 h + e of sample j (zero past d).
    auto screen = [&](const bool valid, const uint32_t idx, const uint32_t old_label, const float(&x)[NK][8])
                      __attribute__((always_inline)) {
        v8h xh[NK], xl[NK];
        float sq = 0.0f;
        {
            const float xs_sc = xs;
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                unsigned int hw[4], lw[4];
                split_eight(x[s][0], x[s][1], x[s][2], x[s][3], x[s][4], x[s][5], x[s][6], x[s][7], xs_sc, hw, lw);
                xh[s] = __builtin_bit_cast(v8h, make_uint4(hw[0], hw[1], hw[2], hw[3]));
                xl[s] = __builtin_bit_cast(v8h, make_uint4(lw[0], lw[1], lw[2], lw[3]));
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = x[s][e] * xs_sc;
                    sq = fmaf(v, v, sq);
                }
            }
        }
        sq += __shfl_xor(sq, 32, 64);
        // Arg-max by groups of eight registers, with the second largest of the group maxima; the eight
        // registers of the winning group are kept as they are, the place inside is looked up once.
        float best = neg_inf, second = neg_inf;
        unsigned int code = 0;
        double w0, w1, w2, w3;
        asm volatile("" : "=v"(w0), "=v"(w1), "=v"(w2), "=v"(w3));
        for (int cb = 0; cb < kp / 32; ++cb) {
            v16f sc;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f v = *reinterpret_cast<const v4f*>(hneg_s + 32 * cb + 8 * q + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e) sc[4 * q + e] = v[e];
            }
#pragma unroll
            for (int s = 0; s < NK; ++s) {
                const v8h ah = hi_s[(cb * NK + s) * 64 + lane], al = lo_s[(cb * NK + s) * 64 + lane];
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, xh[s], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, xl[s], sc, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, xh[s], sc, 0, 0, 0);
            }
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                float m = __builtin_amdgcn_fmed3f(sc[8 * g], sc[8 * g + 1], pos_inf);
#pragma unroll
                for (int r = 2; r < 8; r += 2)
                    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(m), "v"(sc[8 * g + r]), "v"(sc[8 * g + r + 1]));
                asm("v_med3_f32 %0, %1, %2, %3" : "=v"(second) : "v"(best), "v"(second), "v"(m));
                if (m > best) {  // strict: the earlier group keeps a tie
                    best = m;
                    code = (unsigned int)(2 * cb + g);
                    const v8d ad = __builtin_bit_cast(v8d, sc);
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w0) : "v"(ad[4 * g]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w1) : "v"(ad[4 * g + 1]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w2) : "v"(ad[4 * g + 2]));
                    asm volatile("v_mov_b64 %0, %1" : "+v"(w3) : "v"(ad[4 * g + 3]));
                }
            }
        }
        float sv[8];
        {
            const float2 p0 = __builtin_bit_cast(float2, w0), p1 = __builtin_bit_cast(float2, w1);
            const float2 p2 = __builtin_bit_cast(float2, w2), p3 = __builtin_bit_cast(float2, w3);
            sv[0] = p0.x; sv[1] = p0.y; sv[2] = p1.x; sv[3] = p1.y;
            sv[4] = p2.x; sv[5] = p2.y; sv[6] = p3.x; sv[7] = p3.y;
        }
        unsigned int pos = 7u, n_eq = 0u;
#pragma unroll
        for (int r = 7; r >= 0; --r) {
            const bool eq = sv[r] == best;
            pos = eq ? (unsigned int)r : pos;
            n_eq += eq ? 1u : 0u;
            const float other = eq ? neg_inf : sv[r];
            second = other > second ? other : second;
        }
        second = n_eq > 1u ? best : second;
        const unsigned int reg = (code & 1u) * 8u + pos;
        int label = (int)(32u * (code >> 1) + 8u * (reg >> 2) + 4u * (unsigned int)h + (reg & 3u));
        {
            const float ob = __shfl_xor(best, 32, 64), o2 = __shfl_xor(second, 32, 64);
            const int oc = __shfl_xor(label, 32, 64);
            const float lower = ob < best ? ob : best, upper2 = second > o2 ? second : o2;
            second = lower > upper2 ? lower : upper2;
            if (ob > best || (ob == best && oc < label)) {
                best = ob;
                label = oc;
            }
        }
        // certain when the lead exceeds two errors (a NaN anywhere makes it uncertain)
        const float norm = sqrtf(sq) * 1.001f;
        const float e_scr = fmaf(scr_x, norm, scr_0);
        const bool owner = valid && h == 0;
        const bool unsure = owner && !(best - second > 2.01f * e_scr);
        if (owner && !unsure) {
            const float e_chain = n_round * chain_ulp<TX>() * (norm + r_max) * r_max + chain_0;
            settle(idx, old_label, (uint32_t)label, margin_of(sq, best, second, rel, e_scr, e_chain));
        }
        const unsigned long long um = __ballot(unsure);
        if (um != 0ull) {
            const unsigned int n_unsure = (unsigned int)__popcll(um);
            unsigned int base = 0u;
            if (lane == 0) base = atomicAdd(&unsure_count, n_unsure);
            base = (unsigned int)__builtin_amdgcn_readfirstlane((int)base);
            if (base + n_unsure <= (unsigned int)UNSURE_MAX) {
                if (unsure) {
                    const unsigned int slot = base + (unsigned int)__popcll(um & ((1ull << lane) - 1ull));
                    u_index[slot] = idx;
                    u_label[slot] = (uint16_t)old_label;
                }
            } else {
                // (no room: at once, a lane per sample and one centroid after the other; slots below the limit that
                // this leaves unwritten are marked)
                if (unsure) {
                    const unsigned int slot = base + (unsigned int)__popcll(um & ((1ull << lane) - 1ull));
                    if (slot < (unsigned int)UNSURE_MAX) u_index[slot] = 0xffffffffu;
                    TX top = -kmx_inf<TX>();
                    int arg = 0;  // (no score compares: the reference's running arg-min keeps 0)
                    for (int c = 0; c < k; ++c) {
                        TX v = half_s[c];
                        for (int f = 0; f < d; ++f) v = chain_fma(value_of(idx, f), frag[place(f, c)], v);
                        arg = v > top ? c : arg;
                        top = v > top ? v : top;
                    }
                    settle(idx, old_label, (uint32_t)arg, 0.0f);
                }
            }
        }
    };

    if constexpr (ENTER) {
        const int64_t n_tiles = (n + TILE - 1) / TILE, stride = (int64_t)gridDim.x * WAVES;
        TX raw[NK][8];
        uint32_t old_label = 0u;
        auto request = [&](const int64_t t) __attribute__((always_inline)) {
            const int64_t i = t * TILE + j, ic = i < n ? i : n - 1;
#pragma unroll
            for (int s = 0; s < NK; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int f = 16 * s + 8 * h + e;
                    raw[s][e] = X_t[(size_t)(f < d ? f : d - 1) * n + ic];
                }
            old_label = labels_a[ic];
        };
        constexpr bool EARLY = !F64 && NK <= 2;  // (registers: the next tile's values during this one)
        const int64_t first = (int64_t)blockIdx.x * WAVES + wave;
        if (EARLY && first < n_tiles) request(first);
        for (int64_t t = first; t < n_tiles; t += stride) {
            if (!EARLY) request(t);
            const int64_t i = t * TILE + j;
            const bool valid = i < n;
            float x[NK][8];
#pragma unroll
            for (int s = 0; s < NK; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[s][e] = 16 * s + 8 * h + e < d ? (float)raw[s][e] : 0.0f;
            const uint32_t old_now = old_label;
            if (EARLY && t + stride < n_tiles) request(t + stride);
            if (valid) {
#pragma unroll
                for (int s = 0; s < NK; ++s)
                    if (16 * s + 8 * h < ds) {
                        float* __restrict__ out = rows + (size_t)i * ds + 16 * s + 8 * h;
                        *reinterpret_cast<v4f*>(out) = v4f{x[s][0], x[s][1], x[s][2], x[s][3]};
                        *reinterpret_cast<v4f*>(out + 4) = v4f{x[s][4], x[s][5], x[s][6], x[s][7]};
                    }
            }
            screen(valid, (uint32_t)(valid ? i : n - 1), old_now, x);
        }
    } else {
        auto work_off = [&](const int count) __attribute__((always_inline)) {
            v4f raw[NK][2];
            uint32_t idx = 0u, old_label = 0u;
            bool valid = false;
            auto request = [&](const int t) __attribute__((always_inline)) {
                valid = t * TILE + j < count;
                const uint32_t entry = queue[valid ? t * TILE + j : t * TILE];
                const uint32_t local = entry >> LABEL_BITS;
                old_label = entry & LABEL_MASK;
                idx = (blockIdx.x + (local / UNIT) * gridDim.x) * UNIT + local % UNIT;
                const float* __restrict__ row = rows + (size_t)idx * ds;
#pragma unroll
                for (int s = 0; s < NK; ++s) {
                    const int f = 16 * s + 8 * h < ds ? 16 * s + 8 * h : 0;
                    raw[s][0] = *reinterpret_cast<const v4f*>(row + f);
                    raw[s][1] = *reinterpret_cast<const v4f*>(row + f + 4);
                }
            };
            constexpr bool EARLY = NK <= 2;  // (registers: the next tile's rows during this one)
            if (EARLY && wave * TILE < count) request(wave);
            for (int t = wave; t * TILE < count; t += WAVES) {
                if (!EARLY) request(t);
                float x[NK][8];
#pragma unroll
                for (int s = 0; s < NK; ++s)
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[s][e] = 16 * s + 8 * h + e < d ? raw[s][e >> 2][e & 3] : 0.0f;
                const uint32_t idx_now = idx, old_now = old_label;
                const bool valid_now = valid;
                if (EARLY && (t + WAVES) * TILE < count) request(t + WAVES);
                screen(valid_now, idx_now, old_now, x);
            }
        };
        int room = q_cap / (UNIT * WAVES);  // loads of words per wave that are sure to fit the queue (the same in all threads)
        for (int64_t step = 0; step < n_steps;) {
            const int now = room < GROUP ? room : GROUP;
            v2u at[GROUP];
#pragma unroll
            for (int g = 0; g < GROUP; ++g) at[g] = ahead[g];
            const int64_t base_step = step;
            step += now;
            room -= now;
            const bool more = step < n_steps && room > 0;  // (the same for the whole workgroup)
            if (more) fetch(step);
            // (the group's reads of the LDS, and its place in the queue, each in one go)
            float by_now[GROUP][2];
#pragma unroll
            for (int g = 0; g < GROUP; ++g)
#pragma unroll
                for (int e = 0; e < 2; ++e) by_now[g][e] = drift_s[at[g][e] & LABEL_MASK];  // (past n: some word of the LDS)
            unsigned long long look[GROUP][2];
            unsigned int total = 0u;
#pragma unroll
            for (int g = 0; g < GROUP; ++g) {
                const int64_t i0 = unit_of(base_step + g) * UNIT + lane * 2;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float margin = __uint_as_float(at[g][e] & ~LABEL_MASK);
                    look[g][e] = __ballot(g < now && i0 + e < n && (full_mode || !inside || !(margin > by_now[g][e])));
                    total += (unsigned int)__popcll(look[g][e]);
                }
            }
            if (total != 0u) {
                unsigned int base = 0u;
                if (lane == 0) base = atomicAdd(&queued, total);
                base = (unsigned int)__builtin_amdgcn_readfirstlane((int)base);
#pragma unroll
                for (int g = 0; g < GROUP; ++g)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        if ((look[g][e] >> lane) & 1ull) {
                            const unsigned int slot = base + (unsigned int)__popcll(look[g][e] & ((1ull << lane) - 1ull));
                            queue[slot] = (uint32_t)(((base_step + g) * WAVES + wave) * UNIT + lane * 2 + e) << LABEL_BITS |
                                          (at[g][e] & LABEL_MASK);
                        }
                        base += (unsigned int)__popcll(look[g][e]);
                    }
            }
            if (more) continue;
            __syncthreads();
            int waiting = (int)queued;
            if (step >= n_steps || q_cap - waiting < UNIT * WAVES) {
                work_off(waiting);
                looked += (unsigned int)waiting;
                __syncthreads();
                if (threadIdx.x == 0) queued = 0u;
                waiting = 0;
            }
            room = (q_cap - waiting) / (UNIT * WAVES);
            if (step < n_steps) fetch(step);
            __syncthreads();  // (everyone has read the count, or it is zero again)
        }
    }
    __syncthreads();
    {
        const int count = (int)min(unsure_count, (unsigned int)UNSURE_MAX);
        for (int t = wave; t * TILE < count; t += WAVES) {
            const int e = t * TILE + j;
            const uint32_t idx = e < count ? u_index[e] : 0xffffffffu;
            const bool valid = idx != 0xffffffffu;
            chain(valid, valid ? idx : 0u, valid ? (uint32_t)u_label[e] : 0u);
        }
    }
    if (changed) atomicAdd(&changed_s, changed);
    __syncthreads();
    // the samples that move: thread (entry, value), four reads in flight
    {
        const int total = (int)min(moved_count, (unsigned int)MOVED_MAX) * (d + 1);
        for (int first = 0; first < total; first += 4 * THREADS) {
            double xv[4], wv[4];
            uint32_t lab[4];
            int f[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int item = first + u * THREADS + (int)threadIdx.x;
                f[u] = -1;
                xv[u] = wv[u] = 0.0;
                lab[u] = 0u;
                if (item < total) {
                    const int e = item / (d + 1);
                    f[u] = item - e * (d + 1);
                    const uint32_t idx = moved[2 * e];
                    lab[u] = moved[2 * e + 1];
                    wv[u] = (double)sample_weight[idx];
                    if (f[u] < d) xv[u] = (double)value_of(idx, f[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (f[u] >= 0) add_value(f[u], xv[u], wv[u], lab[u] >> 16, lab[u] & 0xffffu);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (changed_s) atomicAdd(&status->n_changed, changed_s);
        if (unsure_count) atomicAdd(tail.clear_word, unsure_count);
        if (!ENTER && looked) atomicAdd(tail.looked_word, looked);
        if (ENTER && blockIdx.x == 0) atomicAdd(tail.looked_word, (unsigned int)n);
    }
    // (every workgroup starts at another word: they finish together)
    const int n_out = (d + 1) * k;
    const int rot = (int)(((int64_t)blockIdx.x * n_out) / gridDim.x);
    for (int jy = threadIdx.x; jy < n_out; jy += THREADS) {
        const int jx = jy + rot < n_out ? jy + rot : jy + rot - n_out;
        const unsigned long long v = acc[jx];
        if (v) atomicAdd(gsum + jx, v);
    }
    // the last workgroup ends the iteration
    if (lloyd_last_workgroup(status)) {
        lloyd_small_finalize_body<TX, true, true>(gsum, q_exp, tail, reinterpret_cast<TX*>(bounds_raw));
        if (threadIdx.x == 0) status->ticket = 0u;
    }
}

// Root mean square distance of a thousand samples to their centroids, for the host (system scope): how far
// centroids may move before bounds are of no use.  One workgroup; 64 samples in a row at sixteen places (a thousand
// places take 30 to 110 us, a page of memory and its translation per value).  Zero, no use at all, for data beyond
// these magnitudes: an fp32 chain whose products leave its range does not find what the screen certifies, and which
// sample goes which way then decides its label.  Rounding to a multiple of fp32's smallest normal number is 4e-3 of
// scaled squares at the lower end, a hundredth of the least lead that the screen certifies where the largest centroid is
// a tenth of the largest coordinate; at the upper end 64 squares stay within fp32.
constexpr float BOUNDS_LEAST = 5.7e-14f, BOUNDS_MOST = 1.1e18f;  // 2^-44, 2^60
template <typename TX>
__global__ __launch_bounds__(1024) void spread_kernel(const TX* __restrict__ X_t, const TX* __restrict__ centroids_t,
                                                      const uint32_t* __restrict__ labels,
                                                      const kmx_lloyd_status* __restrict__ status,
                                                      const unsigned int* __restrict__ absmax,
                                                      unsigned long long* __restrict__ out, int64_t n, int d, int k) {
    if (status->state != KMX_RUNNING) return;
    unsigned int most = (int)threadIdx.x < d ? absmax[threadIdx.x] : 0u;  // (d <= 64: the first wave)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) most = max(most, (unsigned int)__shfl_xor((int)most, off, 64));
    const bool within = __uint_as_float(most) >= BOUNDS_LEAST && __uint_as_float(most) <= BOUNDS_MOST;
    __shared__ double scratch[16];
    const int64_t place = (int64_t)(threadIdx.x >> 6) * n / 16 + (threadIdx.x & 63);
    const int64_t i = place < n ? place : n - 1;
    const uint32_t c = labels[i];
    double sq = 0.0;
    if (c < (uint32_t)k) {
#pragma unroll 16
        for (int f = 0; f < d; ++f) {
            const double e = (double)X_t[(size_t)f * n + i] - (double)centroids_t[(size_t)f * k + c];
            sq = fma(e, e, sq);
        }
    }
    const double total = kmx_block_sum<double>(sq, scratch);
    if (threadIdx.x == 0)
        __hip_atomic_store(out, (unsigned long long)__double_as_longlong(within ? sqrt(total / 1024.0) : 0.0),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename TX, int NK>
int32_t launch_bounds(const LloydLayout& L, bool enter, char* area, int parity, const void* X_t, const void* w,
                      const void* centroids_t, const void* before_t, uint32_t* labels_a, uint32_t* labels_b,
                      const LloydTail<TX>& tail, char* ws, int64_t n, int d, int k, hipStream_t stream) {
    const BoundsArea a = bounds_area(n, d, k);
    const unsigned int* absmax = reinterpret_cast<const unsigned int*>(ws + L.off_scales);
    const int* q_exp = reinterpret_cast<const int*>(absmax + (d + 1));
    float* drift = reinterpret_cast<float*>(area + a.off_drift);
    const size_t lds = bounds_lds(d, k, NK, (int)sizeof(TX)).total;
    constexpr int THREADS = 64 * bounds_waves((int)sizeof(TX), NK);
    const int64_t grid = bounds_grid(n, THREADS / 64, kmx_num_cus());
#define KMX_BOUNDS(ENTER_)                                                                                              \
    do {                                                                                                                \
        if (lds > 64 * 1024) {                                                                                          \
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&bounds_kernel<TX, NK, ENTER_>),     \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);             \
            if (e != hipSuccess) return (int32_t)e;                                                                     \
        }                                                                                                               \
        hipLaunchKernelGGL((bounds_kernel<TX, NK, ENTER_>), dim3((unsigned)grid), dim3(THREADS), lds, stream,           \
                           (const TX*)X_t, (float*)(area + a.off_rows), (const TX*)w, (const TX*)centroids_t,              \
                           (const TX*)before_t, labels_a, labels_b, (uint32_t*)(area + a.off_words),                    \
                           drift + (size_t)parity * k, drift + (size_t)(parity ^ 1) * k, tail.status, absmax, q_exp,    \
                           (unsigned long long*)(ws + L.off_gsum), n, d, k, a.ds, tail);               \
    } while (0)
    if (enter) KMX_BOUNDS(true); else KMX_BOUNDS(false);
#undef KMX_BOUNDS
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

template <typename TX>
int32_t iter_bounds(const LloydLayout& L, bool enter, char* area, int parity, const void* X_t, const void* w,
                    const void* centroids_t, void* new_centroids_t, uint32_t* labels_a, uint32_t* labels_b, void* sizes,
                    uint32_t* empty_clusters, char* ws, int64_t n, int d, int k, hipStream_t stream) {
    LloydTail<TX> tail;
    tail.sums_t = (TX*)new_centroids_t;
    tail.sizes = (TX*)sizes;
    tail.empty_clusters = empty_clusters;
    tail.old_centroids_t = (const TX*)centroids_t;
    tail.cpack = reinterpret_cast<TX*>(ws + L.off_cpack);
    tail.half_norms = reinterpret_cast<TX*>(ws + L.off_half);
    tail.status = reinterpret_cast<kmx_lloyd_status*>(ws + L.off_status);
    tail.d = d;
    tail.k = k;
    tail.dpad = L.dpad;
    tail.progress = L.progress;
    tail.clear_word = reinterpret_cast<uint32_t*>(ws + L.off_bucket);  // (the screened steps' counter block)
    tail.looked_word = tail.clear_word + 3;
    tail.n_samples = n;
    tail.delta_divisor = 3;  // (as the screened steps)
    tail.list_divisor = 24;
#define KMX_BOUNDS_NK(NK_)                                                                                              \
    return launch_bounds<TX, NK_>(L, enter, area, parity, X_t, w, centroids_t, new_centroids_t, labels_a, labels_b, tail, \
                                  ws, n, d, k, stream)
    switch ((d + 15) / 16) {
        case 1: KMX_BOUNDS_NK(1);
        case 2: KMX_BOUNDS_NK(2);
        case 3: KMX_BOUNDS_NK(3);
        case 4: KMX_BOUNDS_NK(4);
        default: return KMX_ERR_UNSUPPORTED;
    }
#undef KMX_BOUNDS_NK
}

}  // namespace

bool kmx_bounds_fit(int64_t n, int d, int k, int dtype) {
    const int esize = dtype == KMX_F64 ? 8 : 4, nk = (d + 15) / 16;
    if (d > 64 || k > (int)LABEL_MASK || n >= ((int64_t)1 << 29)) return false;  // (as the screened steps)
    if (!bounds_entries_fit(n, bounds_waves(esize, nk), kmx_num_cus())) return false;
    // (one load of words by every wave must fit the queue)
    return bounds_lds(d, k, nk, esize).q_cap >= UNIT * bounds_waves(esize, nk);
}

size_t kmx_bounds_bytes(int64_t n, int d, int k) { return bounds_area(n, d, k).total; }

// One iteration of a plan whose step is a screened one (L.screen, L.screen64), `enter` over all samples.  Old
// labels are those of `labels_a`, or of the words; the new ones go to both arrays.  `parity`: which copy of the
// drift the iteration reads (it alternates).  `new_centroids_t` holds the centroids of the iteration before.
int32_t kmx_lloyd_iter_bounds(const LloydLayout& L, bool enter, char* area, int parity, const void* X_t, const void* w,
                              const void* centroids_t, void* new_centroids_t, uint32_t* labels_a, uint32_t* labels_b,
                              void* sizes, uint32_t* empty_clusters, char* ws, int64_t n, int d, int k, int dtype,
                              hipStream_t stream) {
    if (dtype == KMX_F32)
        return iter_bounds<float>(L, enter, area, parity, X_t, w, centroids_t, new_centroids_t, labels_a, labels_b, sizes,
                                  empty_clusters, ws, n, d, k, stream);
    return iter_bounds<double>(L, enter, area, parity, X_t, w, centroids_t, new_centroids_t, labels_a, labels_b, sizes,
                               empty_clusters, ws, n, d, k, stream);
}

int32_t kmx_bounds_spread(const void* X_t, const void* centroids_t, const uint32_t* labels, const kmx_lloyd_status* status,
                          const unsigned int* absmax, unsigned long long* out, int64_t n, int d, int k, int dtype, hipStream_t stream) {
    if (dtype == KMX_F32)
        hipLaunchKernelGGL((spread_kernel<float>), dim3(1), dim3(1024), 0, stream, (const float*)X_t, (const float*)centroids_t,
                           labels, status, absmax, out, n, d, k);
    else
        hipLaunchKernelGGL((spread_kernel<double>), dim3(1), dim3(1024), 0, stream, (const double*)X_t,
                           (const double*)centroids_t, labels, status, absmax, out, n, d, k);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}
