// kmeans++ seeding for gfx950, with no host round trip between centres.
//
// State lives in a caller-provided workspace:
//   header      best row of the last step, total potential of that row
//   candidates  2 x 16 int32 (two buffers so that a fused select+sample launch can read the
//               previous candidates while it writes the next ones)
//   potentials  16 doubles (row sums of the last step)
//   block_pot   (16, n_blocks) doubles: per-workgroup partial row sums; workgroup b owns the
//               samples [b * 1024, (b + 1) * 1024), so these are also the coarse level of the
//               sampler's two-level search
//   cand_rows   (16, d): the feature rows of the current candidates, copied when they are
//               sampled so that the step kernel reads them with wave-uniform (scalar) loads
//   rows        (n_trials, n) in the compute dtype: min(w * ||x - x_cand||^2, closest) for
//               every candidate; `closest` IS the best row, updated in place: a thread reads
//               closest[i] before it writes column i of every row.
//
// Per new centre: [select previous best + sample candidates] then [step].  The sampler is a
// search in the fp64 inclusive scan of `closest`: coarse over the block sums, fine inside one
// block of 1024 samples, so it never re-reads the whole array.
#include "lloyd_layout.h"

#include <type_traits>

namespace {

constexpr int TN_MAX = 16;      // n_local_trials = 2 + floor(ln k) <= 16 for k < 1.2e6
constexpr int CHUNK = 1024;     // samples per workgroup (256 threads x 4)
// Screened steps (kpp_screen_step_kernel): from these sizes on.  The copies they read cost about two
// plain steps, and a step still writes all its rows: with few features there is little to save.
// Measured, whole seedings, plain / screened steps: fp32 1e6 x 32, 128 centres 5.3 / 6.1 ms; 3e5 x 64,
// 32 centres 1.35 / 1.22; 1e6 x 64, 256 centres 15.9 / 15.4;
// 4e5 x 255, 100 centres 10.9 / 8.1; fp64 1e6 x 16, 128 centres 5.5 / 7.2; 5e5 x 50, 100 centres 5.0 / 5.0;
// 5e5 x 64, 200 centres 11.5 / 9.4; 3e5 x 128, 64 centres 6.0 / 5.1.
constexpr int64_t SCREEN_MIN_N = 1 << 17;
constexpr int SCREEN_MIN_K = 32, SCREEN_MIN_D = 64;
constexpr int SPLIT_MIN_D = 64; // from this many features on, few samples are stepped with the
                                // features split over the four waves of a workgroup

struct KppHeader {
    int32_t best_row;
    int32_t pad;
    double total;
};

struct KppLayout {
    size_t off_header, off_cand, off_pot, off_cand_rows, off_block_pot, off_rows, off_rows2, total;
    int64_t n_blocks;
    int chunk;  // samples per block sum: CHUNK, or 64 * split
    int split;  // 0, or the samples per thread (1, 2, 4) of the feature-split step kernel
    int joint;  // 0, or the samples per thread (1, 2, 4) of the kernel that selects, samples and steps at once
};

// Samples per thread of the feature-split step kernel, 0 when the shape keeps the plain one.
// With CHUNK samples per workgroup a short, wide array gives the chip a few dozen workgroups
// that each walk every feature; 64 * split samples per workgroup and a quarter of the features
// per wave give it thousands of waves.  The block sums stay at most 1 024, which the selection
// kernel keeps in registers.
int kpp_split(int64_t n, int d, int n_trials, int dtype) {
    if (d < SPLIT_MIN_D) return 0;
    // (the partial distances of a workgroup: 4 waves x trials x samples, at most 32 KB)
    const int most = (dtype == KMX_F32 ? 4 : 2) / (n_trials > 8 ? 2 : 1);
    const int spt = n <= 65536 ? 1 : n <= 131072 ? 2 : n <= 262144 ? 4 : 8;
    return spt <= most ? spt : 0;
}

// Samples per thread of kpp_joint_kernel, 0 when a centre takes two launches: every workgroup repeats the
// selection and the search for the candidates, which pays while there are at most JOINT_BLOCKS block sums
// to look through and the candidates' rows are short.  Beyond one sample per thread a step is the time to
// read X once it has more than JOINT_BYTES, and one workgroup per compute unit does not hide that.  Whole
// seedings, us, two launches a centre / one: fp32 20 000 x 50, 200 centres 5 981 / 3 198; 80 223 x 9, 85 1 766 /
// 1 162; 131 072 x 40 (21 MB), 50 1 068 / 892; 260 000 x 10, 100 2 008 / 1 640; 262 144 x 63 (66 MB), 30 946 / 1 137;
// fp64 1 500 x 20, 8 252 / 212; 65 536 x 63, 100 3 065 / 1 958; 100 000 x 30 (24 MB), 20 516 / 503; 131 072 x 63
// (66 MB), 30 1 010 / 1 061.
// The line is where the first kind of shape loses; some of the others would gain a little beyond it.  50 centres,
// two launches / one: fp32, two samples per thread, 131 072 x 56 (29 MB) 1 203 / 1 013, 63 (33 MB) 1 266 / 1 143; four,
// 262 144 x 32 (34 MB) 1 053 / 1 177, 40 1 281 / 1 333, 48 (50 MB) 1 311 / 1 470; fp64 131 072 x 32 (34 MB) 1 164 / 1 076,
// 48 (50 MB) 1 393 / 1 363; 200 000 x 20 (32 MB) 1 119 / 1 171; 262 144 x 24 (50 MB) 1 309 / 1 245.
constexpr int JOINT_BLOCKS = 256, JOINT_TN = 8, JOINT_D = 64;
constexpr int64_t JOINT_BYTES = 24 << 20;
int kpp_joint(int64_t n, int d, int n_trials, int dtype) {
    if (d >= JOINT_D || n_trials > JOINT_TN || n > 4 * 256 * JOINT_BLOCKS) return 0;
    if (n <= 256 * JOINT_BLOCKS) return 1;
    if (n * d * (int64_t)kmx_dtype_size(dtype) > JOINT_BYTES) return 0;
    return n <= 2 * 256 * JOINT_BLOCKS ? 2 : 4;
}

// The layout, the block sums included, depends on the shape only: calls with either sampler
// may follow one another on one workspace.
KppLayout kpp_layout(int64_t n, int d, int n_trials, int dtype) {
    KppLayout L;
    L.split = kpp_split(n, d, n_trials, dtype);
    L.chunk = L.split ? 64 * L.split : CHUNK;
    L.n_blocks = kmx_cdiv(n, L.chunk);
    L.off_header = 0;
    L.off_cand = 256;
    L.off_pot = 512;
    L.off_cand_rows = 768;  // (TN_MAX, d): the candidates' feature rows, read by the step kernel a batch at a time
    L.off_block_pot = L.off_cand_rows + kmx_align256((size_t)TN_MAX * d * kmx_dtype_size(dtype));
    L.off_rows = L.off_block_pot + kmx_align256((size_t)L.n_blocks * TN_MAX * sizeof(double));
    L.total = L.off_rows + kmx_align256((size_t)n_trials * n * kmx_dtype_size(dtype));
    // (its steps read the rows of the one before while they write their own; two sets of block sums)
    L.joint = kpp_joint(n, d, n_trials, dtype);
    L.off_rows2 = L.total;
    if (L.joint)
        L.total += kmx_align256((size_t)n_trials * n * kmx_dtype_size(dtype)) + 2 * JOINT_TN * JOINT_BLOCKS * sizeof(double);
    return L;
}

// acc + diff^2.  FUSED: one rounding (fused multiply-add), the default.  Not FUSED: product and
// sum rounded separately, the two statements of the reference's kernels taken literally
// (kmeans/kernels/kmeans_plusplus.py:44-48, 226-230); the literal sampler's running sum in the
// compute dtype amplifies a last-bit difference in one distance into another candidate, so
// the literal mode has to reproduce the distances bit for bit as well.
template <bool FUSED, typename T>
__device__ __forceinline__ T kpp_sq_acc(T diff, T acc) {
    if constexpr (FUSED) {
        return fma(diff, diff, acc);
    } else {
#pragma clang fp contract(off)
        const T p = diff * diff;
        return acc + p;
    }
}

// The value lane `src` (a constant) holds, as a wave-uniform scalar.
template <typename T>
__device__ __forceinline__ T kpp_readlane(T v, int src) {
    if constexpr (sizeof(T) == 4) {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
    } else {
        const long long b = __double_as_longlong(v);
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, src);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), src);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
}

// The candidates' values of one batch of FB features, fetched with the samples' own loads:
// lane l of load q asks for feature f0 + l % FB of trial q * (64 / FB) + l / FB (indices
// clamped to the rows in use), and the feature loop reads each value back from its lane as a
// scalar.  One scalar load per value, each waited for where it is used, took a round trip
// per candidate and feature instead.
template <typename T, int TN, int FB>
struct KppCandBatch {
    static constexpr int TPL = 64 / FB;  // trials per load
    static constexpr int NQ = (TN + TPL - 1) / TPL;
    T v[NQ];
    __device__ __forceinline__ void load(const T* __restrict__ cand_rows, int f0, int d, int n_trials, int lane) {
        const int f = f0 + lane % FB < d ? f0 + lane % FB : d - 1;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int t = q * TPL + lane / FB;
            v[q] = cand_rows[(size_t)(t < n_trials ? t : n_trials - 1) * d + f];
        }
    }
    __device__ __forceinline__ T get(int t, int j) const { return kpp_readlane<T>(v[t / TPL], (t % TPL) * FB + j); }
};

// The end of a step for a workgroup's 1 024 samples: `value` yields the new closest distances of four
// samples (4 q .. 4 q + 3, q = thread % 256) for a trial; they go to its row, and their sum over the
// workgroup to the block sums.  HALVES = 2: 512 threads, whose halves take every other trial.
template <typename T, int TN, int HALVES, bool full, typename V>
__device__ __forceinline__ void kpp_finish_block(T* __restrict__ rows, double* __restrict__ block_pot,
                                                 double (*wave_pot)[TN], int64_t i0, int64_t n, int n_trials,
                                                 V&& value) {
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int half = HALVES == 1 ? 0 : (int)(threadIdx.x >> 8);
    double pot[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        pot[t] = 0.0;
        if (t < n_trials && t % HALVES == half) {
            T v[4];
            value(t, v);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (i0 + r < n) pot[t] += (double)v[r];
            kmx_store4<T>(rows + (size_t)t * n, i0, n, full, v);
        }
    }
    // all row sums of the workgroup with one barrier: waves first, then one thread per trial
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        if (t < n_trials && t % HALVES == half) {
            const double ws = kmx_wave_sum<double>(pot[t]);
            if (lane == 0) wave_pot[wave][t] = ws;
        }
    }
    __syncthreads();
    if (threadIdx.x < n_trials)
        block_pot[(size_t)threadIdx.x * gridDim.x + blockIdx.x] =
            (wave_pot[0][threadIdx.x] + wave_pot[1][threadIdx.x]) +
            (wave_pot[2][threadIdx.x] + wave_pot[3][threadIdx.x]);
}

// rows[t, i] = min(w_i * ||x_i - x_cand_t||^2, closest_i) and per-block row sums.
// Candidate rows come from a small (TN, d) buffer, a batch of features at a time spread over
// the lanes and read back as scalars (no LDS, no barriers in the feature loop); every thread
// streams 4 consecutive samples of a batch of features with 128-bit loads.
// INIT: the first distances instead, closest = w * ||x - x_start||^2 into row 0 with its block
// sums, and slot 0 of the outputs: one trial whose candidate is sample `start`, no minimum.
template <typename T, int TN, bool FUSED, bool INIT>
__global__ __launch_bounds__(256) void kpp_step_kernel(
    const T* __restrict__ X_t, const T* __restrict__ sample_weight, const T* __restrict__ cand_rows,
    T* __restrict__ rows, double* __restrict__ block_pot, KppHeader* __restrict__ header,
    int64_t n, int d, int k, int n_trials, int32_t start, T* __restrict__ centers_t,
    int32_t* __restrict__ center_indices) {
    __shared__ double wave_pot[4][TN];
    const int best = INIT ? 0 : header->best_row;
    const int64_t i0 = (int64_t)blockIdx.x * CHUNK + threadIdx.x * 4;
    const int lane = threadIdx.x & 63;
    // Whether every sample of the workgroup exists is decided once and known at compile time inside
    // the body: with a test per access every load sat in a branch of its own and was waited for
    // before the next one was issued.
    auto body = [&](auto full_tag) {
    constexpr bool full = decltype(full_tag)::value;

    // weights and the closest distances so far are needed after the feature loop: requested
    // with its last batch
    T w[4], cl[4];

    T acc[TN][4];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = T(0);

    // Features in batches of FB rows: 16 loads of 16 bytes per lane in flight at a time in fp32
    // (a wave has 64 KB to stream and only four of them share a SIMD).
    constexpr int FB = sizeof(T) == 4 ? 16 : 8;
    for (int f0 = 0; f0 < d; f0 += FB) {
        T xv[FB][4];
#pragma unroll
        for (int j = 0; j < FB; ++j) {
            const int f = f0 + j < d ? f0 + j : d - 1;  // past the end: a valid row, ignored below
            const T* __restrict__ row = X_t + (size_t)f * n;
            kmx_load4<T>(row, i0, n, full, xv[j]);
        }
        KppCandBatch<T, TN, FB> cand;
        if constexpr (INIT) {
            const int f = f0 + lane % FB < d ? f0 + lane % FB : d - 1;
            cand.v[0] = X_t[(size_t)f * n + start];
        } else {
            cand.load(cand_rows, f0, d, n_trials, lane);
        }
        if (f0 + FB >= d) {
            kmx_load4<T>(sample_weight, i0, n, full, w);
            if constexpr (!INIT) kmx_load4<T>(rows + (size_t)best * n, i0, n, full, cl);
        }
        auto accumulate = [&](auto whole_tag) {
            constexpr bool whole = decltype(whole_tag)::value;  // all FB features exist
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if (t < n_trials) {
#pragma unroll
                    for (int j = 0; j < FB; ++j) {
                        if (whole || f0 + j < d) {
                            const T cv = cand.get(t, j);
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const T diff = xv[j][r] - cv;
                                acc[t][r] = kpp_sq_acc<FUSED>(diff, acc[t][r]);
                            }
                        }
                    }
                }
            }
        };
        if (f0 + FB <= d)
            accumulate(std::true_type{});
        else
            accumulate(std::false_type{});
    }

    kpp_finish_block<T, TN, 1, full>(rows, block_pot, wave_pot, i0, n, n_trials, [&](int t, T (&v)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = acc[t][r] * w[r];
            if constexpr (!INIT) v[r] = fmin(v[r], cl[r]);
        }
    });
    };
    if ((int64_t)(blockIdx.x + 1) * CHUNK <= n)
        body(std::true_type{});
    else
        body(std::false_type{});
    if (INIT && blockIdx.x == 0) {
        for (int f = threadIdx.x; f < d; f += 256) centers_t[(size_t)f * k] = X_t[(size_t)f * n + start];
        if (threadIdx.x == 0) {
            center_indices[0] = start;
            header->best_row = 0;
            header->total = 0.0;
        }
    }
}


// ---------------------------------------------------------------- screened step
//
// Most candidates are nearer than the closest centre so far for few samples: one in c + 1 for c
// centres already there, and fewer where the data have clusters.  For the rest the new closest
// distance is the old one, and a lower bound of the candidate's distance shows it: the samples'
// half-precision tiles (lloyd_tiles.hip; a candidate's row is read from them as well) give all of a
// workgroup's distances with matrix instructions at 2 bytes per value,
//     D >= sqrt(|x'|^2 + |c'|^2 - 2 <x', c'> - slack) - |e_x| - |e_c|
// (primes: rounded, e: what rounding took, known per sample; slack: fp32 accumulation).  The pairs
// that it does not settle are gathered and their distances taken from the row-major copy exactly
// as the plain step takes them (features in order, one fused multiply-add each): rows, block sums
// and therefore candidates are those of the plain step, bit for bit.  A workgroup with more than
// SCREEN_QUEUE of its 1 024 x trials pairs unsettled takes all of them from X.
constexpr int SCREEN_TN = 8;         // trials: accumulator registers 0 .. 3 of both halves of a wave
constexpr int SCREEN_FROM = 8;       // centres before the first screened step
constexpr int SCREEN_QUEUE = 1792;
constexpr int SCREEN_PITCH = CHUNK + 16;
constexpr float SCREEN_ULP = 1.1920929e-7f;  // 2^-23

typedef float kpp_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 kpp_v8h __attribute__((ext_vector_type(8)));

template <typename T>
size_t screen_lds(int d, int S) {
    return (size_t)S * 1024 + SCREEN_TN * (SCREEN_PITCH + (size_t)((d + 3) & ~3)) * sizeof(T) +
           SCREEN_QUEUE * sizeof(uint16_t);
}

// Eight waves, four tiles of 32 samples each: a wave's tiles travel as items of four steps of 16
// features, four items in flight from the first instruction on (nothing they need depends on the
// candidates).  Bound by memory and, with one or two rounds of workgroups, by the phases that a
// workgroup goes through one after the other: 49 us at 1e6 x 64 (168 MB) where the plain step
// takes 52 (284 MB at 5.5 TB/s); registers for four waves per SIMD, LDS for two workgroups.
template <typename T>
__global__ __launch_bounds__(512, 4) void kpp_screen_step_kernel(
    const T* __restrict__ X_t, const T* __restrict__ X_rm, KmxTiles tiles, const T* __restrict__ sample_weight,
    const int32_t* __restrict__ cand, const T* __restrict__ cand_rows, T* __restrict__ rows,
    double* __restrict__ block_pot, const KppHeader* __restrict__ header, int64_t n, int d, int n_trials) {
    extern __shared__ __align__(16) unsigned char screen_smem[];
    __shared__ double wave_pot[4][SCREEN_TN];
    __shared__ int queued_s;
    const int S = tiles.S, dp = (d + 3) & ~3;
    uint4* a_s = reinterpret_cast<uint4*>(screen_smem);       // the candidates' fragments, S x 64
    T* v_s = reinterpret_cast<T*>(a_s + S * 64);              // new closest distances, trials x SCREEN_PITCH
    T* cand_s = v_s + SCREEN_TN * SCREEN_PITCH;               // the candidates' rows, trials x dp
    uint16_t* queue = reinterpret_cast<uint16_t*>(cand_s + SCREEN_TN * dp);  // unsettled pairs: trial, sample
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int h = lane >> 5, j = lane & 31;
    const int64_t base = (int64_t)blockIdx.x * CHUNK;

    // the wave's tiles (those past the end, there are none in the copy, repeat the last one)
    const int64_t tile0 = base / 32 + wave * 4, last_tile = (n - 1) / 32;
    const int per_tile = (S + 3) / 4, n_items = 4 * per_tile;
    auto load_item = [&](int item, uint4 (&x)[4]) {
        const int u = item / per_tile, s0 = (item - u * per_tile) * 4;
        const int64_t tile = tile0 + u < last_tile ? tile0 + u : last_tile;
        const uint4* __restrict__ src = tiles.xt + (size_t)tile * S * 64 + lane;
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = src[(s0 + q < S ? s0 + q : S - 1) * 64];
    };
    uint4 x[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) load_item(b, x[b]);  // (n_items >= 4)

    if (threadIdx.x == 0) queued_s = 0;
    // (rows past the last trial repeat it; nothing reads their scores)
    const int64_t cj = cand[j < n_trials ? j : n_trials - 1];
    for (int s = wave; s < S; s += 8)
        a_s[s * 64 + lane] = tiles.xt[((size_t)(cj >> 5) * S + s) * 64 + h * 32 + (cj & 31)];
    for (int e = threadIdx.x; e < n_trials * d; e += 512) cand_s[e / d * dp + e % d] = cand_rows[e];
    const int best = header->best_row;
    float xn[4], xe[4];
    T w[4], cl[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int64_t i = (tile0 + u) * 32 + j, ic = i < n ? i : n - 1;
        xn[u] = tiles.norm[ic];
        xe[u] = tiles.err[ic];
        w[u] = sample_weight[ic];
        cl[u] = rows[(size_t)best * n + ic];
    }
    // norm, root and rounding of this lane's four candidates: trials 4 h .. 4 h + 3
    float cn[4], cr[4], ce[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t c = cand[4 * h + r < n_trials ? 4 * h + r : n_trials - 1];
        cn[r] = tiles.norm[c];
        ce[r] = tiles.err[c];
        cr[r] = sqrtf(cn[r]);
    }
    const T inv_scale = T(1) / (T)tiles.scale[0];
    const float rho = SCREEN_ULP * (17.0f * (float)S + 8.0f);
    const T keep = T(1) - T((d + 32) * 2.0 * SCREEN_ULP);  // the roundings of a distance in T, and of the bound
    const T least = sizeof(T) == 4 ? T(1e-30) : T(1e-290); // below: rounding to zero would count
    __syncthreads();

    kpp_v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    auto settle = [&](int u, float xn_u, float xe_u, T w_u, T cl_u) {
        const int sl = (wave * 4 + u) * 32 + j;
        const bool live = base + sl < n;
        const float xr = sqrtf(xn_u);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 4 * h + r;
            const float both = xn_u + cn[r];
            const float d2 = both - 2.0f * acc[r] - rho * (2.0f * xr * cr[r] + both);
            const float root = sqrtf(fmaxf(d2, 0.0f));  // (a NaN: zero, nothing settled)
            const float lb = root * (1.0f - 8.0f * SCREEN_ULP) - (xe_u + ce[r]) * (1.0f + 8.0f * SCREEN_ULP);
            const T true_lb = (T)lb * inv_scale;
            const T lb2 = true_lb * true_lb;
            const bool settled = lb > 1e-6f && lb2 > least && w_u >= T(0) && w_u * lb2 * keep >= cl_u;
            const bool open = live && t < n_trials && !settled;
            if (live && t < n_trials) v_s[t * SCREEN_PITCH + sl] = cl_u;
            const unsigned long long mask = __ballot(open);
            if (mask != 0) {
                int at = 0;
                if (lane == 0) at = atomicAdd(&queued_s, (int)__popcll(mask));
                at = __builtin_amdgcn_readfirstlane(at);
                at += (int)__popcll(mask & ((1ull << lane) - 1));
                if (open && at < SCREEN_QUEUE) queue[at] = (uint16_t)(t << 10 | sl);
            }
        }
    };
    int u = 0, part = 0;  // tile and part of the current item
    for (int item0 = 0; item0 < n_items; item0 += 4) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int s = part * 4 + q;
                if (s < S)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(kpp_v8h, a_s[s * 64 + lane]),
                                                                 __builtin_bit_cast(kpp_v8h, x[b][q]), acc, 0, 0, 0);
            }
            if (item0 + b + 4 < n_items) load_item(item0 + b + 4, x[b]);
            if (++part == per_tile) {
                settle(u, u == 0 ? xn[0] : u == 1 ? xn[1] : u == 2 ? xn[2] : xn[3],
                       u == 0 ? xe[0] : u == 1 ? xe[1] : u == 2 ? xe[2] : xe[3],
                       u == 0 ? w[0] : u == 1 ? w[1] : u == 2 ? w[2] : w[3],
                       u == 0 ? cl[0] : u == 1 ? cl[1] : u == 2 ? cl[2] : cl[3]);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
                part = 0;
                ++u;
            }
        }
    }
    __syncthreads();
    const int queued = queued_s;
    if (queued > SCREEN_QUEUE) {
        // (the same for the whole workgroup) every pair, two samples per thread from X itself
        const int sl = threadIdx.x * 2;
        const bool pair = base + CHUNK <= n;
        T dist[SCREEN_TN][2];
#pragma unroll
        for (int t = 0; t < SCREEN_TN; ++t) dist[t][0] = dist[t][1] = T(0);
        constexpr int FB = 8;
        for (int f0 = 0; f0 < d; f0 += FB) {
            T xv[FB][2];
#pragma unroll
            for (int q = 0; q < FB; ++q) {
                const T* __restrict__ row = X_t + (size_t)(f0 + q < d ? f0 + q : d - 1) * n;
                if (pair) {
                    using V2 = typename KmxVec<T, 2>::type;
                    const V2 v = *reinterpret_cast<const V2*>(row + base + sl);
                    xv[q][0] = v[0]; xv[q][1] = v[1];
                } else {
#pragma unroll
                    for (int r = 0; r < 2; ++r) xv[q][r] = row[base + sl + r < n ? base + sl + r : n - 1];
                }
            }
#pragma unroll
            for (int q = 0; q < FB; ++q) {
                if (f0 + q < d) {
#pragma unroll
                    for (int t = 0; t < SCREEN_TN; ++t) {
                        const T cv = cand_s[t * dp + f0 + q];  // (past n_trials: not used)
#pragma unroll
                        for (int r = 0; r < 2; ++r) dist[t][r] = kpp_sq_acc<true>(xv[q][r] - cv, dist[t][r]);
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (base + sl + r < n) {
                const T wv = sample_weight[base + sl + r];
                for (int t = 0; t < n_trials; ++t) {
                    T* at = v_s + t * SCREEN_PITCH + sl + r;
                    T dt = dist[0][r];
#pragma unroll
                    for (int q = 1; q < SCREEN_TN; ++q) dt = t == q ? dist[q][r] : dt;
                    *at = fmin(dt * wv, *at);
                }
            }
        }
    } else {
        for (int e = threadIdx.x; e < queued; e += 512) {
            const int t = queue[e] >> 10, sl = queue[e] & (CHUNK - 1);
            const T* __restrict__ row = X_rm + (size_t)(base + sl) * d;
            const T* __restrict__ c = cand_s + t * dp;
            T dist = T(0);
            const int whole = d & ~3;
#pragma unroll 8
            for (int f = 0; f < whole; f += 4) {
                T v[4];
                kmx_load4<T>(row, f, d, true, v);
#pragma unroll
                for (int q = 0; q < 4; ++q) dist = kpp_sq_acc<true>(v[q] - c[f + q], dist);
            }
            for (int f = whole; f < d; ++f) dist = kpp_sq_acc<true>(row[f] - c[f], dist);
            T* at = v_s + t * SCREEN_PITCH + sl;
            *at = fmin(dist * sample_weight[base + sl], *at);
        }
    }
    __syncthreads();
    const int q4 = (threadIdx.x & 255) * 4;
    auto finish = [&](auto full_tag) {
        kpp_finish_block<T, SCREEN_TN, 2, decltype(full_tag)::value>(
            rows, block_pot, wave_pot, base + q4, n, n_trials, [&](int t, T (&v)[4]) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = v_s[t * SCREEN_PITCH + q4 + r];
            });
    };
    if (base + CHUNK <= n)
        finish(std::true_type{});
    else
        finish(std::false_type{});
}

// SPT consecutive values of a row at i0: one access of SPT elements when `full`, else element
// by element from indices clamped to the array (the caller ignores what lies past n).
template <typename T, int SPT>
__device__ __forceinline__ void load_spt(const T* __restrict__ row, int64_t i0, int64_t n, bool full, T (&v)[SPT]) {
    if (full) {
        if constexpr (SPT == 1) {
            v[0] = row[i0];
        } else if constexpr (SPT == 2) {
            using V2 = typename KmxVec<T, 2>::type;
            const V2 q = *reinterpret_cast<const V2*>(row + i0);
            v[0] = q[0]; v[1] = q[1];
        } else {
            kmx_load4<T>(row, i0, n, true, v);
        }
    } else {
#pragma unroll
        for (int r = 0; r < SPT; ++r) v[r] = row[i0 + r < n ? i0 + r : n - 1];
    }
}

// The step (or, INIT, the first distances to the starting sample) for few samples of many
// features.  A workgroup owns 64 * SPT samples; its four waves take the feature batches in
// turn, every lane streaming SPT consecutive samples, and leave partial squared distances in
// LDS.  After one barrier wave w finishes trials w, w + 4: the four partial sums added in wave
// order, weight, minimum with the closest distance so far, the row store and the block sum.
// The closest distances are read before the barrier: the finishing waves overwrite the row
// they came from.  LITERAL keeps the reference's roundings (features summed in order, product
// and sum rounded separately): every wave walks all the features and the first one's sums are
// used, so that the block sums have one geometry for both samplers.
template <typename T, int TN, int SPT, bool INIT, bool LITERAL>
__global__ __launch_bounds__(256) void kpp_step_split_kernel(
    const T* __restrict__ X_t, const T* __restrict__ sample_weight, const T* __restrict__ cand_rows,
    T* __restrict__ rows, double* __restrict__ block_pot, KppHeader* __restrict__ header, int64_t n,
    int d, int k, int n_trials, int32_t start, T* __restrict__ centers_t,
    int32_t* __restrict__ center_indices) {
    constexpr int S = 64 * SPT;
    __shared__ T part[4][TN][S];
    // the wave index as a scalar: the feature loop's bounds and the candidates' rows are then
    // wave-uniform for the compiler as well (scalar branches, no lane masks per feature)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t base = (int64_t)blockIdx.x * S;
    const int64_t i0 = base + lane * SPT;
    const int best = INIT ? 0 : header->best_row;

    // what the finish needs of samples base + r * 64 + lane, requested ahead of the feature loop
    T w_fin[SPT], cl_fin[SPT];
#pragma unroll
    for (int r = 0; r < SPT; ++r) {
        const int64_t i = base + r * 64 + lane;
        const int64_t ic = i < n ? i : n - 1;
        w_fin[r] = sample_weight[ic];
        cl_fin[r] = INIT ? T(0) : rows[(size_t)best * n + ic];
    }

    auto body = [&](auto full_tag) {
        constexpr bool full = decltype(full_tag)::value;
        T acc[TN][SPT];
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int r = 0; r < SPT; ++r) acc[t][r] = T(0);
        constexpr int FB = sizeof(T) == 4 ? 16 : 8;
        for (int f0 = LITERAL ? 0 : wave * FB; f0 < d; f0 += LITERAL ? FB : 4 * FB) {
            T xv[FB][SPT];
#pragma unroll
            for (int j = 0; j < FB; ++j) {
                const int f = f0 + j < d ? f0 + j : d - 1;  // past the end: a valid row, ignored below
                load_spt<T, SPT>(X_t + (size_t)f * n, i0, n, full, xv[j]);
            }
            // the candidates' rows, or the starting sample's features
            KppCandBatch<T, TN, FB> cand;
            if constexpr (INIT) {
                const int f = f0 + lane % FB < d ? f0 + lane % FB : d - 1;
                cand.v[0] = X_t[(size_t)f * n + start];
            } else {
                cand.load(cand_rows, f0, d, n_trials, lane);
            }
            auto accumulate = [&](auto whole_tag) {
                constexpr bool whole = decltype(whole_tag)::value;  // all FB features exist
#pragma unroll
                for (int t = 0; t < TN; ++t) {
                    if (t < n_trials) {
#pragma unroll
                        for (int j = 0; j < FB; ++j) {
                            if (whole || f0 + j < d) {
                                const T cv = cand.get(t, j);
#pragma unroll
                                for (int r = 0; r < SPT; ++r) {
                                    const T diff = xv[j][r] - cv;
                                    acc[t][r] = kpp_sq_acc<!LITERAL>(diff, acc[t][r]);
                                }
                            }
                        }
                    }
                }
            };
            if (f0 + FB <= d)
                accumulate(std::true_type{});
            else
                accumulate(std::false_type{});
        }
#pragma unroll
        for (int t = 0; t < TN; ++t)
            if (t < n_trials)
#pragma unroll
                for (int r = 0; r < SPT; ++r) part[wave][t][lane * SPT + r] = acc[t][r];
    };
    if (base + S <= n)
        body(std::true_type{});
    else
        body(std::false_type{});
    __syncthreads();

    for (int t = wave; t < n_trials; t += 4) {
        double pot = 0.0;
#pragma unroll
        for (int r = 0; r < SPT; ++r) {
            const int sl = r * 64 + lane;
            const int64_t i = base + sl;
            if (i < n) {
                const T dist = LITERAL ? part[0][t][sl]
                                       : ((part[0][t][sl] + part[1][t][sl]) + part[2][t][sl]) + part[3][t][sl];
                T v = dist * w_fin[r];
                if (!INIT) v = fmin(v, cl_fin[r]);
                rows[(size_t)t * n + i] = v;
                pot += (double)v;
            }
        }
        const double ws = kmx_wave_sum<double>(pot);
        if (lane == 0) block_pot[(size_t)t * gridDim.x + blockIdx.x] = ws;
    }
    if (INIT && blockIdx.x == 0) {
        for (int f = threadIdx.x; f < d; f += 256) centers_t[(size_t)f * k] = X_t[(size_t)f * n + start];
        if (threadIdx.x == 0) {
            center_indices[0] = start;
            header->best_row = 0;
            header->total = 0.0;
        }
    }
}

// Block-wide exclusive scan of one double per thread (256 threads); returns the exclusive
// prefix of the calling thread and the block total.
__device__ __forceinline__ double block_exclusive_scan(double v, double* wave_tot, double& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    __syncthreads();
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    double base = 0.0;
    for (int w2 = 0; w2 < wave; ++w2) base += wave_tot[w2];
    total = wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
    return base + incl - v;
}

__device__ __forceinline__ int64_t block_min_i64(int64_t v, int64_t* scratch) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int64_t o = __shfl_xor(v, off, 64);
        v = o < v ? o : v;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    int64_t m = scratch[0];
    for (int w2 = 1; w2 < 4; ++w2) m = scratch[w2] < m ? scratch[w2] : m;
    return m;
}

// One workgroup per trial, plus one that records the selection.
//   do_select: sum the block potentials of every row of the last step, pick the best row
//              (lowest index on ties); the last workgroup records potentials, header and the
//              centre slot and does not sample.
//   do_sample: candidate t = first j with scan(closest)_j >= uniforms[t] * total, and the
//              candidate's feature row for the step kernel.
//   merge:     0, or how many of these block sums make one of `merged`, which the last workgroup then writes
//              row by row (the end of a run with one launch per centre: the sums that calls step by step read).
// Thread i owns the block sums [i * P, (i + 1) * P); with P <= KPP_OWN they are read once and
// stay in registers for the row totals, the coarse scan and the search.
// Bound by the latency of its chain of loads.  The block sums lie row by row, so that neighbouring
// threads read neighbouring words: with the rows of a block together every lane of a load met a
// cache line of its own (a million samples, 7 trials: 12.7 -> 9.5 us).
// (KPP_OWN = 4 covers a million samples; 8, for up to 8 trials, two million)
template <typename T, int TN, int KPP_OWN = 4>
__global__ __launch_bounds__(256) void kpp_select_sample_kernel(
    const T* __restrict__ X_t, const double* __restrict__ uniforms,
    const int32_t* __restrict__ cand_prev, int32_t* __restrict__ cand_next,
    int32_t* __restrict__ cand_out, T* __restrict__ centers_t,
    int32_t* __restrict__ center_indices, const T* __restrict__ rows,
    const double* __restrict__ block_pot, double* __restrict__ potentials,
    KppHeader* __restrict__ header, T* __restrict__ cand_rows, int64_t n, int64_t n_blocks, int chunk,
    int d, int k, int n_trials, int center_slot, int do_select, int do_sample, double* __restrict__ merged, int merge) {
    __shared__ double wave_tot[4];
    __shared__ double wave_pot[4][TN];
    __shared__ int64_t iscratch[4];
    __shared__ double prefix_s;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;

    const int64_t per_thread = (n_blocks + 255) / 256;
    const bool cached = per_thread <= KPP_OWN;
    const int64_t b0 = (int64_t)threadIdx.x * per_thread;
    int64_t b1 = b0 + per_thread;
    if (b1 > n_blocks) b1 = n_blocks;

    int best;
    double own_best[KPP_OWN];  // the owned block sums of the best row (cached mode)
#pragma unroll
    for (int i = 0; i < KPP_OWN; ++i) own_best[i] = 0.0;

    if (do_select) {
        double acc[TN];
        double own[KPP_OWN][TN];
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[t] = 0.0;
        if (cached) {
#pragma unroll
            for (int i = 0; i < KPP_OWN; ++i) {
                const int64_t b = b0 + i;
                const double* __restrict__ colp = block_pot + (b < n_blocks ? b : 0);
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    own[i][t] = (b < b1 && t < n_trials) ? colp[(size_t)t * n_blocks] : 0.0;
            }
#pragma unroll
            for (int i = 0; i < KPP_OWN; ++i)
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[t] += own[i][t];
        } else {
            for (int64_t b = b0; b < b1; ++b) {
                const double* __restrict__ colp = block_pot + b;
#pragma unroll
                for (int t = 0; t < TN; ++t)
                    if (t < n_trials) acc[t] += colp[(size_t)t * n_blocks];
            }
        }
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            if (t < n_trials) {
                const double ws = kmx_wave_sum<double>(acc[t]);
                if (lane == 0) wave_pot[wave][t] = ws;
            }
        }
        __syncthreads();
        // do_select == 2: the potentials are compared after rounding to T, as the reference's
        // argmin over its T-typed row sums does (kmeans/drivers.py:895-901)
        const bool in_T = do_select == 2;
        double best_pot = (wave_pot[0][0] + wave_pot[1][0]) + (wave_pot[2][0] + wave_pot[3][0]);
        if (in_T) best_pot = (double)(T)best_pot;
        best = 0;
        for (int t = 1; t < n_trials; ++t) {
            double pt = (wave_pot[0][t] + wave_pot[1][t]) + (wave_pot[2][t] + wave_pot[3][t]);
            if (in_T) pt = (double)(T)pt;
            if (pt < best_pot) {
                best_pot = pt;
                best = t;
            }
        }
        if (cached) {
#pragma unroll
            for (int i = 0; i < KPP_OWN; ++i)
#pragma unroll
                for (int t = 0; t < TN; ++t) own_best[i] = (t == best) ? own[i][t] : own_best[i];
        }
        if (blockIdx.x == gridDim.x - 1) {
            const int32_t chosen = cand_prev[best];
            for (int f = threadIdx.x; f < d; f += 256)
                centers_t[(size_t)f * k + center_slot] = X_t[(size_t)f * n + chosen];
            if (threadIdx.x < n_trials)
                potentials[threadIdx.x] = (wave_pot[0][threadIdx.x] + wave_pot[1][threadIdx.x]) +
                                          (wave_pot[2][threadIdx.x] + wave_pot[3][threadIdx.x]);
            if (threadIdx.x == 0) {
                center_indices[center_slot] = chosen;
                header->best_row = best;
                header->total = best_pot;
            }
            if (merge > 0) {
                const int n_merged = (int)((n_blocks + merge - 1) / merge);
                for (int i = threadIdx.x; i < n_trials * n_merged; i += 256) {
                    const int t = i / n_merged, first = (i - t * n_merged) * merge;
                    double sum = 0.0;
                    for (int b = first; b < first + merge && b < n_blocks; ++b) sum += block_pot[(size_t)t * n_blocks + b];
                    merged[i] = sum;
                }
            }
            return;
        }
    } else {
        best = header->best_row;
        if (cached) {
#pragma unroll
            for (int i = 0; i < KPP_OWN; ++i)
                if (b0 + i < b1) own_best[i] = block_pot[(size_t)best * n_blocks + b0 + i];
        }
    }
    if (!do_sample) return;

    const int trial = blockIdx.x;
    // ---- coarse level: exclusive scan of the block sums of the best row
    double local = 0.0;
    if (cached) {
#pragma unroll
        for (int i = 0; i < KPP_OWN; ++i) local += own_best[i];
    } else {
        for (int64_t b = b0; b < b1; ++b) local += block_pot[(size_t)best * n_blocks + b];
    }
    double total;
    const double excl = block_exclusive_scan(local, wave_tot, total);
    const double rv = uniforms[trial] * total;
    int64_t found = INT64_MAX;
    double cum = excl, found_prefix = 0.0;
    if (cached) {
#pragma unroll
        for (int i = 0; i < KPP_OWN; ++i) {
            const double before = cum;
            cum += own_best[i];
            if (found == INT64_MAX && b0 + i < b1 && cum >= rv) {
                found = b0 + i;
                found_prefix = before;
            }
        }
    } else {
        for (int64_t b = b0; b < b1; ++b) {
            const double before = cum;
            cum += block_pot[(size_t)best * n_blocks + b];
            if (cum >= rv) {
                found = b;
                found_prefix = before;
                break;
            }
        }
    }
    const int64_t bstar_raw = block_min_i64(found, iscratch);
    const int64_t bstar = bstar_raw == INT64_MAX ? n_blocks - 1 : bstar_raw;
    if (found == bstar_raw && found != INT64_MAX) prefix_s = found_prefix;
    if (bstar_raw == INT64_MAX && threadIdx.x == 0) prefix_s = total;  // rounding: rv above every cum
    __syncthreads();
    const double prefix = prefix_s;

    // ---- fine level: scan the samples of block bstar (chunk: a multiple of 4, at most 1024)
    const T* __restrict__ closest = rows + (size_t)best * n;
    const int64_t j0 = bstar * chunk + threadIdx.x * 4;
    const bool in_block = (int)threadIdx.x * 4 < chunk;
    double v[4], s = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[r] = (in_block && j0 + r < n) ? (double)closest[j0 + r] : 0.0;
        s += v[r];
    }
    double tot2;
    double c2 = prefix + block_exclusive_scan(s, wave_tot, tot2);
    int64_t hit = INT64_MAX;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        c2 += v[r];
        if (hit == INT64_MAX && in_block && j0 + r < n && c2 >= rv) hit = j0 + r;
    }
    int64_t cand = block_min_i64(hit, iscratch);
    if (cand == INT64_MAX) {
        cand = (bstar + 1) * chunk;  // rounding pushed the crossing just past this block
    }
    if (cand > n - 1) cand = n - 1;
    if (threadIdx.x == 0) {
        cand_next[trial] = (int32_t)cand;
        if (cand_out) cand_out[trial] = (int32_t)cand;
    }
    // the candidate's feature row, for the step kernel
    for (int f = threadIdx.x; f < d; f += 256) cand_rows[(size_t)trial * d + f] = X_t[(size_t)f * n + cand];
}

// ---------------------------------------------------------------- one launch per centre
//
// Few samples: the two launches of a centre are chains of trips to memory on an idle chip, 8 us for the
// selection and 12 for the step at 80 000 x 9.  Here every workgroup finds the winner of the last step and
// this step's candidates by itself - the block sums (one per thread), the waves' share of the candidates'
// blocks, their rows - while its own samples are on their way, and then steps.  What a workgroup looks up, all
// others look up too, from L2.  The rows read are those of the step before, the rows written another set: no
// workgroup waits for another.  Distances and roundings are those of the plain step; sums of sums are taken in
// another order, in fp64.
// INIT: the first distances, closest = w * ||x - x_start||^2, into row 0.

// Sums over the wave of eight values at once: lane l returns the total of value l >> 3 (in its bits 5, 4, 3).
__device__ __forceinline__ double wave_sum_of_eight(const double (&v)[8], int lane) {
    double a[4], b[2], c;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = (lane & 32 ? v[i + 4] : v[i]) + __shfl_xor(lane & 32 ? v[i] : v[i + 4], 32, 64);
#pragma unroll
    for (int i = 0; i < 2; ++i) b[i] = (lane & 16 ? a[i + 2] : a[i]) + __shfl_xor(lane & 16 ? a[i] : a[i + 2], 16, 64);
    c = (lane & 8 ? b[1] : b[0]) + __shfl_xor(lane & 8 ? b[0] : b[1], 8, 64);
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    return c;
}

__device__ __forceinline__ double wave_inclusive_scan(double v, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(v, off, 64);
        if (lane >= off) v += o;
    }
    return v;
}

template <typename T, int SPT, bool INIT>
__global__ __launch_bounds__(256) void kpp_joint_kernel(
    const T* __restrict__ X_t, const T* __restrict__ sample_weight, const double* __restrict__ uniforms,
    const int32_t* __restrict__ cand_prev, int32_t* __restrict__ cand_next, const T* __restrict__ rows_in,
    T* __restrict__ rows_out, const double* __restrict__ pot_in, double* __restrict__ pot_out,
    T* __restrict__ centers_t, int32_t* __restrict__ center_indices, double* __restrict__ potentials,
    KppHeader* __restrict__ header, int64_t n, int d, int k, int n_trials, int center_slot, int32_t start) {
    constexpr int TN = INIT ? 1 : JOINT_TN, CH = 256 * SPT;
    constexpr int FB = 16 / SPT < 8 ? 8 : 16 / SPT;  // features of a batch
    constexpr int V = 16 / (int)sizeof(T);
    __shared__ double wave_pot[4][8], wave_tot[4], excl_s[256];
    __shared__ int first_s[4][JOINT_TN], cand_s[JOINT_TN];
    __shared__ __align__(16) T row_s[TN][JOINT_D];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n_blocks = (int)gridDim.x;
    const int64_t base = (int64_t)blockIdx.x * CH, i0 = base + threadIdx.x * SPT;
    const bool full = base + CH <= n;  // (the same for the whole workgroup)

    auto load_own = [&](const T* __restrict__ row, T(&v)[SPT]) __attribute__((always_inline)) {
        if (SPT > 1 && full) {
            if constexpr (SPT == 4) {
                kmx_load4<T>(row, i0, n, true, v);
            } else if constexpr (SPT == 2) {
                const auto q = *reinterpret_cast<const typename KmxVec<T, 2>::type*>(row + i0);
                v[0] = q[0]; v[1] = q[1];
            }
        } else {
#pragma unroll
            for (int r = 0; r < SPT; ++r) v[r] = row[i0 + r < n ? i0 + r : n - 1];
        }
    };
    T xv[FB][SPT], w[SPT], cl[SPT];
    auto load_batch = [&](const int f0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < FB; ++j) load_own(X_t + (size_t)(f0 + j < d ? f0 + j : d - 1) * n, xv[j]);
    };
    load_batch(0);
    load_own(sample_weight, w);

    if constexpr (INIT) {
        if ((int)threadIdx.x < d) row_s[0][threadIdx.x] = X_t[(size_t)threadIdx.x * n + start];
        __syncthreads();
    } else {
        // ---- the winner of the last step (slot 0: the starting sample is in row 0)
        const int b = threadIdx.x, n_rows = center_slot > 0 ? n_trials : 1;
        double own[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const double v = pot_in[(size_t)(t < n_rows ? t : 0) * n_blocks + (b < n_blocks ? b : 0)];
            own[t] = b < n_blocks && t < n_rows ? v : 0.0;
        }
        const double part = wave_sum_of_eight(own, lane);
        if ((lane & 7) == 0) wave_pot[wave][lane >> 3] = part;
        __syncthreads();
        int best = 0;
        double best_pot = (wave_pot[0][0] + wave_pot[1][0]) + (wave_pot[2][0] + wave_pot[3][0]);
        for (int t = 1; t < n_rows; ++t) {
            const double pt = (wave_pot[0][t] + wave_pot[1][t]) + (wave_pot[2][t] + wave_pot[3][t]);
            if (pt < best_pot) {
                best_pot = pt;
                best = t;
            }
        }
        best = __builtin_amdgcn_readfirstlane(best);
        const T* __restrict__ closest = rows_in + (size_t)best * n;
        load_own(closest, cl);
        if (blockIdx.x == 0 && center_slot > 0) {
            const int32_t chosen = cand_prev[best];
            if ((int)threadIdx.x < d) centers_t[(size_t)threadIdx.x * k + center_slot] = X_t[(size_t)threadIdx.x * n + chosen];
            if ((int)threadIdx.x < n_trials)
                potentials[threadIdx.x] = (wave_pot[0][threadIdx.x] + wave_pot[1][threadIdx.x]) +
                                          (wave_pot[2][threadIdx.x] + wave_pot[3][threadIdx.x]);
            if (threadIdx.x == 0) {
                center_indices[center_slot] = chosen;
                header->best_row = best;
                header->total = best_pot;
            }
        }
        // ---- the block of every candidate: the first whose inclusive sum reaches u * total
        double mine = own[0];
#pragma unroll
        for (int t = 1; t < 8; ++t) mine = t == best ? own[t] : mine;
        const double incl = wave_inclusive_scan(mine, lane);
        if (lane == 63) wave_tot[wave] = incl;
        __syncthreads();
        double before = 0.0, total = 0.0;
#pragma unroll
        for (int w2 = 0; w2 < 4; ++w2) {
            if (w2 == wave) before = total;
            total += wave_tot[w2];
        }
        const double excl = before + incl - mine, cum = excl + mine;
        excl_s[threadIdx.x] = excl;
#pragma unroll
        for (int t = 0; t < JOINT_TN; ++t) {
            const double rv = uniforms[t < n_trials ? t : 0] * total;
            const unsigned long long at = __ballot(b < n_blocks && cum >= rv);
            if (lane == 0) first_s[wave][t] = at != 0ull ? 64 * wave + __builtin_ctzll(at) : n_blocks;
        }
        __syncthreads();
        // ---- the sample in that block, trials wave and wave + 4
        constexpr int PER = CH / 64;  // values per lane
        T fv[2][PER];
        int block[2];
        double prefix[2], rv[2];
        int64_t j0[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int t = wave + 4 * q < n_trials ? wave + 4 * q : 0;
            const int at = min(min(first_s[0][t], first_s[1][t]), min(first_s[2][t], first_s[3][t]));
            // (rounding: u * total above every inclusive sum)
            block[q] = at < n_blocks ? at : n_blocks - 1;
            prefix[q] = at < n_blocks ? excl_s[block[q]] : total;
            rv[q] = uniforms[t] * total;
            j0[q] = (int64_t)block[q] * CH + lane * PER;
            if ((int64_t)(block[q] + 1) * CH <= n) {
#pragma unroll
                for (int r = 0; r < PER; r += 4) {
                    T four[4];
                    kmx_load4<T>(closest, j0[q] + r, n, true, four);
#pragma unroll
                    for (int e = 0; e < 4; ++e) fv[q][r + e] = four[e];
                }
            } else {
#pragma unroll
                for (int r = 0; r < PER; ++r) fv[q][r] = j0[q] + r < n ? closest[j0[q] + r] : T(0);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < PER; ++r) s += (double)fv[q][r];
            double c2 = prefix[q] + (wave_inclusive_scan(s, lane) - s);
            int hit = -1;
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                c2 += (double)fv[q][r];
                if (hit < 0 && j0[q] + r < n && c2 >= rv[q]) hit = (int)j0[q] + r;
            }
            const unsigned long long at = __ballot(hit >= 0);
            // (rounding pushed the crossing just past the block)
            int64_t cand = (int64_t)(block[q] + 1) * CH;
            if (at != 0ull) cand = __builtin_amdgcn_readlane(hit, __builtin_ctzll(at));
            if (cand > n - 1) cand = n - 1;
            if (lane == 0) cand_s[wave + 4 * q] = (int)cand;
        }
        __syncthreads();
        {
            const int t = threadIdx.x >> 5, f = threadIdx.x & 31, c = cand_s[t];  // (past n_trials: trial 0's block, not used)
            const T v0 = X_t[(size_t)(f < d ? f : d - 1) * n + c], v1 = X_t[(size_t)(f + 32 < d ? f + 32 : d - 1) * n + c];
            row_s[t][f] = v0;
            row_s[t][f + 32] = v1;
            if (blockIdx.x == 0 && f == 0 && t < n_trials) cand_next[t] = c;
        }
        __syncthreads();
    }

    // ---- the step: features in order, as in kpp_step_kernel
    T acc[TN][SPT];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int r = 0; r < SPT; ++r) acc[t][r] = T(0);
    for (int f0 = 0; f0 < d; f0 += FB) {
        auto accumulate = [&](auto whole_tag) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                if (t < n_trials) {
#pragma unroll
                    for (int j = 0; j < FB; j += V) {
                        struct alignas(16) Piece { T e[V]; };
                        const Piece cv = *reinterpret_cast<const Piece*>(&row_s[t][f0 + j]);  // (a broadcast)
#pragma unroll
                        for (int e = 0; e < V; ++e)
                            if (decltype(whole_tag)::value || f0 + j + e < d) {
#pragma unroll
                                for (int r = 0; r < SPT; ++r) {
                                    const T diff = xv[j + e][r] - cv.e[e];
                                    acc[t][r] = kpp_sq_acc<true>(diff, acc[t][r]);
                                }
                            }
                    }
                }
            }
        };
        if (f0 + FB <= d) accumulate(std::true_type{});
        else accumulate(std::false_type{});
        if (f0 + FB < d) load_batch(f0 + FB);
    }
    double pot[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        pot[t] = 0.0;
        if (t < TN && t < n_trials) {
            T v[SPT];
#pragma unroll
            for (int r = 0; r < SPT; ++r) {
                v[r] = acc[t < TN ? t : 0][r] * w[r];
                if constexpr (!INIT) v[r] = fmin(v[r], cl[r]);
                if (full || i0 + r < n) pot[t] += (double)v[r];
            }
            T* __restrict__ to = rows_out + (size_t)t * n;
            if constexpr (SPT == 4) {
                kmx_store4<T>(to, i0, n, full, v);
            } else {
#pragma unroll
                for (int r = 0; r < SPT; ++r)
                    if (full || i0 + r < n) to[i0 + r] = v[r];
            }
        }
    }
    const double part = wave_sum_of_eight(pot, lane);
    __syncthreads();  // (wave_pot has been read)
    if ((lane & 7) == 0) wave_pot[wave][lane >> 3] = part;
    __syncthreads();
    if ((int)threadIdx.x < n_trials)
        pot_out[(size_t)threadIdx.x * n_blocks + blockIdx.x] = (wave_pot[0][threadIdx.x] + wave_pot[1][threadIdx.x]) +
                                                               (wave_pot[2][threadIdx.x] + wave_pot[3][threadIdx.x]);
    if (INIT && blockIdx.x == 0) {
        if ((int)threadIdx.x < d) centers_t[(size_t)threadIdx.x * k] = row_s[0][threadIdx.x];
        if (threadIdx.x == 0) {
            center_indices[0] = start;
            header->best_row = 0;
            header->total = 0.0;
        }
    }
}

// The reference's sampler taken literally (kmeans/kernels/kmeans_plusplus.py:79-100): a
// running sum of `closest` in T, element by element from sample 0, and per trial the first j
// whose running sum reaches rv_t = T(u_t) * T(total), clipped to n - 1.  A floating-point
// running sum cannot be split over threads without changing its roundings, so one wave walks the
// array once for all trials (sorted by rv: the sum of non-negative terms never decreases, so
// the trials are met in that order) while the workgroup's 256 threads keep the next 1 024
// values on their way into LDS.  A trial with rv <= 0 leaves the reference's loop at once with
// candidate -1, which its next kernel uses as an index from the end: sample n - 1.
// About 8 ns per sample (8 ms per centre on 10^6 samples): a parity mode, not the default.
template <typename T>
__global__ __launch_bounds__(256) void kpp_sample_literal_kernel(
    const T* __restrict__ X_t, const double* __restrict__ uniforms, int32_t* __restrict__ cand_next,
    int32_t* __restrict__ cand_out, const T* __restrict__ rows, const double* __restrict__ block_pot,
    const KppHeader* __restrict__ header, T* __restrict__ cand_rows, int64_t n, int64_t n_blocks, int d,
    int n_trials) {
    __shared__ T buf[2][CHUNK];
    __shared__ double wave_tot[4];
    __shared__ T rv_sorted[TN_MAX + 1];
    __shared__ int trial_sorted[TN_MAX];
    __shared__ int cand_s[TN_MAX];
    __shared__ int done_s;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int best = header->best_row;
    const T* __restrict__ closest = rows + (size_t)best * n;

    // total potential: the block sums of the best row in fp64, rounded to T once
    double local = 0.0;
    for (int64_t b = threadIdx.x; b < n_blocks; b += 256) local += block_pot[(size_t)best * n_blocks + b];
    const double ws = kmx_wave_sum<double>(local);
    if (lane == 0) wave_tot[wave] = ws;
    __syncthreads();
    const T total = (T)((wave_tot[0] + wave_tot[1]) + (wave_tot[2] + wave_tot[3]));

    if (threadIdx.x == 0) {
        // insertion sort of the trials by rv; rv <= 0 (or NaN) first
        int m = 0;
        for (int t = 0; t < n_trials; ++t) {
            const T rv = (T)uniforms[t] * total;
            const bool low = !(rv > T(0));
            int pos = m;
            while (pos > 0) {
                const T prev = rv_sorted[pos - 1];
                const bool prev_low = !(prev > T(0));
                if (prev_low || (!low && !(rv < prev))) break;
                rv_sorted[pos] = prev;
                trial_sorted[pos] = trial_sorted[pos - 1];
                --pos;
            }
            rv_sorted[pos] = rv;
            trial_sorted[pos] = t;
            ++m;
        }
        rv_sorted[n_trials] = T(0);
        done_s = 0;
    }
    const int64_t n_chunks = (n + CHUNK - 1) / CHUNK;  // the walk's own chunks, not the block sums
    // first chunk
    {
        const int64_t j0 = (int64_t)threadIdx.x * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) buf[0][threadIdx.x * 4 + r] = (j0 + r < n) ? closest[j0 + r] : T(0);
    }
    __syncthreads();

    int cur = 0;
    T cum = T(0);
    if (wave == 0) {
        // trials that never enter the loop
        while (cur < n_trials && !(rv_sorted[cur] > T(0))) {
            if (lane == 0) cand_s[trial_sorted[cur]] = (int)(n - 1);
            ++cur;
        }
    }
    for (int64_t c = 0; c < n_chunks; ++c) {
        T nxt[4] = {T(0), T(0), T(0), T(0)};
        if (c + 1 < n_chunks) {
            const int64_t j0 = (c + 1) * CHUNK + (int64_t)threadIdx.x * 4;
#pragma unroll
            for (int r = 0; r < 4; ++r) nxt[r] = (j0 + r < n) ? closest[j0 + r] : T(0);
        }
        if (wave == 0) {
            const T* __restrict__ b = buf[c & 1];
            const int64_t base = c * CHUNK;
            const int lim = (int)((n - base) < CHUNK ? (n - base) : CHUNK);
            T rv_cur = rv_sorted[cur];
            for (int i = 0; i < lim && cur < n_trials; i += 16) {
                if (i + 16 <= lim) {
                    T v[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) v[r] = b[i + r];
                    T cc = cum;
#pragma unroll
                    for (int r = 0; r < 16; ++r) cc = cc + v[r];
                    if (rv_cur > cc) {
                        cum = cc;
                        continue;
                    }
                }
                for (int r = 0; r < 16 && i + r < lim; ++r) {
                    cum = cum + b[i + r];
                    while (cur < n_trials && !(rv_cur > cum)) {
                        if (lane == 0) cand_s[trial_sorted[cur]] = (int)(base + i + r);
                        ++cur;
                        rv_cur = rv_sorted[cur];
                    }
                }
            }
            if (lane == 0 && cur >= n_trials) done_s = 1;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) buf[(c + 1) & 1][threadIdx.x * 4 + r] = nxt[r];
        __syncthreads();
        if (done_s) break;
    }
    if (wave == 0 && lane == 0) {
        // the running sum never reached these: the reference's loop stops at the last sample
        for (; cur < n_trials; ++cur) cand_s[trial_sorted[cur]] = (int)(n - 1);
    }
    __syncthreads();
    if (threadIdx.x < n_trials) {
        cand_next[threadIdx.x] = cand_s[threadIdx.x];
        if (cand_out) cand_out[threadIdx.x] = cand_s[threadIdx.x];
    }
    for (int t = 0; t < n_trials; ++t) {
        const int64_t cand = cand_s[t];
        for (int f = threadIdx.x; f < d; f += 256) cand_rows[(size_t)t * d + f] = X_t[(size_t)f * n + cand];
    }
}

struct KppPtrs {
    KppHeader* header;
    void* cand_rows;
    int32_t* cand;
    double* potentials;
    double* block_pot;
    void* rows;
};

KppPtrs kpp_ptrs(char* ws, const KppLayout& L) {
    KppPtrs p;
    p.header = (KppHeader*)(ws + L.off_header);
    p.cand = (int32_t*)(ws + L.off_cand);
    p.cand_rows = ws + L.off_cand_rows;
    p.potentials = (double*)(ws + L.off_pot);
    p.block_pot = (double*)(ws + L.off_block_pot);
    p.rows = ws + L.off_rows;
    return p;
}

int32_t kpp_check(const void* X_t, const void* w, void* ws, size_t ws_bytes, int64_t n, int d, int k,
                  int n_trials, int dtype) {
    KMX_REQUIRE_PTR(X_t);
    KMX_REQUIRE_PTR(w);
    KMX_REQUIRE_PTR(ws);
    if (n <= 0 || d <= 0 || k <= 0 || n > INT32_MAX) return KMX_ERR_BAD_SHAPE;
    if (n_trials <= 0 || n_trials > TN_MAX) return KMX_ERR_UNSUPPORTED;
    KMX_REQUIRE_DTYPE(dtype);
    if (ws_bytes < kpp_layout(n, d, n_trials, dtype).total) return KMX_ERR_WORKSPACE;
    return KMX_OK;
}

template <typename T>
void launch_init(const void* X_t, const void* w, int32_t start, void* centers_t, int32_t* idx,
                 const KppPtrs& p, const KppLayout& L, int64_t n, int d, int k, hipStream_t s, bool literal) {
    if (L.split) {
#define KMX_KPP_INIT_SPLIT_(SPT, LIT)                                                                 \
    hipLaunchKernelGGL((kpp_step_split_kernel<T, 1, SPT, true, LIT>), dim3((unsigned)L.n_blocks),    \
                       dim3(256), 0, s, (const T*)X_t, (const T*)w, (const T*)nullptr, (T*)p.rows,    \
                       p.block_pot, p.header, n, d, k, 1, start, (T*)centers_t, idx)
#define KMX_KPP_INIT_SPLIT(SPT) \
    do { if (literal) KMX_KPP_INIT_SPLIT_(SPT, true); else KMX_KPP_INIT_SPLIT_(SPT, false); } while (0)
        if (L.split == 1) KMX_KPP_INIT_SPLIT(1);
        else if (L.split == 2) KMX_KPP_INIT_SPLIT(2);
        else if constexpr (sizeof(T) == 4) KMX_KPP_INIT_SPLIT(4);  // (kpp_split: fp32 only)
#undef KMX_KPP_INIT_SPLIT_
#undef KMX_KPP_INIT_SPLIT
        return;
    }
#define KMX_KPP_INIT(FUSED)                                                                          \
    hipLaunchKernelGGL((kpp_step_kernel<T, 1, FUSED, true>), dim3((unsigned)L.n_blocks), dim3(256), 0, s, \
                       (const T*)X_t, (const T*)w, (const T*)nullptr, (T*)p.rows, p.block_pot, p.header, \
                       n, d, k, 1, start, (T*)centers_t, idx)
    if (literal) KMX_KPP_INIT(false); else KMX_KPP_INIT(true);
#undef KMX_KPP_INIT
}

template <typename T>
void launch_step(const void* X_t, const void* w, const int32_t* cand, const KppPtrs& p,
                 const KppLayout& L, int64_t n, int d, int n_trials, hipStream_t s, bool literal) {
    (void)cand;  // the candidates' rows were copied to p.cand_rows when they were sampled
    if (L.split) {
#define KMX_KPP_STEP_SPLIT_(TN, SPT, LIT)                                                              \
    hipLaunchKernelGGL((kpp_step_split_kernel<T, TN, SPT, false, LIT>), dim3((unsigned)L.n_blocks),    \
                       dim3(256), 0, s, (const T*)X_t, (const T*)w, (const T*)p.cand_rows, (T*)p.rows, \
                       p.block_pot, p.header, n, d, 0, n_trials, 0, (T*)nullptr,            \
                       (int32_t*)nullptr)
#define KMX_KPP_STEP_SPLIT(TN, SPT) \
    do { if (literal) KMX_KPP_STEP_SPLIT_(TN, SPT, true); else KMX_KPP_STEP_SPLIT_(TN, SPT, false); } while (0)
        // (which of these exist is kpp_split's choice: the workgroup's partial distances within 32 KB)
        if (n_trials <= 8) {
            if (L.split == 1) KMX_KPP_STEP_SPLIT(8, 1);
            else if (L.split == 2) KMX_KPP_STEP_SPLIT(8, 2);
            else if constexpr (sizeof(T) == 4) KMX_KPP_STEP_SPLIT(8, 4);
        } else {
            if (L.split == 1) KMX_KPP_STEP_SPLIT(TN_MAX, 1);
            else if constexpr (sizeof(T) == 4) KMX_KPP_STEP_SPLIT(TN_MAX, 2);
        }
#undef KMX_KPP_STEP_SPLIT
#undef KMX_KPP_STEP_SPLIT_
        return;
    }
#define KMX_KPP_STEP(TN, FUSED)                                                                      \
    hipLaunchKernelGGL((kpp_step_kernel<T, TN, FUSED, false>), dim3((unsigned)L.n_blocks), dim3(256), 0, s, \
                       (const T*)X_t, (const T*)w, (const T*)p.cand_rows, (T*)p.rows, p.block_pot,   \
                       p.header, n, d, 0, n_trials, 0, (T*)nullptr, (int32_t*)nullptr)
    if (n_trials <= 8) {
        if (literal) KMX_KPP_STEP(8, false); else KMX_KPP_STEP(8, true);
    } else {
        if (literal) KMX_KPP_STEP(TN_MAX, false); else KMX_KPP_STEP(TN_MAX, true);
    }
#undef KMX_KPP_STEP
}

// Whether kmx_kpp_run screens its steps where the workspace has room for the copies of X they read,
// and that room: the row-major copy, then the samples' tiles.
bool screen_wanted(const KppLayout& L, int64_t n, int d, int k, int n_trials) {
    return !L.split && n_trials <= SCREEN_TN && n >= SCREEN_MIN_N && k >= SCREEN_MIN_K && d >= SCREEN_MIN_D &&
           kmx_tiles_fit(n, d, k);
}

size_t screen_bytes(const KppLayout& L, int64_t n, int d, int k, int n_trials, int dtype) {
    if (!screen_wanted(L, n, d, k, n_trials)) return 0;
    return kmx_align256((size_t)n * d * kmx_dtype_size(dtype)) + kmx_align256(kmx_tiles_samples_bytes(n, d));
}

template <typename T>
int32_t launch_screen_step(const void* X_t, const void* X_rm, const KmxTiles& tiles, const void* w, const int32_t* cand,
                           const KppPtrs& p, const KppLayout& L, int64_t n, int d, int n_trials, hipStream_t s) {
    const size_t lds = screen_lds<T>(d, tiles.S);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&kpp_screen_step_kernel<T>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int32_t)e;
    }
    hipLaunchKernelGGL((kpp_screen_step_kernel<T>), dim3((unsigned)L.n_blocks), dim3(512), lds, s, (const T*)X_t,
                       (const T*)X_rm, tiles, (const T*)w, cand, (const T*)p.cand_rows, (T*)p.rows, p.block_pot,
                       p.header, n, d, n_trials);
    return KMX_OK;
}

template <typename T>
void launch_select_sample(const void* X_t, const double* uniforms, const int32_t* cand_prev,
                          int32_t* cand_next, int32_t* cand_out, void* centers_t, int32_t* idx,
                          const KppPtrs& p, const KppLayout& L, int64_t n, int d, int k,
                          int n_trials, int slot, int do_select, int do_sample, hipStream_t s,
                          bool literal = false, double* merged = nullptr, int merge = 0) {
    if (literal) {
        // the selection alone (potentials compared in T), then the serial walk of one workgroup
        if (do_select)
            launch_select_sample<T>(X_t, uniforms, cand_prev, cand_next, cand_out, centers_t, idx, p, L, n, d, k,
                                    n_trials, slot, 2, 0, s);
        if (do_sample)
            hipLaunchKernelGGL((kpp_sample_literal_kernel<T>), dim3(1), dim3(256), 0, s, (const T*)X_t, uniforms,
                               cand_next, cand_out, (const T*)p.rows, p.block_pot, p.header, (T*)p.cand_rows, n,
                               L.n_blocks, d, n_trials);
        return;
    }
    // one workgroup per trial when sampling, one more when a selection is recorded
    const unsigned grid = (do_sample ? (unsigned)n_trials : 0u) + (do_select ? 1u : 0u);
    if (grid == 0) return;
#define KMX_KPP_SELECT(...)                                                                       \
    hipLaunchKernelGGL((kpp_select_sample_kernel<T, __VA_ARGS__>), dim3(grid), dim3(256), 0, s,    \
                       (const T*)X_t, uniforms, cand_prev, cand_next, cand_out, (T*)centers_t, idx, \
                       (const T*)p.rows, p.block_pot, p.potentials, p.header, (T*)p.cand_rows, n,   \
                       L.n_blocks, L.chunk, d, k, n_trials, slot, do_select, do_sample, merged, merge)
    if (n_trials <= 8) {
        // (more than four block sums per thread: eight in registers rather than re-read)
        if (L.n_blocks > 4 * 256 && L.n_blocks <= 8 * 256) KMX_KPP_SELECT(8, 8);
        else KMX_KPP_SELECT(8);
    } else {
        KMX_KPP_SELECT(TN_MAX);
    }
#undef KMX_KPP_SELECT
}

// A whole seeding with one launch per centre (L.joint).
template <typename T>
int32_t run_joint(const void* X_t, const void* w, const double* uniforms, int32_t start, void* centers_t, int32_t* idx,
                  char* ws, const KppPtrs& p, const KppLayout& L, int64_t n, int d, int k, int n_trials, hipStream_t s) {
    const int n_blocks = (int)kmx_cdiv(n, 256 * L.joint);
    // step k - 1 writes the rows that kmx_kpp_closest_ptr names
    T* rows[2];
    rows[(k - 1) & 1] = (T*)p.rows;
    rows[k & 1] = (T*)(ws + L.off_rows2);
    double* pot = (double*)(ws + L.off_rows2 + kmx_align256((size_t)n_trials * n * sizeof(T)));
    double* pots[2] = {pot, pot + JOINT_TN * JOINT_BLOCKS};
#define KMX_KPP_JOINT(SPT, INIT, U, CP, CN, RI, RO, PI, PO, TRIALS, SLOT)                                                \
    hipLaunchKernelGGL((kpp_joint_kernel<T, SPT, INIT>), dim3((unsigned)n_blocks), dim3(256), 0, s, (const T*)X_t,      \
                       (const T*)w, U, CP, CN, RI, RO, PI, PO, (T*)centers_t, idx, p.potentials, p.header, n, d, k,     \
                       TRIALS, SLOT, start)
#define KMX_KPP_JOINT_SPT(...)                                              \
    do {                                                                    \
        if (L.joint == 1) KMX_KPP_JOINT(1, __VA_ARGS__);                    \
        else if (L.joint == 2) KMX_KPP_JOINT(2, __VA_ARGS__);               \
        else KMX_KPP_JOINT(4, __VA_ARGS__);                                 \
    } while (0)
    KMX_KPP_JOINT_SPT(true, (const double*)nullptr, (const int32_t*)nullptr, (int32_t*)nullptr, (const T*)nullptr, rows[0],
                      (const double*)nullptr, pots[0], 1, 0);
    KMX_LAUNCH_CHECK();
    for (int c = 1; c < k; ++c) {
        const double* u = uniforms + (size_t)(c - 1) * n_trials;
        KMX_KPP_JOINT_SPT(false, u, p.cand + ((c - 1) & 1) * TN_MAX, p.cand + (c & 1) * TN_MAX, (const T*)rows[(c - 1) & 1],
                          rows[c & 1], pots[(c - 1) & 1], pots[c & 1], n_trials, c - 1);
        KMX_LAUNCH_CHECK();
    }
#undef KMX_KPP_JOINT_SPT
#undef KMX_KPP_JOINT
    if (k > 1) {
        KppPtrs last = p;
        last.block_pot = pots[(k - 1) & 1];
        KppLayout geometry = L;
        geometry.n_blocks = n_blocks;
        geometry.chunk = 256 * L.joint;
        static_assert(JOINT_D <= SPLIT_MIN_D, "the block sums of the layout are those of CHUNK samples");
        launch_select_sample<T>(X_t, nullptr, p.cand + ((k - 1) & 1) * TN_MAX, nullptr, nullptr, centers_t, idx, last,
                                geometry, n, d, k, n_trials, k - 1, 1, 0, s, false, p.block_pot, CHUNK / geometry.chunk);
        KMX_LAUNCH_CHECK();
    }
    return KMX_OK;
}

}  // namespace

extern "C" {

size_t kmx_kpp_workspace_bytes(int64_t n, int32_t d, int32_t k, int32_t n_trials, int32_t dtype) {
    (void)k;
    if (n <= 0 || n_trials <= 0 || n_trials > TN_MAX || (dtype != KMX_F32 && dtype != KMX_F64))
        return 0;
    return kpp_layout(n, d, n_trials, dtype).total;
}

size_t kmx_kpp_screen_bytes(int64_t n, int32_t d, int32_t k, int32_t n_trials, int32_t dtype) {
    if (n <= 0 || d <= 0 || k <= 0 || n_trials <= 0 || n_trials > TN_MAX || (dtype != KMX_F32 && dtype != KMX_F64))
        return 0;
    return screen_bytes(kpp_layout(n, d, n_trials, dtype), n, d, k, n_trials, dtype);
}

int32_t kmx_kpp_init(const void* X_t, const void* sample_weight, int32_t start_index,
                     void* centers_t, int32_t* center_indices, void* workspace,
                     size_t workspace_bytes, int64_t n, int32_t d, int32_t k, int32_t n_trials,
                     int32_t dtype, uint32_t flags, void* stream_) {
    KMX_ENTRY();
    const int32_t rc = kpp_check(X_t, sample_weight, workspace, workspace_bytes, n, d, k, n_trials, dtype);
    if (rc != KMX_OK) return rc;
    KMX_REQUIRE_PTR(centers_t);
    KMX_REQUIRE_PTR(center_indices);
    if (flags & ~(uint32_t)KMX_KPP_SAMPLER_LITERAL) return KMX_ERR_BAD_ARGUMENT;
    const bool literal = (flags & KMX_KPP_SAMPLER_LITERAL) != 0;
    if (start_index < 0 || start_index >= n) return KMX_ERR_BAD_ARGUMENT;
    const KppLayout L = kpp_layout(n, d, n_trials, dtype);
    const KppPtrs p = kpp_ptrs((char*)workspace, L);
    hipStream_t s = (hipStream_t)stream_;
    if (dtype == KMX_F32)
        launch_init<float>(X_t, sample_weight, start_index, centers_t, center_indices, p, L, n, d, k, s, literal);
    else
        launch_init<double>(X_t, sample_weight, start_index, centers_t, center_indices, p, L, n, d, k, s, literal);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_kpp_sample_candidates(const void* X_t, const double* uniforms_for_step,
                                  int32_t* candidates, void* workspace, size_t workspace_bytes,
                                  int64_t n, int32_t d, int32_t k, int32_t n_trials, int32_t dtype,
                                  uint32_t flags, void* stream_) {
    KMX_ENTRY();
    KMX_REQUIRE_PTR(uniforms_for_step);
    if (flags & ~(uint32_t)KMX_KPP_SAMPLER_LITERAL) return KMX_ERR_BAD_ARGUMENT;
    const bool literal = (flags & KMX_KPP_SAMPLER_LITERAL) != 0;
    const int32_t rc = kpp_check(X_t, uniforms_for_step, workspace, workspace_bytes, n, d, k, n_trials, dtype);
    if (rc != KMX_OK) return rc;
    const KppLayout L = kpp_layout(n, d, n_trials, dtype);
    const KppPtrs p = kpp_ptrs((char*)workspace, L);
    hipStream_t s = (hipStream_t)stream_;
    if (dtype == KMX_F32)
        launch_select_sample<float>(X_t, uniforms_for_step, p.cand, p.cand, candidates, nullptr,
                                    nullptr, p, L, n, d, k, n_trials, 0, 0, 1, s, literal);
    else
        launch_select_sample<double>(X_t, uniforms_for_step, p.cand, p.cand, candidates, nullptr,
                                     nullptr, p, L, n, d, k, n_trials, 0, 0, 1, s, literal);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_kpp_step(const void* X_t, const void* sample_weight, int32_t center_slot,
                     void* centers_t, int32_t* center_indices, void* workspace,
                     size_t workspace_bytes, int64_t n, int32_t d, int32_t k, int32_t n_trials,
                     int32_t dtype, uint32_t flags, void* stream_) {
    KMX_ENTRY();
    const int32_t rc = kpp_check(X_t, sample_weight, workspace, workspace_bytes, n, d, k, n_trials, dtype);
    if (rc != KMX_OK) return rc;
    KMX_REQUIRE_PTR(centers_t);
    KMX_REQUIRE_PTR(center_indices);
    if (flags & ~(uint32_t)KMX_KPP_SAMPLER_LITERAL) return KMX_ERR_BAD_ARGUMENT;
    const bool literal = (flags & KMX_KPP_SAMPLER_LITERAL) != 0;
    if (center_slot < 1 || center_slot >= k) return KMX_ERR_BAD_ARGUMENT;
    const KppLayout L = kpp_layout(n, d, n_trials, dtype);
    const KppPtrs p = kpp_ptrs((char*)workspace, L);
    hipStream_t s = (hipStream_t)stream_;
    if (dtype == KMX_F32) {
        launch_step<float>(X_t, sample_weight, p.cand, p, L, n, d, n_trials, s, literal);
        launch_select_sample<float>(X_t, nullptr, p.cand, nullptr, nullptr, centers_t, center_indices,
                                    p, L, n, d, k, n_trials, center_slot, 1, 0, s, literal);
    } else {
        launch_step<double>(X_t, sample_weight, p.cand, p, L, n, d, n_trials, s, literal);
        launch_select_sample<double>(X_t, nullptr, p.cand, nullptr, nullptr, centers_t,
                                     center_indices, p, L, n, d, k, n_trials, center_slot, 1, 0, s, literal);
    }
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

int32_t kmx_kpp_run(const void* X_t, const void* sample_weight, const double* uniforms,
                    int32_t start_index, void* centers_t, int32_t* center_indices,
                    void* workspace, size_t workspace_bytes, int64_t n, int32_t d, int32_t k,
                    int32_t n_trials, int32_t dtype, uint32_t flags, void* stream_) {
    KMX_ENTRY();
    if (flags & ~(uint32_t)KMX_KPP_SAMPLER_LITERAL) return KMX_ERR_BAD_ARGUMENT;
    const bool literal = (flags & KMX_KPP_SAMPLER_LITERAL) != 0;
    int32_t rc = kpp_check(X_t, sample_weight, workspace, workspace_bytes, n, d, k, n_trials, dtype);
    if (rc != KMX_OK) return rc;
    const KppLayout L = kpp_layout(n, d, n_trials, dtype);
    const KppPtrs p = kpp_ptrs((char*)workspace, L);
    hipStream_t s = (hipStream_t)stream_;
    if (L.joint && !literal && k > 1) {
        KMX_REQUIRE_PTR(centers_t);
        KMX_REQUIRE_PTR(center_indices);
        KMX_REQUIRE_PTR(uniforms);
        if (start_index < 0 || start_index >= n) return KMX_ERR_BAD_ARGUMENT;
        return dtype == KMX_F32
                   ? run_joint<float>(X_t, sample_weight, uniforms, start_index, centers_t, center_indices,
                                      (char*)workspace, p, L, n, d, k, n_trials, s)
                   : run_joint<double>(X_t, sample_weight, uniforms, start_index, centers_t, center_indices,
                                       (char*)workspace, p, L, n, d, k, n_trials, s);
    }
    rc = kmx_kpp_init(X_t, sample_weight, start_index, centers_t, center_indices, workspace, workspace_bytes, n, d, k,
                      n_trials, dtype, flags, stream_);
    if (rc != KMX_OK) return rc;
    if (k == 1) return KMX_OK;
    KMX_REQUIRE_PTR(uniforms);
    const size_t extra = literal ? 0 : screen_bytes(L, n, d, k, n_trials, dtype);
    const bool screened = extra != 0 && workspace_bytes >= L.total + extra && ((uintptr_t)workspace & 15) == 0;
    void* X_rm = nullptr;
    KmxTiles tiles = {};
    if (screened) {
        X_rm = (char*)workspace + L.total;
        char* area = (char*)X_rm + kmx_align256((size_t)n * d * kmx_dtype_size(dtype));
        rc = kmx_tiles_prepare_samples(X_t, X_rm, area, n, d, dtype, s);
        if (rc != KMX_OK) return rc;
        tiles = kmx_tiles_view(area, n, d);
    }
    for (int c = 1; c < k; ++c) {
        const bool screen = screened && c >= SCREEN_FROM;
        // candidates alternate between two buffers: the fused launch reads the previous
        // step's candidates (to record its winner) while it writes the next ones
        int32_t* cand_prev = p.cand + ((c - 1) & 1) * TN_MAX;
        int32_t* cand_next = p.cand + (c & 1) * TN_MAX;
        const double* u = uniforms + (size_t)(c - 1) * n_trials;
        const int do_select = c > 1 ? 1 : 0;
        if (dtype == KMX_F32) {
            launch_select_sample<float>(X_t, u, cand_prev, cand_next, nullptr, centers_t,
                                        center_indices, p, L, n, d, k, n_trials, c - 1, do_select, 1, s, literal);
            if (screen)
                rc = launch_screen_step<float>(X_t, X_rm, tiles, sample_weight, cand_next, p, L, n, d, n_trials, s);
            else
                launch_step<float>(X_t, sample_weight, cand_next, p, L, n, d, n_trials, s, literal);
        } else {
            launch_select_sample<double>(X_t, u, cand_prev, cand_next, nullptr, centers_t,
                                         center_indices, p, L, n, d, k, n_trials, c - 1, do_select, 1, s, literal);
            if (screen)
                rc = launch_screen_step<double>(X_t, X_rm, tiles, sample_weight, cand_next, p, L, n, d, n_trials, s);
            else
                launch_step<double>(X_t, sample_weight, cand_next, p, L, n, d, n_trials, s, literal);
        }
        if (rc != KMX_OK) return rc;
        KMX_LAUNCH_CHECK();
    }
    int32_t* cand_last = p.cand + ((k - 1) & 1) * TN_MAX;
    if (dtype == KMX_F32)
        launch_select_sample<float>(X_t, nullptr, cand_last, nullptr, nullptr, centers_t,
                                    center_indices, p, L, n, d, k, n_trials, k - 1, 1, 0, s, literal);
    else
        launch_select_sample<double>(X_t, nullptr, cand_last, nullptr, nullptr, centers_t,
                                     center_indices, p, L, n, d, k, n_trials, k - 1, 1, 0, s, literal);
    KMX_LAUNCH_CHECK();
    return KMX_OK;
}

void* kmx_kpp_closest_ptr(void* workspace, int64_t n, int32_t d, int32_t k, int32_t n_trials,
                          int32_t dtype) {
    (void)k;
    if (!workspace || n <= 0 || n_trials <= 0) return nullptr;
    // start of the rows; the caller adds best_row * n elements (best_row from the header)
    return (char*)workspace + kpp_layout(n, d, n_trials, dtype).off_rows;
}

double* kmx_kpp_potentials_ptr(void* workspace, int64_t n, int32_t d, int32_t k, int32_t n_trials,
                               int32_t dtype) {
    (void)k;
    if (!workspace || n <= 0 || n_trials <= 0) return nullptr;
    return (double*)((char*)workspace + kpp_layout(n, d, n_trials, dtype).off_pot);
}

int32_t* kmx_kpp_candidates_ptr(void* workspace, int64_t n, int32_t d, int32_t k, int32_t n_trials,
                                int32_t dtype) {
    (void)k;
    if (!workspace || n <= 0 || n_trials <= 0) return nullptr;
    return (int32_t*)((char*)workspace + kpp_layout(n, d, n_trials, dtype).off_cand);
}

}  // extern "C"
