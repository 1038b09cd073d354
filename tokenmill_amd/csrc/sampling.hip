// Sampling over rows of 32-bit logits: argmax, and temperature sampling with optional top-k and
// top-p filters, one token per row                    (reference src/infer/sampling.py:12-46).
//
// The random number of a row is given by the caller (u in [0, 1), drawn from the request's own
// counter-based stream), so a request's tokens do not depend on its batch-mates. The token is the
// inverse CDF of the filtered softmax in vocabulary order. Filters are found by a radix descent
// over the bit patterns of the logits with integer histograms, so no sort is needed and the
// result does not depend on the order in which threads or blocks add.
#include "common.h"
#include "api.h"

#include <mutex>
#include <type_traits>

#define SM_NT 1024

// monotonic map float -> uint32 (larger float, larger key)
__device__ __forceinline__ uint32_t order_key(float f) {
    uint32_t u = f == 0.f ? 0u : __float_as_uint(f);        // -0 and +0 are one value: one key
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct ArgMax {
    float v;
    int i;
};

__device__ __forceinline__ ArgMax better(ArgMax a, ArgMax b) {
    // larger value wins; equal values: the lower index (the first maximum); NaN never wins
    if (b.i >= 0 && (a.i < 0 || b.v > a.v || (b.v == a.v && b.i < a.i))) return b;
    return a;
}

__device__ ArgMax block_argmax(const float* __restrict__ row, int V, ArgMax* smem /* SM_NT/64 */) {
    ArgMax best{-INFINITY, -1};
    for (int i = threadIdx.x; i < V; i += SM_NT) {
        const float v = row[i];
        if (v == v) best = better(best, ArgMax{v, i});
    }
#pragma unroll
    for (int off = TM_WAVE / 2; off > 0; off >>= 1) {
        ArgMax o{__shfl_xor(best.v, off, TM_WAVE), __shfl_xor(best.i, off, TM_WAVE)};
        best = better(best, o);
    }
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    __syncthreads();
    if (lane == 0) smem[wave] = best;
    __syncthreads();
    ArgMax r = smem[0];
    for (int w = 1; w < SM_NT / TM_WAVE; ++w) r = better(r, smem[w]);
    if (r.i < 0) r.i = 0;
    return r;
}

__global__ __launch_bounds__(SM_NT) void argmax_rows_kernel(const float* __restrict__ logits, int V,
                                                            int* __restrict__ out) {
    __shared__ ArgMax smem[SM_NT / TM_WAVE];
    const ArgMax r = block_argmax(logits + (size_t)blockIdx.x * V, V, smem);
    if (threadIdx.x == 0) out[blockIdx.x] = r.i;
}

// Two stages for wide vocabularies: a row is cut into NB chunks, one block each, then the NB
// candidates are reduced. Ties go to the lower index in both stages (the first maximum).
#define AM_NT 256
// clear (may be null): clear_per_row 64-bit words per row that the row's blocks set to zero between them
// (the sampler's histograms: no launch of its own for that). wave_v (may be null): the maximum of every wavefront's share
// (the entries threadIdx.x + j AM_NT of the chunk), NaN if it has none.
// Bound by reading the logits once; eight loads of a lane in flight (64 rows of 151,936: 20.0 us with one, 13.2 with eight).
__global__ __launch_bounds__(AM_NT) void argmax_partial_kernel(const float* __restrict__ logits, int V, int chunk,
                                                               float* __restrict__ part_v, int* __restrict__ part_i,
                                                               unsigned long long* __restrict__ clear,
                                                               int clear_per_row, float* __restrict__ wave_v) {
    __shared__ ArgMax smem[AM_NT / TM_WAVE];
    const int row = blockIdx.x, c = blockIdx.y, NB = gridDim.y;
    if (clear) {
        const int share = (clear_per_row + NB - 1) / NB;
        const int first = c * share, last = first + share < clear_per_row ? first + share : clear_per_row;
        for (int i = first + threadIdx.x; i < last; i += AM_NT) clear[(size_t)row * clear_per_row + i] = 0ull;
    }
    const int lo = c * chunk, hi = lo + chunk < V ? lo + chunk : V;
    const float* src = logits + (size_t)row * V;
    ArgMax best{-INFINITY, -1};
    for (int i = lo + threadIdx.x; i < hi; i += 8 * AM_NT) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = src[i + j * AM_NT < hi ? i + j * AM_NT : i];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (i + j * AM_NT < hi && v[j] == v[j]) best = better(best, ArgMax{v[j], i + j * AM_NT});
    }
#pragma unroll
    for (int off = TM_WAVE / 2; off > 0; off >>= 1) {
        ArgMax o{__shfl_xor(best.v, off, TM_WAVE), __shfl_xor(best.i, off, TM_WAVE)};
        best = better(best, o);
    }
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    if (lane == 0) {
        smem[wave] = best;
        if (wave_v) wave_v[((size_t)row * NB + c) * (AM_NT / TM_WAVE) + wave] = best.i < 0 ? NAN : best.v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        ArgMax r = smem[0];
        for (int w = 1; w < AM_NT / TM_WAVE; ++w) r = better(r, smem[w]);
        part_v[(size_t)row * NB + c] = r.v;
        part_i[(size_t)row * NB + c] = r.i;
    }
}

__global__ __launch_bounds__(TM_WAVE) void argmax_final_kernel(const float* __restrict__ part_v,
                                                               const int* __restrict__ part_i, int NB,
                                                               int* __restrict__ out) {
    const int row = blockIdx.x;
    ArgMax best{-INFINITY, -1};
    for (int c = threadIdx.x; c < NB; c += TM_WAVE)
        best = better(best, ArgMax{part_v[(size_t)row * NB + c], part_i[(size_t)row * NB + c]});
#pragma unroll
    for (int off = TM_WAVE / 2; off > 0; off >>= 1) {
        ArgMax o{__shfl_xor(best.v, off, TM_WAVE), __shfl_xor(best.i, off, TM_WAVE)};
        best = better(best, o);
    }
    if (threadIdx.x == 0) out[row] = best.i < 0 ? 0 : best.i;
}

// work: at least R * tm_argmax_work_chunks(V) floats and as many ints (may be null when that is 1 chunk)
extern "C" int tm_argmax_work_chunks(int V) {
    int nb = (V + 4095) / 4096;
    return nb < 1 ? 1 : (nb > 256 ? 256 : nb);
}

extern "C" int tm_argmax_rows(const float* logits, int R, int V, int* out, float* work_v, int* work_i,
                              hipStream_t stream) {
    if (R <= 0) return TM_OK;
    if (V <= 0) return TM_ERR_ARG;
    const int NB = tm_argmax_work_chunks(V);
    if (NB == 1 || !work_v || !work_i) {
        argmax_rows_kernel<<<R, SM_NT, 0, stream>>>(logits, V, out);
        TM_CHECK_LAUNCH();
        return TM_OK;
    }
    const int chunk = (V + NB - 1) / NB;
    argmax_partial_kernel<<<dim3(R, NB), AM_NT, 0, stream>>>(logits, V, chunk, work_v, work_i, nullptr, 0, nullptr);
    TM_CHECK_LAUNCH();
    argmax_final_kernel<<<R, TM_WAVE, 0, stream>>>(work_v, work_i, NB, out);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ---------------------------------------------------------------------------------------------------------
// The same argmax for callers that cannot allocate: the chunk candidates of the two-stage path live in
// a fixed array in device memory that is part of this library's image on every GPU it runs on.
//
// `argmax_scratch` names that array. In host code the name is only a handle for the runtime (not a
// device address): its address on the current device is asked for once per device
// (hipGetSymbolAddress) and kept; the kernels get that address as an argument, exactly as they get
// the caller's work buffers in tm_argmax_rows.
#define AM_STATIC_PAIRS (64 * 1024)                       // most (row, chunk) candidates: 512 KiB per GPU
#define AM_STATIC_DEVICES 64
static __device__ __align__(256) unsigned char argmax_scratch[AM_STATIC_PAIRS * (sizeof(float) + sizeof(int))];

static void* g_argmax_scratch[AM_STATIC_DEVICES];         // device address of the array, per device
static std::mutex g_argmax_scratch_mutex;

// The array's address on the device that is current now; null if the runtime cannot give it.
static void* argmax_scratch_here() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= AM_STATIC_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_argmax_scratch_mutex);
    if (!g_argmax_scratch[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(argmax_scratch)) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_argmax_scratch[dev] = p;
    }
    return g_argmax_scratch[dev];
}

extern "C" int tm_argmax_rows_static_max_pairs(void) { return AM_STATIC_PAIRS; }

extern "C" int tm_argmax_rows_static(const float* logits, int R, int V, int* out, hipStream_t stream) {
    if (R <= 0) return TM_OK;
    if (V <= 0 || !logits || !out) return TM_ERR_ARG;
    const int NB = tm_argmax_work_chunks(V);
    if (NB == 1) {                                         // a narrow row: one block, no scratch at all
        argmax_rows_kernel<<<R, SM_NT, 0, stream>>>(logits, V, out);
        TM_CHECK_LAUNCH();
        return TM_OK;
    }
    if ((long long)R * NB > AM_STATIC_PAIRS) return TM_ERR_ARG;      // beyond the fixed array: refused, nothing launched
    unsigned char* base = (unsigned char*)argmax_scratch_here();
    if (!base) return TM_ERR_LAUNCH;
    float* part_v = (float*)base;                                      // [R, NB]
    int* part_i = (int*)(base + (size_t)AM_STATIC_PAIRS * sizeof(float));   // [R, NB]
    // Nothing has to start at zero: the first kernel writes every (row, chunk) entry that the second reads.
    const int chunk = (V + NB - 1) / NB;
    argmax_partial_kernel<<<dim3(R, NB), AM_NT, 0, stream>>>(logits, V, chunk, part_v, part_i, nullptr, 0, nullptr);
    TM_CHECK_LAUNCH();
    argmax_final_kernel<<<R, TM_WAVE, 0, stream>>>(part_v, part_i, NB, out);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ---------------------------------------------------------------------------------------------------------
// Temperature sampling with top-k and top-p.
//
// A row of a wide vocabulary is cut into the chunks of the two-stage argmax (one block each), so a
// step's few rows still fill the chip; every stage is a launch over (row, chunk):
//   1. the chunk maxima (argmax_partial_kernel, which also clears the row's histograms) and the row
//      maximum (sample_bound_kernel): zmax for the softmax, and the token of a greedy row; and, for top-k, a
//      key that at least k entries reach, from the maxima of the chunks' wavefronts;
//   2. top-k, if some row asks for it: three launches, one per level of a radix descent (11, 11 and
//      10 bits of the order-preserving key of logit / temperature) that add the counts of the entries from that key up to
//      the row's histogram of that level; the blocks of the next level find the bucket that holds
//      the k-th largest entry from the histograms before it;
//   3. top-p over what top-k kept, if some row asks for it: the same descent with fixed-point
//      weights exp(z - zmax) * 2^32 instead of counts (the first level's histogram sums to the
//      kept mass Z, so the limit p * Z needs no pass of its own);
//   (2 to 4 where every row's k is small: one launch that gathers what may count into a list a row, and a block a row on it)
//   4. the kept mass of every chunk (sample_chunk_mass_kernel), then one block per row that walks
//      the chunks in vocabulary order to the one holding u * total and finds the token in it
//      (sample_pick_kernel).
// All histogram sums are integers, so they do not depend on the order in which blocks add; the
// float sums are taken in a fixed order that depends on V alone. A row's token depends on nothing
// but the row, its parameters and u.
// Ties at the k-th largest value are kept in vocabulary order until k entries are kept, and ties at the
// smallest value the nucleus reaches while the mass before them is at most p of the kept mass: the reference
// keeps entries by their rank in a descending sort (reference src/infer/sampling.py:15-23), which leaves the
// order of equal entries open; here, as in a stable sort, it is vocabulary order. -0 and +0 are equal.

#define SR_NT 256
#define SR_BINS 2048
#define SR_HIST_PER_ROW (6 * SR_BINS)        // three levels of the top-k descent, three of the top-p descent
#define SM_FIX 4294967296.0f                 // 2^32: fixed-point weight of exp(z - zmax) in (0, 1]

__device__ __forceinline__ unsigned long long fix_weight(float e) { return (unsigned long long)(e * SM_FIX); }
__device__ __forceinline__ int level_shift(int level) { return level == 0 ? 21 : (level == 1 ? 10 : 0); }
__device__ __forceinline__ int level_bins(int level) { return level == 2 ? 1024 : 2048; }
__device__ __forceinline__ float key_value(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key ^ 0x80000000u) : ~key);
}

struct RowParams {
    bool greedy, need_k, need_p;
    int k;
    float p, inv_t, zmax;
};

__device__ __forceinline__ RowParams row_params(int r, int V, const float* temperature, const int* top_k,
                                                const float* top_p, const float* rowmax) {
    RowParams rp;
    const float temp = temperature[r];
    const int k_raw = top_k[r];
    rp.greedy = temp <= 1e-5f || k_raw == 1;           // reference src/infer/engine/sequence.py:29-31
    rp.inv_t = rp.greedy ? 1.f : 1.f / temp;
    rp.k = (k_raw <= 0 || k_raw >= V) ? V : k_raw;
    rp.need_k = !rp.greedy && rp.k < V;
    rp.p = top_p[r];
    rp.need_p = !rp.greedy && rp.p < 1.f;
    rp.zmax = rowmax ? rowmax[r] * rp.inv_t : 0.f;
    return rp;
}

// Block-wide (SR_NT threads, all of them call): the bucket of one level's histogram, walking from
// the largest bucket down, in which
//   by count: the running count first reaches `limit`;
//   by mass : the running weight would first exceed `limit`
// (bucket 0 if that never happens), and the weight of the buckets above it added to `above`.
// frac >= 0: limit = frac * (the histogram's total - drop), returned through `limit` (first level by mass;
// drop: weight in the histogram that belongs to entries top-k does not keep after all, ties beyond its budget).
__device__ void pick_bucket(const unsigned long long* __restrict__ hist, int bins, bool by_mass, double frac,
                            unsigned long long drop, unsigned long long& limit, unsigned long long& above,
                            uint32_t& bucket, unsigned long long* s_scan /* SR_NT / 64 */, unsigned long long* s_res /* 2 */) {
    const int t = threadIdx.x, per = bins / SR_NT;
    unsigned long long local[SR_BINS / SR_NT];
    unsigned long long sum = 0;
#pragma unroll
    for (int j = 0; j < SR_BINS / SR_NT; ++j) {
        local[j] = j < per ? hist[bins - 1 - (t * per + j)] : 0ull;
        sum += local[j];
    }
    const int wave = t / TM_WAVE, lane = t % TM_WAVE;
    unsigned long long incl = sum;                       // inclusive scan over the threads
#pragma unroll
    for (int off = 1; off < TM_WAVE; off <<= 1) {
        const unsigned long long up = __shfl_up(incl, off, TM_WAVE);
        if (lane >= off) incl += up;
    }
    __syncthreads();                                     // s_scan and s_res may still be read from the call before
    if (lane == TM_WAVE - 1) s_scan[wave] = incl;
    __syncthreads();
    unsigned long long total = 0;
    for (int v = 0; v < SR_NT / TM_WAVE; ++v) {
        if (v < wave) incl += s_scan[v];
        total += s_scan[v];
    }
    const unsigned long long excl = incl - sum;
    if (frac >= 0.0) limit = (unsigned long long)((double)(total > drop ? total - drop : 0ull) * frac);
    auto reached = [&](unsigned long long run) { return by_mass ? run > limit : run >= limit; };
    if (t == SR_NT - 1 && !reached(above + total)) {     // never: bucket 0, everything above it counts
        s_res[0] = 0ull;
        s_res[1] = above + total - hist[0];
    }
    if (reached(above + incl) && !reached(above + excl)) {
        unsigned long long run = above + excl;
        int pick = per - 1;                              // the last of the thread's buckets if no earlier one
        bool open = true;
#pragma unroll
        for (int j = 0; j < SR_BINS / SR_NT; ++j) {
            if (open && j < per - 1) {
                if (reached(run + local[j])) {
                    pick = j;
                    open = false;
                } else {
                    run += local[j];
                }
            }
        }
        s_res[0] = (unsigned long long)(bins - 1 - (t * per + pick));
        s_res[1] = run;
    }
    __syncthreads();
    bucket = (uint32_t)s_res[0];
    above = s_res[1];
}

// Where a descent stands after some of its levels, left by the launch of each level for the next one: a block then walks one
// histogram, not all before it (64 rows of 151,936 with both filters: a launch of the top-p descent 28.6 to 12.3 us, with the shares below).
struct Descent {
    unsigned long long limit, above;
    uint32_t prefix, pad;
};

// The key of the k-th largest entry (by count) or the smallest key the nucleus keeps (by mass) from a
// row's three finished histograms; `above` = count / weight of the entries with a larger key. saved (may be null):
// [levels - 1] is where the descent stood one level earlier, for levels of two or more.
__device__ uint32_t descend(const unsigned long long* __restrict__ hist3, int levels, bool by_mass, double frac,
                            unsigned long long& limit, unsigned long long& above, uint32_t& mask,
                            unsigned long long* s_scan, unsigned long long* s_res, const Descent* __restrict__ saved,
                            unsigned long long drop = 0ull) {
    uint32_t prefix = 0;
    int first = 0;
    mask = 0;
    above = 0;
    if (saved && levels >= 2) {
        first = levels - 1;
        prefix = saved[first].prefix;
        above = saved[first].above;
        limit = saved[first].limit;
        for (int level = 0; level < first; ++level) mask |= (uint32_t)(level_bins(level) - 1) << level_shift(level);
    }
    for (int level = first; level < levels; ++level) {
        uint32_t bucket;
        pick_bucket(hist3 + (size_t)level * SR_BINS, level_bins(level), by_mass, level == 0 ? frac : -1.0, drop, limit,
                    above, bucket, s_scan, s_res);
        prefix |= bucket << level_shift(level);
        mask |= (uint32_t)(level_bins(level) - 1) << level_shift(level);
    }
    return prefix;
}

// Where top-k ends in a row (block-wide, all threads call; the row's three count histograms are finished):
// the key of the k-th largest entry, how many of the entries with that key stay (the first `budget` in
// vocabulary order: the entries with a larger key are fewer than k, the ties fill up to k), and the weight
// of the ties that do not stay (they are in the top-p histograms, which take every entry from that key up).
struct KEdge {
    uint32_t key;
    int budget;
    unsigned long long dropped;
};
__device__ KEdge k_edge(const unsigned long long* __restrict__ hist_k, const RowParams& rp,
                        unsigned long long* s_scan, unsigned long long* s_res, const Descent* __restrict__ saved) {
    unsigned long long limit = (unsigned long long)rp.k, above = 0;
    uint32_t mask;
    KEdge e;
    e.key = descend(hist_k, 3, false, -1.0, limit, above, mask, s_scan, s_res, saved);
    const long long budget = (long long)rp.k - (long long)above;         // above: entries strictly larger
    e.budget = budget > 0x7fffffffLL ? 0x7fffffff : (budget < 0 ? 0 : (int)budget);
    const unsigned long long ties = hist_k[2 * SR_BINS + (e.key & (uint32_t)(level_bins(2) - 1))];
    const unsigned long long cut = ties > (unsigned long long)e.budget ? ties - (unsigned long long)e.budget : 0ull;
    e.dropped = cut * fix_weight(expf(key_value(e.key) - rp.zmax));
    return e;
}

// What the launches of a row hand on.
struct RowState {
    Descent k[3], p[3];         // [level], level 1 and 2
    KEdge edge;                 // where top-k ends, from the first level of the top-p descent
    uint32_t bound;             // at least k entries have this key or a larger one (0: not known)
};

// A wavefront's share of a chunk in which every entry's key is below `floor` (block-wide thread layout of the chunk maxima).
__device__ __forceinline__ bool share_below(const float* __restrict__ wave_v, size_t chunk_at, float inv_t, uint32_t floor) {
    const float z = wave_v[chunk_at * (AM_NT / TM_WAVE) + threadIdx.x / TM_WAVE] * inv_t;
    return z == z && order_key(z) < floor;
}
static_assert(AM_NT == SR_NT && SR_NT == 256, "the wavefronts' shares of a chunk are the same in all launches");

// The k-th largest of the shares' maxima bounds the k-th largest entry from below: each maximum is an entry of its own. Shares
// below it take no part in top-k, and the ones below top-k's end none in what follows: with k = 50 two thirds of the shares of a
// row of 151,936 are passed over without a read, and next to no entry reaches the histograms' atomics. A share is a wavefront's,
// or, in rows of more than 64 chunks, a whole chunk's: one key a thread, and every thread counts the keys larger than its own,
// n steps (2.5 us for 152 keys; with all 980 wavefronts of a row of 1,000,000 it was 60 us, more than the bound saves: a row
// sampled with k = 50 68.9 us without a bound, 116.1 with that, 57.9 so).
__global__ __launch_bounds__(SR_NT) void sample_bound_kernel(const float* __restrict__ part_v, const int* __restrict__ part_i,
                                                             const float* __restrict__ wave_v, int NB, int V,
                                                             const float* __restrict__ temperature, const int* __restrict__ top_k,
                                                             const float* __restrict__ top_p, float* __restrict__ rowmax,
                                                             int* __restrict__ rowarg, RowState* __restrict__ state, int* __restrict__ counts) {
    __shared__ uint32_t s_key[SR_NT];
    __shared__ ArgMax s_best[SR_NT / TM_WAVE];
    __shared__ uint32_t s_bound;
    constexpr int WAVES = AM_NT / TM_WAVE;
    const int row = blockIdx.x, t = threadIdx.x;
    const bool by_wave = NB * WAVES <= SR_NT;
    const int n = by_wave ? NB * WAVES : NB;             // (a row has at most SR_NT chunks)
    const RowParams rp = row_params(row, V, temperature, top_k, top_p, nullptr);
    ArgMax best{-INFINITY, -1};
    if (t < NB) best = ArgMax{part_v[(size_t)row * NB + t], part_i[(size_t)row * NB + t]};
    uint32_t key = 0u;                                   // (no number's key is 0)
    if (t < n) {
        const float z = (by_wave ? wave_v[(size_t)row * n + t] : best.i < 0 ? NAN : best.v) * rp.inv_t;
        if (z == z) key = order_key(z);
    }
#pragma unroll
    for (int off = TM_WAVE / 2; off > 0; off >>= 1) {
        ArgMax o{__shfl_xor(best.v, off, TM_WAVE), __shfl_xor(best.i, off, TM_WAVE)};
        best = better(best, o);
    }
    if (t % TM_WAVE == 0) s_best[t / TM_WAVE] = best;
    s_key[t] = key;
    if (t == 0) s_bound = 0u;
    __syncthreads();
    if (t == 0) {
        for (int v = 1; v < SR_NT / TM_WAVE; ++v) best = better(best, s_best[v]);
        rowmax[row] = best.i < 0 ? 0.f : best.v;
        rowarg[row] = best.i < 0 ? 0 : best.i;
    }
    if (rp.need_k && rp.k <= n && t < n) {
        int larger = 0, level = 0;
        for (int j = 0; j < n; ++j) {
            larger += s_key[j] > key;
            level += s_key[j] == key;
        }
        if (larger < rp.k && larger + level >= rp.k) s_bound = key;        // (threads that write it write one value)
    }
    __syncthreads();
    if (t == 0) {
        state[row].bound = s_bound;
        counts[row] = 0;
    }
}

// The entries of a chunk that match the buckets picked so far, in a thread's share of it, into a histogram in LDS.
template <bool BY_MASS>
__device__ __forceinline__ void add_chunk(const float* __restrict__ row, int V, int chunk, int c, const RowParams& rp, int level, uint32_t floor_key,
                                          uint32_t prefix, uint32_t mask, unsigned long long* s_hist) {
    const int lo = c * chunk, hi = lo + chunk < V ? lo + chunk : V;
    const int shift = level_shift(level);
    const uint32_t digit_mask = (uint32_t)(level_bins(level) - 1);
    for (int i = lo + threadIdx.x; i < hi; i += 8 * SR_NT) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = row[i + j * SR_NT < hi ? i + j * SR_NT : i];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float z = v[j] * rp.inv_t;
            if (i + j * SR_NT >= hi || !(z == z)) continue;
            const uint32_t key = order_key(z);
            if (key < floor_key || (key & mask) != prefix) continue;
            atomicAdd(&s_hist[(key >> shift) & digit_mask], BY_MASS ? fix_weight(expf(z - rp.zmax)) : 1ull);
        }
    }
}

// One level of a descent: the chunk's entries that match the buckets picked so far, into the row's
// histogram of this level. BY_MASS: the top-p descent (weights, over what top-k kept).
template <bool BY_MASS>
__global__ __launch_bounds__(SR_NT) void sample_hist_kernel(const float* __restrict__ logits, int V, int chunk,
                                                            const float* __restrict__ temperature,
                                                            const int* __restrict__ top_k,
                                                            const float* __restrict__ top_p,
                                                            const float* __restrict__ rowmax,
                                                            unsigned long long* __restrict__ hist_all, int level,
                                                            const float* __restrict__ wave_v,
                                                            RowState* __restrict__ row_state, int stages) {
    __shared__ unsigned long long s_hist[SR_BINS];
    __shared__ unsigned long long s_scan[SR_NT / TM_WAVE];
    __shared__ unsigned long long s_res[2];
    const int r = blockIdx.x, c = blockIdx.y;
    const RowParams rp = row_params(r, V, temperature, top_k, top_p, rowmax);
    if (BY_MASS ? !rp.need_p : !rp.need_k) return;       // block-uniform
    unsigned long long* hist_k = hist_all + (size_t)r * SR_HIST_PER_ROW;
    unsigned long long* hist_p = hist_k + 3 * SR_BINS;
    uint32_t floor_key = 0, prefix = 0, mask = 0;
    unsigned long long limit = 0, above = 0;
    RowState& state = row_state[r];
    const bool writes = c == 0 && threadIdx.x == 0;
    if (BY_MASS) {
        unsigned long long dropped = 0;
        if (rp.need_k) {
            const KEdge e = level > 0 ? state.edge : k_edge(hist_k, rp, s_scan, s_res, (stages & 1) ? state.k : nullptr);
            floor_key = e.key;
            dropped = e.dropped;
            if (level == 0 && writes) state.edge = e;
        }
        prefix = descend(hist_p, level, true, (double)rp.p, limit, above, mask, s_scan, s_res, state.p, dropped);
    } else {
        limit = (unsigned long long)rp.k;
        prefix = descend(hist_k, level, false, -1.0, limit, above, mask, s_scan, s_res, state.k);
        floor_key = state.bound;
    }
    if (level > 0 && writes) (BY_MASS ? state.p : state.k)[level] = Descent{limit, above, prefix, 0u};
    const bool skip = share_below(wave_v, (size_t)r * gridDim.y + c, rp.inv_t, floor_key > prefix ? floor_key : prefix);
    if (__syncthreads_and(skip)) return;                 // nothing of this chunk counts
    for (int b = threadIdx.x; b < SR_BINS; b += SR_NT) s_hist[b] = 0ull;
    __syncthreads();
    if (!skip) add_chunk<BY_MASS>(logits + (size_t)r * V, V, chunk, c, rp, level, floor_key, prefix, mask, s_hist);
    __syncthreads();
    unsigned long long* dst = (BY_MASS ? hist_p : hist_k) + (size_t)level * SR_BINS;
    for (int b = threadIdx.x; b < SR_BINS; b += SR_NT)
        if (s_hist[b]) atomicAdd(&dst[b], s_hist[b]);
}

// What a row keeps, as the last two stages need it.
struct RowKeep {
    uint32_t p_key;             // entries with a larger key stay, entries with a smaller one go
    int ties_matter;            // entries equal to p_key stay only until tie_budget of them are kept, in
    int tie_budget;             // vocabulary order (top-k: until k entries stay; top-p: while the mass before
};                              // the entry is at most p; both: the smaller of the two)

// The kept weight of one entry without the ties at p_key (0 if it is dropped or such a tie), and whether
// it is such a tie.
__device__ __forceinline__ float entry_weight(float logit, const RowParams& rp, const RowKeep& keep, bool& tie) {
    const float z = logit * rp.inv_t;
    tie = false;
    if (!(z == z)) return 0.f;
    const uint32_t key = order_key(z);
    if (key < keep.p_key) return 0.f;
    if (keep.ties_matter && key == keep.p_key) {
        tie = true;
        return 0.f;
    }
    return expf(z - rp.zmax);
}

// Block-wide sums in a fixed order: lanes by a butterfly, wavefronts one after the other.
__device__ __forceinline__ void block_sums(float& w, int& n, float* s_w /* SR_NT / 64 */, int* s_n) {
#pragma unroll
    for (int off = TM_WAVE / 2; off > 0; off >>= 1) {
        w += __shfl_xor(w, off, TM_WAVE);
        n += __shfl_xor(n, off, TM_WAVE);
    }
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    __syncthreads();
    if (lane == 0) {
        s_w[wave] = w;
        s_n[wave] = n;
    }
    __syncthreads();
    w = s_w[0];
    n = s_n[0];
    for (int i = 1; i < SR_NT / TM_WAVE; ++i) {
        w += s_w[i];
        n += s_n[i];
    }
}

// What top-p leaves of what top-k kept: pk is the smallest key the nucleus reaches, limit = p * mass, above = mass of larger keys; the entries with that key
// stay while the mass before them is at most p of the kept mass (reference src/infer/sampling.py:20-23: ties in sorted order, which here is
// vocabulary order; the first always stays).
__device__ __forceinline__ void cut_nucleus(RowKeep& keep, const RowParams& rp, uint32_t pk, unsigned long long limit, unsigned long long above) {
    if (rp.need_k && pk < keep.p_key) return;
    const unsigned long long w = fix_weight(expf(key_value(pk) - rp.zmax));
    const unsigned long long room = limit > above ? limit - above : 0ull;
    const unsigned long long fit = w ? room / w + 1ull : 0x7fffffffull;
    const int by_mass = fit > 0x7fffffffull ? 0x7fffffff : (int)fit;
    const bool same = rp.need_k && pk == keep.p_key;
    keep.tie_budget = same && keep.tie_budget < by_mass ? keep.tie_budget : by_mass;
    keep.p_key = pk;
    keep.ties_matter = 1;
}

// The kept weight and the ties of a thread's share of a chunk.
__device__ __forceinline__ void chunk_share(const float* __restrict__ row, int V, int chunk, int c, const RowParams& rp, const RowKeep& keep, float& w,
                                            int& ties) {
    const int lo = c * chunk, hi = lo + chunk < V ? lo + chunk : V;
    for (int i = lo + threadIdx.x; i < hi; i += 8 * SR_NT) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = row[i + j * SR_NT < hi ? i + j * SR_NT : i];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            bool tie = false;
            if (i + j * SR_NT < hi) w += entry_weight(v[j], rp, keep, tie);
            ties += tie;
        }
    }
}

__global__ __launch_bounds__(SR_NT) void sample_chunk_mass_kernel(const float* __restrict__ logits, int V, int chunk,
                                                                  const float* __restrict__ temperature,
                                                                  const int* __restrict__ top_k,
                                                                  const float* __restrict__ top_p,
                                                                  const float* __restrict__ rowmax,
                                                                  const unsigned long long* __restrict__ hist_all,
                                                                  float* __restrict__ chunk_weight,
                                                                  int* __restrict__ chunk_ties,
                                                                  RowKeep* __restrict__ row_keep,
                                                                  const float* __restrict__ wave_v,
                                                                  const RowState* __restrict__ row_state, int stages) {
    __shared__ unsigned long long s_scan[SR_NT / TM_WAVE];
    __shared__ unsigned long long s_res[2];
    __shared__ float s_w[SR_NT / TM_WAVE];
    __shared__ int s_n[SR_NT / TM_WAVE];
    const int r = blockIdx.x, c = blockIdx.y, NB = gridDim.y;
    const RowParams rp = row_params(r, V, temperature, top_k, top_p, rowmax);
    if (rp.greedy) return;                               // block-uniform
    const unsigned long long* hist_k = hist_all + (size_t)r * SR_HIST_PER_ROW;
    const unsigned long long* hist_p = hist_k + 3 * SR_BINS;
    RowKeep keep{0u, 0, 0};
    unsigned long long dropped = 0;
    if (rp.need_k) {
        const KEdge e = rp.need_p && (stages & 2) ? row_state[r].edge : k_edge(hist_k, rp, s_scan, s_res, (stages & 1) ? row_state[r].k : nullptr);
        keep = RowKeep{e.key, 1, e.budget};
        dropped = e.dropped;
    }
    if (rp.need_p) {
        unsigned long long limit = 0, above = 0;
        uint32_t mask;
        const uint32_t pk = descend(hist_p, 3, true, (double)rp.p, limit, above, mask, s_scan, s_res,
                                    (stages & 2) ? row_state[r].p : nullptr, dropped);
        cut_nucleus(keep, rp, pk, limit, above);
    }
    if (c == 0 && threadIdx.x == 0) row_keep[r] = keep;
    float w = 0.f;
    int ties = 0;
    if (!share_below(wave_v, (size_t)r * NB + c, rp.inv_t, keep.p_key)) chunk_share(logits + (size_t)r * V, V, chunk, c, rp, keep, w, ties);
    block_sums(w, ties, s_w, s_n);
    if (threadIdx.x == 0) {
        chunk_weight[(size_t)r * NB + c] = w;
        chunk_ties[(size_t)r * NB + c] = ties;
    }
}

// --- rows whose top-k is small -----------------------------------------------------------------------------------------------
//
// What lies above the bound of sample_bound_kernel is little more than the k entries (k = 50 of 151,936: 60 to 70), so where every row of a call has such
// a k the entries are gathered into a list a row, one read of the shares that hold any, and a block a row finds in the list where top-k and
// top-p end, by counting, and sums the chunks' masses in the order of sample_chunk_mass_kernel. Of entries at the bound their number in every chunk is enough: a
// level that fills the shares (a masked vocabulary with fewer than k entries left, equal logits) needs no list. Seven launches over all chunks (six levels and
// the masses, 84 us for 64 rows of 151,936 with both filters, most of it launches whose blocks find nothing) are two of 15: a whole call of 64 / 8 / 1 rows
// 107.6 / 62.4 / 56.9 to 57.2 / 41.8 / 36.4 us, with k = 20 47.4 / 35.6 / 31.0, with 100 70.4 / 52.4 / 45.9.
//
// Where the large entries lie in fewer than k shares, far more are above the bound. A chunk with more than 2 k of them gathers again, what its k-th
// largest thread has and more, and the row's block narrows what is more than worth counting, up to SR_LIST_ALL entries, to the largest first, digit by
// digit. 1 / 64 rows, us, by the launches and so: 30 entries in -inf 65 / 224 and 37 / 59; 4,000 in one place, the rest -inf, k = 50 60 / 113 and 52 / 64, k =
// 100 60 / 114 and 68 / 86; half a vocabulary raised, k = 100, 60 / 124 and 63 / 90; 20,000 raised, k = 50, 58 / 91 and 50 / 61; sorted logits, k = 50 63 /
// 113 and 59 / 74, k = 100 65 / 124 and 74 / 97, of a million with k = 112 one row 96 and 130. What a list has no room for, more than SR_LIST equal entries
// above the bound in a chunk, is narrowed from the row itself (40,000 of two levels above a third: 65 / 137 and 224 / 246).
#define SR_LIST 256             // entries counted, one a thread
#define SR_LIST_ALL 16384       // entries a row's list has room for (SR_LIST of a chunk)

__global__ __launch_bounds__(SR_NT) void sample_gather_kernel(const float* __restrict__ logits, int V, int chunk, const float* __restrict__ temperature,
                                                              const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                              const float* __restrict__ rowmax, const float* __restrict__ wave_v,
                                                              const RowState* __restrict__ row_state, uint2* __restrict__ lists, int* __restrict__ counts,
                                                              int* __restrict__ chunk_ties) {
    __shared__ uint2 s_list[SR_LIST];
    __shared__ uint32_t s_best[SR_NT], s_floor;
    __shared__ int s_n, s_ties, s_base;
    const int r = blockIdx.x, c = blockIdx.y;
    const RowParams rp = row_params(r, V, temperature, top_k, top_p, rowmax);
    const uint32_t bound = row_state[r].bound;
    if (!rp.need_k || bound == 0u) return;               // block-uniform
    const bool skip = share_below(wave_v, (size_t)r * gridDim.y + c, rp.inv_t, bound);
    if (threadIdx.x == 0) s_n = s_ties = 0;
    if (__syncthreads_and(skip)) {
        if (threadIdx.x == 0) chunk_ties[(size_t)r * gridDim.y + c] = 0;
        return;
    }
    const float* row = logits + (size_t)r * V;
    const int lo = c * chunk, hi = lo + chunk < V ? lo + chunk : V;
    int ties = 0;
    uint32_t best = 0u;
    auto gather = [&](uint32_t floor) {
        for (int i = lo + threadIdx.x; i < hi && !skip; i += 8 * SR_NT) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = row[i + j * SR_NT < hi ? i + j * SR_NT : i];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float z = v[j] * rp.inv_t;
                if (i + j * SR_NT >= hi || !(z == z)) continue;
                const uint32_t key = order_key(z);
                ties += key == bound;
                if (key < floor) continue;
                best = key > best ? key : best;
                const int at = atomicAdd(&s_n, 1);
                if (at < SR_LIST) s_list[at] = uint2{key, (uint32_t)(i + j * SR_NT)};
            }
        }
    };
    gather(bound + 1);
    if (ties) atomicAdd(&s_ties, ties);
    __syncthreads();
    int n = s_n;
    if (threadIdx.x == 0) chunk_ties[(size_t)r * gridDim.y + c] = s_ties;
    if (n > 2 * rp.k && rp.k <= SR_NT) {
        // far more than can count: none below the k-th largest of the threads' largest does
        s_best[threadIdx.x] = best;
        if (threadIdx.x == 0) s_floor = bound + 1;
        __syncthreads();
        int larger = 0, level = 0;
#pragma unroll 8
        for (int i = 0; i < SR_NT; ++i) {
            larger += s_best[i] > best;
            level += s_best[i] == best;
        }
        if (best > bound && larger < rp.k && larger + level >= rp.k) s_floor = best;        // (threads that write it write one value)
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        gather(s_floor);
        __syncthreads();
        n = s_n;
    }
    if (threadIdx.x == 0 && n) s_base = atomicAdd(&counts[r], n <= SR_LIST ? n : SR_LIST_ALL + 1);
    __syncthreads();
    const int base = n ? s_base : 0;
    for (int i = threadIdx.x; i < n && i < SR_LIST && base + i < SR_LIST_ALL; i += SR_NT) lists[(size_t)r * SR_LIST_ALL + base + i] = s_list[i];
}

// Where narrow_list takes a row's entries from: its list, or, where that does not hold them, the row itself.
struct Entries {
    const uint2* list;
    int n;                      // in the list
    const float *row, *tops;    // tops: the largest of the shares of every chunk
    int V, chunk, NB;
    float inv_t;
};

// f(is there one, key, index) by every lane of a wavefront, for entries among which are all with keys of `floor` and more, 16 loads at a time. Of the row a
// wavefront goes through those of its shares by itself that hold such a key.
template <typename F>
__device__ __forceinline__ void for_entries(const Entries& e, uint32_t floor, F&& f) {
    constexpr int WAVES = SR_NT / TM_WAVE, DEEP = 16;
    static_assert(SR_LIST_ALL % (DEEP * SR_NT) == 0, "");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const bool listed = e.n <= SR_LIST_ALL;
    for (int c0 = 0; c0 < (listed ? 1 : e.NB); c0 += TM_WAVE) {
        unsigned long long left = 1ull;
        if (!listed) {
            const float top = e.tops[(c0 + lane < e.NB ? c0 + lane : e.NB - 1) * WAVES + wave] * e.inv_t;
            left = __ballot(c0 + lane < e.NB && !(top == top && order_key(top) < floor));
        }
        for (; left; left &= left - 1) {
            const int lo = listed ? 0 : (c0 + __builtin_ctzll(left)) * e.chunk, hi = listed ? e.n : lo + e.chunk < e.V ? lo + e.chunk : e.V;
            for (int o = lo + threadIdx.x; o - lane < hi; o += DEEP * SR_NT) {
                uint32_t key[DEEP], at[DEEP];
#pragma unroll
                for (int j = 0; j < DEEP; ++j) {
                    const int i = o + j * SR_NT < hi ? o + j * SR_NT : hi - 1;
                    if (listed) {
                        const uint2 x = e.list[i];
                        key[j] = x.x, at[j] = x.y;
                    } else {
                        key[j] = __float_as_uint(e.row[i]), at[j] = i;
                    }
                }
#pragma unroll
                for (int j = 0; j < DEEP; ++j) {
                    const float z = __uint_as_float(key[j]) * e.inv_t;
                    f(o + j * SR_NT < hi && (listed || z == z), listed ? key[j] : order_key(z), (int)at[j]);
                }
            }
        }
    }
}

// More than `most` entries of a row lie above the bound (one block, all threads call): a bound that leaves at most so many above it, or fewer than k (s_key,
// s_idx; s_ties the entries at it by chunk, where they are needed to fill up to k), from the k-th largest entry's key digit by digit.
__device__ __forceinline__ int narrow_list(const Entries& e, const RowParams& rp, int most, uint32_t& bound, unsigned long long* s_hist, unsigned long long* s_scan,
                                           unsigned long long* s_res, uint32_t* s_key, uint32_t* s_idx, int* s_ties, int* s_count) {
    const int t = threadIdx.x, lane = t % TM_WAVE;
    unsigned long long limit = (unsigned long long)rp.k, above = 0;
    uint32_t prefix = 0, mask = 0;
    bool exact = true;
    for (int level = 0; level < 3; ++level) {
        const int shift = level_shift(level);
        const uint32_t digit_mask = (uint32_t)(level_bins(level) - 1);
        for (int b = t; b < SR_BINS; b += SR_NT) s_hist[b] = 0ull;
        __syncthreads();
        for_entries(e, bound + 1 > prefix ? bound + 1 : prefix, [&](bool in, uint32_t key, int) {
            in = in && key > bound && (key & mask) == prefix;
            const uint32_t digit = (key >> shift) & digit_mask;
            // equal digits of a wavefront at once (large entries share their exponents, and one counter would take them one by one)
            unsigned long long left = __ballot(in);
            for (int turn = 0; left && turn < 3; ++turn) {
                const uint32_t d = __builtin_amdgcn_readlane(digit, __builtin_ctzll(left));
                const unsigned long long same = __ballot(in && digit == d);
                if (lane == __builtin_ctzll(same)) atomicAdd(&s_hist[d], (unsigned long long)__popcll(same));
                left &= ~same;
                in = in && digit != d;
            }
            if (in) atomicAdd(&s_hist[digit], 1ull);
        });
        __syncthreads();
        uint32_t bucket;
        pick_bucket(s_hist, level_bins(level), false, -1.0, 0ull, limit, above, bucket, s_scan, s_res);
        const int held = (int)s_hist[bucket];
        __syncthreads();
        prefix |= bucket << shift;
        mask |= digit_mask << shift;
        if (level < 2 && above + (unsigned long long)held <= (unsigned long long)most) {      // (they hold the k-th largest: no tie at the bound is needed)
            exact = false;
            --prefix;
            break;
        }
    }
    bound = prefix;
    for (int c = t; c < e.NB; c += SR_NT) s_ties[c] = 0;
    if (t == 0) *s_count = 0;
    __syncthreads();
    for_entries(e, exact ? bound : bound + 1, [&](bool in, uint32_t key, int i) {
        if (exact && in && key == bound) atomicAdd(&s_ties[i / e.chunk], 1);
        if (in && key > bound) {
            const int at = atomicAdd(s_count, 1);
            if (at < SR_LIST) {                          // (no more are above the bound)
                s_key[at] = key;
                s_idx[at] = (uint32_t)i;
            }
        }
    });
    __syncthreads();
    return *s_count;
}

// The same from the row itself, by one block: rows without a bound, which a caller who says that every k is small does not have.
__device__ void select_from_row(const float* __restrict__ row, int V, int chunk, int NB, const RowParams& rp, unsigned long long* __restrict__ hist,
                                unsigned long long* s_hist, unsigned long long* s_scan, unsigned long long* s_res, float* s_w, int* s_n,
                                float* __restrict__ chunk_weight, int* __restrict__ chunk_ties, RowKeep& keep) {
    keep = RowKeep{0u, 0, 0};
    unsigned long long dropped = 0, limit = 0, above = 0;
    uint32_t mask, floor_key = 0;
    auto levels = [&](auto BY_MASS, unsigned long long* h, double frac) {
        constexpr bool by_mass = decltype(BY_MASS)::value;
        for (int level = 0; level < 3; ++level) {
            limit = (unsigned long long)rp.k;
            const uint32_t prefix = descend(h, level, by_mass, frac, limit, above, mask, s_scan, s_res, nullptr, dropped);
            for (int b = threadIdx.x; b < SR_BINS; b += SR_NT) s_hist[b] = 0ull;
            __syncthreads();
            for (int c = 0; c < NB; ++c) add_chunk<by_mass>(row, V, chunk, c, rp, level, floor_key, prefix, mask, s_hist);
            __syncthreads();
            for (int b = threadIdx.x; b < SR_BINS; b += SR_NT) h[(size_t)level * SR_BINS + b] = s_hist[b];
            __threadfence_block();
            __syncthreads();
        }
    };
    if (rp.need_k) {
        levels(std::false_type{}, hist, -1.0);
        const KEdge e = k_edge(hist, rp, s_scan, s_res, nullptr);
        keep = RowKeep{e.key, 1, e.budget};
        floor_key = e.key;
        dropped = e.dropped;
    }
    if (rp.need_p) {
        unsigned long long* h = hist + 3 * SR_BINS;
        levels(std::true_type{}, h, (double)rp.p);
        const uint32_t pk = descend(h, 3, true, (double)rp.p, limit, above, mask, s_scan, s_res, nullptr, dropped);
        cut_nucleus(keep, rp, pk, limit, above);
    }
    for (int c = 0; c < NB; ++c) {
        float w = 0.f;
        int ties = 0;
        chunk_share(row, V, chunk, c, rp, keep, w, ties);
        block_sums(w, ties, s_w, s_n);
        if (threadIdx.x == 0) {
            chunk_weight[c] = w;
            chunk_ties[c] = ties;
        }
    }
}

__global__ __launch_bounds__(SR_NT) void sample_select_kernel(const float* __restrict__ logits, int V, int chunk, int NB,
                                                              const float* __restrict__ temperature, const int* __restrict__ top_k,
                                                              const float* __restrict__ top_p, const float* __restrict__ rowmax,
                                                              const float* __restrict__ wave_v, const RowState* __restrict__ row_state,
                                                              const uint2* __restrict__ lists, const int* __restrict__ counts,
                                                              unsigned long long* __restrict__ hist_all, float* __restrict__ chunk_weight,
                                                              int* __restrict__ chunk_ties, RowKeep* __restrict__ row_keep) {
    __shared__ unsigned long long s_hist[SR_BINS];       // (the list's weights lie in it)
    __shared__ uint32_t s_key[SR_LIST], s_idx[SR_LIST];
    __shared__ unsigned long long s_scan[SR_NT / TM_WAVE], s_res[2];
    __shared__ float s_w[SR_NT / TM_WAVE];
    __shared__ int s_n[SR_NT / TM_WAVE];
    __shared__ int s_begin[256], s_ties[256], s_total, s_count;
    __shared__ RowKeep s_keep;
    __shared__ unsigned long long s_limit;
    constexpr int GROUP = 8;
    const int r = blockIdx.x, t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / TM_WAVE), lane = t % TM_WAVE;
    const RowParams rp = row_params(r, V, temperature, top_k, top_p, rowmax);
    if (rp.greedy) return;                               // block-uniform
    int n = counts[r];
    uint32_t bound = row_state[r].bound;
    chunk_weight += (size_t)r * NB;
    chunk_ties += (size_t)r * NB;
    if (!rp.need_k || bound == 0u) {
        RowKeep keep;
        select_from_row(logits + (size_t)r * V, V, chunk, NB, rp, hist_all + (size_t)r * SR_HIST_PER_ROW, s_hist, s_scan, s_res, s_w, s_n, chunk_weight,
                        chunk_ties, keep);
        if (t == 0) row_keep[r] = keep;
        return;
    }
    // the list, and how many entries of every chunk are at the bound
    uint2 mine[SR_LIST / SR_NT];
    const int most = 2 * rp.k + 32 < SR_LIST ? 2 * rp.k + 32 : SR_LIST;     // (an entry costs 0.1 us, narrowing some 15)
    if (n > most) {
        const Entries e{lists + (size_t)r * SR_LIST_ALL, n, logits + (size_t)r * V, wave_v + (size_t)r * NB * (AM_NT / TM_WAVE), V, chunk, NB, rp.inv_t};
        n = narrow_list(e, rp, most, bound, s_hist, s_scan, s_res, s_key, s_idx, s_ties, &s_count);
#pragma unroll
        for (int j = 0; j < SR_LIST / SR_NT; ++j) mine[j] = uint2{s_key[t + j * SR_NT], s_idx[t + j * SR_NT]};
    } else {
#pragma unroll
        for (int j = 0; j < SR_LIST / SR_NT; ++j) mine[j] = lists[(size_t)r * SR_LIST_ALL + (t + j * SR_NT < n ? t + j * SR_NT : 0)];
        for (int c = t; c < NB; c += SR_NT) s_ties[c] = chunk_ties[c];
    }
    if (t == 0) s_total = 0;
    __syncthreads();
    for (int c = t; c < NB; c += SR_NT) {
        s_begin[c] = n;
        if (s_ties[c]) atomicAdd(&s_total, s_ties[c]);
    }
    // ... by vocabulary order
#pragma unroll
    for (int j = 0; j < SR_LIST / SR_NT; ++j)            // (what pads the list to whole groups is behind all, smaller than all, and weighs nothing)
        s_idx[t + j * SR_NT] = t + j * SR_NT < n ? mine[j].y : 0xffffffffu;
    __syncthreads();
    const int padded = (n + GROUP - 1) / GROUP * GROUP;
    int place[SR_LIST / SR_NT];
#pragma unroll
    for (int j = 0; j < SR_LIST / SR_NT; ++j) place[j] = 0;
    for (int i0 = 0; i0 < padded; i0 += GROUP) {
        uint32_t other[GROUP];
#pragma unroll
        for (int i = 0; i < GROUP; ++i) other[i] = s_idx[i0 + i];
#pragma unroll
        for (int i = 0; i < GROUP; ++i)
#pragma unroll
            for (int j = 0; j < SR_LIST / SR_NT; ++j) place[j] += other[i] < mine[j].y;
    }
    __syncthreads();
    unsigned long long* s_weight = s_hist;
    for (int i = n + t; i < padded; i += SR_NT) {
        s_key[i] = 0u;
        s_weight[i] = 0ull;
    }
#pragma unroll
    for (int j = 0; j < SR_LIST / SR_NT; ++j) {
        if (t + j * SR_NT >= n) continue;
        s_key[place[j]] = mine[j].x;
        s_idx[place[j]] = mine[j].y;
        s_weight[place[j]] = fix_weight(expf(key_value(mine[j].x) - rp.zmax));
    }
    __syncthreads();
    // of every entry: how many are larger, their mass, and how many are equal
    int larger[SR_LIST / SR_NT], equal[SR_LIST / SR_NT];
    unsigned long long above[SR_LIST / SR_NT];
    uint32_t key[SR_LIST / SR_NT];
#pragma unroll
    for (int j = 0; j < SR_LIST / SR_NT; ++j) {
        larger[j] = equal[j] = 0;
        above[j] = 0ull;
        key[j] = t + j * SR_NT < n ? s_key[t + j * SR_NT] : 0u;
    }
    for (int i0 = 0; i0 < padded; i0 += GROUP) {
        uint32_t other[GROUP];
        unsigned long long w[GROUP];
#pragma unroll
        for (int i = 0; i < GROUP; ++i) other[i] = s_key[i0 + i], w[i] = s_weight[i0 + i];
#pragma unroll
        for (int i = 0; i < GROUP; ++i)
#pragma unroll
            for (int j = 0; j < SR_LIST / SR_NT; ++j) {
                larger[j] += other[i] > key[j];
                equal[j] += other[i] == key[j];
                above[j] += other[i] > key[j] ? w[i] : 0ull;
            }
    }
    // the k-th largest; the mass from it up, without the ties that do not stay, times p
#pragma unroll
    for (int j = 0; j < SR_LIST / SR_NT; ++j) {
        if (t + j * SR_NT >= n || larger[j] >= rp.k || larger[j] + equal[j] < rp.k) continue;
        const unsigned long long w = s_weight[t + j * SR_NT];
        const int budget = rp.k - larger[j];
        const unsigned long long dropped = (unsigned long long)(equal[j] - budget) * w, total = above[j] + (unsigned long long)equal[j] * w;
        s_keep = RowKeep{key[j], 1, budget};             // (threads that write them write the same)
        s_limit = (unsigned long long)((double)(total > dropped ? total - dropped : 0ull) * (double)rp.p);
    }
    // ... which is the bound, where the list is shorter than k
    const unsigned long long w_bound = fix_weight(expf(key_value(bound) - rp.zmax));
    unsigned long long listed = 0ull;
    if (n < rp.k) {
        for (int i = 0; i < padded; i += GROUP)
#pragma unroll
            for (int j = 0; j < GROUP; ++j) listed += s_weight[i + j];
        if (t == 0) {
            const int ties = s_total, budget = rp.k - n;
            const unsigned long long dropped = ties > budget ? (unsigned long long)(ties - budget) * w_bound : 0ull;
            const unsigned long long total = listed + (unsigned long long)ties * w_bound;
            s_keep = RowKeep{bound, 1, budget};
            s_limit = (unsigned long long)((double)(total > dropped ? total - dropped : 0ull) * (double)rp.p);
        }
    }
    __syncthreads();
    if (rp.need_p) {
        const unsigned long long limit = s_limit;
        const RowKeep kept = s_keep;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SR_LIST / SR_NT; ++j) {
            if (t + j * SR_NT >= n || key[j] < kept.p_key) continue;
            if (above[j] > limit || above[j] + (unsigned long long)equal[j] * s_weight[t + j * SR_NT] <= limit) continue;
            RowKeep keep = kept;
            cut_nucleus(keep, rp, key[j], limit, above[j]);
            s_keep = keep;
        }
        if (t == 0 && n < rp.k && listed <= limit && listed + (unsigned long long)s_total * w_bound > limit) {
            RowKeep keep = kept;
            cut_nucleus(keep, rp, bound, limit, listed);
            s_keep = keep;
        }
        __syncthreads();
    }
    const RowKeep keep = s_keep;
    const bool at_bound = keep.p_key == bound;           // (the ties are the bound's, none of which is in the list)
    if (t == 0) row_keep[r] = keep;
    // the chunks' masses: lanes and wavefronts have the entries that are theirs in sample_chunk_mass_kernel, added as there
    for (int i = t; i < n; i += SR_NT) {
        const int c = (int)s_idx[i] / chunk;
        if (i == 0 || (int)s_idx[i - 1] / chunk != c) s_begin[c] = i;
    }
    __syncthreads();
    for (int c = t; c < NB; c += SR_NT)
        if (s_begin[c] == n) {
            chunk_weight[c] = 0.f;
            chunk_ties[c] = at_bound ? s_ties[c] : 0;
        }
    for (int c0 = 0; c0 < NB; c0 += TM_WAVE) {
        // of the chunks that have entries, a wavefront takes every fourth
        unsigned long long left = __ballot(c0 + lane < NB && s_begin[c0 + lane < NB ? c0 + lane : 0] < n);
        for (int turn = 0; left; left &= left - 1, ++turn) {
            if (turn % (SR_NT / TM_WAVE) != wave) continue;
            const int c = c0 + __builtin_ctzll(left), lo = c * chunk, hi = lo + chunk;
            float w[SR_NT / TM_WAVE];
            int ties = 0;
#pragma unroll
            for (int v = 0; v < SR_NT / TM_WAVE; ++v) w[v] = 0.f;
            for (int i = s_begin[c]; i < n && (int)s_idx[i] < hi; ++i) {     // the same in every lane
                const int off = (int)s_idx[i] - lo;
                const uint32_t k = s_key[i];
                ties += k == keep.p_key;
                const float e = k > keep.p_key ? expf(key_value(k) - rp.zmax) : 0.f;
#pragma unroll
                for (int v = 0; v < SR_NT / TM_WAVE; ++v)
                    if (off % SR_NT == v * TM_WAVE + lane) w[v] += e;
            }
#pragma unroll
            for (int v = 0; v < SR_NT / TM_WAVE; ++v) w[v] = lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(lane_sum<16>(lane_sum<32>(w[v]))))));
            float sum = w[0];
#pragma unroll
            for (int v = 1; v < SR_NT / TM_WAVE; ++v) sum += w[v];
            if (lane == 0) {
                chunk_weight[c] = sum;
                chunk_ties[c] = at_bound ? s_ties[c] : ties;
            }
        }
    }
}

// The largest k for which the calls of a vocabulary may say that their rows' entries fit a list: three quarters of the shares whose maxima bound them
// (up to 1.4 entries a share reach it then), and no more than counting them is worth.
extern "C" int tm_sample_list_k(int V) {
    const int NB = tm_argmax_work_chunks(V), shares = NB * (AM_NT / TM_WAVE) <= SR_NT ? NB * (AM_NT / TM_WAVE) : NB;
    return V > 0 && NB > 1 ? (shares * 3 / 4 < 112 ? shares * 3 / 4 : 112) : 0;
}

// Of `ties` ties that follow `seen` earlier ones, how many stay.
__device__ __forceinline__ int kept_ties(const RowKeep& keep, int seen, int ties) {
    const int room = keep.tie_budget - seen;
    return room <= 0 ? 0 : (room < ties ? room : ties);
}

// Walks n masses (weight[i] + kept ties of ties[i] * w_tie) in order to the one that holds `target`
// (the last one with any mass if rounding left the target beyond the end); one thread calls it.
struct Walk {
    int pick, seen;             // -1 if nothing has mass; ties before the picked one
    float before;               // mass before the picked one
};
__device__ __forceinline__ Walk walk_to(const float* weight, const int* ties, int n, const RowKeep& keep, float w_tie,
                                        float target, float run, int seen) {
    Walk last{-1, 0, 0.f};
    for (int i = 0; i < n; ++i) {
        const float mass = weight[i] + (float)kept_ties(keep, seen, ties[i]) * w_tie;
        if (mass > 0.f) {
            last = Walk{i, seen, run};
            if (target < run + mass) return last;
        }
        run += mass;
        seen += ties[i];
    }
    return last;
}

#define SR_MAX_CHUNKS 256
#define SR_MAX_ROWS 16          // a chunk has at most 4096 entries: 16 lines of SR_NT

__global__ __launch_bounds__(SR_NT) void sample_pick_kernel(const float* __restrict__ logits, int V, int chunk, int NB,
                                                            const float* __restrict__ temperature,
                                                            const int* __restrict__ top_k,
                                                            const float* __restrict__ top_p,
                                                            const float* __restrict__ rowmax,
                                                            const int* __restrict__ rowarg,
                                                            const float* __restrict__ chunk_weight,
                                                            const int* __restrict__ chunk_ties,
                                                            const RowKeep* __restrict__ row_keep,
                                                            const float* __restrict__ u, int* __restrict__ out) {
    __shared__ float s_cw[SR_MAX_CHUNKS];
    __shared__ int s_ct[SR_MAX_CHUNKS];
    __shared__ float s_lw[SR_MAX_ROWS];
    __shared__ int s_lt[SR_MAX_ROWS];
    __shared__ float s_w[SR_NT / TM_WAVE];
    __shared__ int s_n[SR_NT / TM_WAVE];
    __shared__ float s_pw[SR_NT / TM_WAVE][SR_MAX_ROWS];
    __shared__ int s_pn[SR_NT / TM_WAVE][SR_MAX_ROWS];
    __shared__ Walk s_walk;
    __shared__ float s_target;
    __shared__ int s_first, s_last;
    const int r = blockIdx.x;
    const RowParams rp = row_params(r, V, temperature, top_k, top_p, rowmax);
    if (rp.greedy) {
        if (threadIdx.x == 0) out[r] = rowarg[r];
        return;
    }
    const RowKeep keep = row_keep[r];
    const float u_row = u[r];
    const float w_tie = keep.ties_matter ? expf(key_value(keep.p_key) - rp.zmax) : 0.f;
    // 1. the chunk that holds u * total, walking the chunks in vocabulary order
    for (int c = threadIdx.x; c < NB; c += SR_NT) {
        s_cw[c] = chunk_weight[(size_t)r * NB + c];
        s_ct[c] = chunk_ties[(size_t)r * NB + c];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        int seen = 0;
        for (int c = 0; c < NB; ++c) {
            total += s_cw[c] + (float)kept_ties(keep, seen, s_ct[c]) * w_tie;
            seen += s_ct[c];
        }
        s_target = u_row * total;
        s_walk = walk_to(s_cw, s_ct, NB, keep, w_tie, s_target, 0.f, 0);
        s_first = 0x7fffffff;
        s_last = -1;
    }
    __syncthreads();
    const Walk at_chunk = s_walk;
    const float target = s_target;
    if (at_chunk.pick < 0) {                             // nothing kept (every entry NaN): the first maximum
        if (threadIdx.x == 0) out[r] = rowarg[r];
        return;
    }
    // 2. the line of SR_NT consecutive entries of that chunk: a thread holds one entry of every line (all
    //    loads in flight at once), the lines are summed lanes first, wavefronts one after the other
    const float* row = logits + (size_t)r * V;
    const int lo = at_chunk.pick * chunk, hi = lo + chunk < V ? lo + chunk : V;
    const int lines = (hi - lo + SR_NT - 1) / SR_NT;
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    float raw[SR_MAX_ROWS];
#pragma unroll
    for (int j = 0; j < SR_MAX_ROWS; ++j) {
        const int i = lo + j * SR_NT + (int)threadIdx.x;
        raw[j] = row[i < hi ? i : hi - 1];
    }
    float wj[SR_MAX_ROWS];
    uint32_t tie_bits = 0;
#pragma unroll
    for (int j = 0; j < SR_MAX_ROWS; ++j) {
        const int i = lo + j * SR_NT + (int)threadIdx.x;
        bool tie = false;
        wj[j] = i < hi ? entry_weight(raw[j], rp, keep, tie) : 0.f;
        tie_bits |= (tie ? 1u : 0u) << j;
        // (by the vector unit and a ballot: through LDS the launch took 2 us longer)
        const float w = lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(lane_sum<16>(lane_sum<32>(wj[j]))))));
        const int n = __popcll(__ballot(tie));
        if (lane == 0) {
            s_pw[wave][j] = w;
            s_pn[wave][j] = n;
        }
    }
    __syncthreads();
    if (threadIdx.x < SR_MAX_ROWS) {
        float w = s_pw[0][threadIdx.x];
        int n = s_pn[0][threadIdx.x];
        for (int v = 1; v < SR_NT / TM_WAVE; ++v) {
            w += s_pw[v][threadIdx.x];
            n += s_pn[v][threadIdx.x];
        }
        s_lw[threadIdx.x] = w;
        s_lt[threadIdx.x] = n;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const Walk in_chunk = walk_to(s_lw, s_lt, lines, keep, w_tie, target, at_chunk.before, at_chunk.seen);
        s_walk = in_chunk;
    }
    __syncthreads();
    const Walk at_line = s_walk;
    if (at_line.pick < 0) {                              // (sums of another order saw mass here: take the maximum)
        if (threadIdx.x == 0) out[r] = rowarg[r];
        return;
    }
    // 3. the entry of that line: each thread its entry of it, a running sum over the threads in order
    const int i = lo + at_line.pick * SR_NT + (int)threadIdx.x;
    float w = 0.f;
#pragma unroll
    for (int j = 0; j < SR_MAX_ROWS; ++j) w = j == at_line.pick ? wj[j] : w;
    const bool tie = (tie_bits >> at_line.pick) & 1u;
    if (keep.ties_matter) {                              // a tie stays if fewer than the budget came before it
        const unsigned long long ballot = __ballot(tie);
        int rank = __popcll(ballot & ((1ull << lane) - 1ull));
        __syncthreads();
        if (lane == 0) s_n[wave] = __popcll(ballot);
        __syncthreads();
        for (int v = 0; v < wave; ++v) rank += s_n[v];
        if (tie && at_line.seen + rank < keep.tie_budget) w = w_tie;
    }
    float incl = w;
#pragma unroll
    for (int off = 1; off < TM_WAVE; off <<= 1) {
        const float up = __shfl_up(incl, off, TM_WAVE);
        if (lane >= off) incl += up;
    }
    __syncthreads();
    if (lane == TM_WAVE - 1) s_w[wave] = incl;
    __syncthreads();
    float base = at_line.before;
    for (int v = 0; v < wave; ++v) base += s_w[v];
    incl += base;
    // the first entry with mass whose running sum passes the target; else the last entry with mass
    if (w > 0.f) {
        if (target < incl) atomicMin(&s_first, i);
        atomicMax(&s_last, i);
    }
    __syncthreads();
    if (threadIdx.x == 0) out[r] = s_first != 0x7fffffff ? s_first : (s_last >= 0 ? s_last : rowarg[r]);
}

// Bytes of device memory tm_sample_rows needs for R rows of V logits (16-byte aligned start).
static size_t sample_hist_bytes(int R) { return (size_t)R * SR_HIST_PER_ROW * sizeof(unsigned long long); }
extern "C" size_t tm_sample_work_bytes(int R, int V) {
    const size_t NB = (size_t)tm_argmax_work_chunks(V);
    const size_t per_chunk = (size_t)R * NB * 4;         // part_v, part_i, chunk_weight, chunk_ties, wave_v
    return sample_hist_bytes(R) + (size_t)R * sizeof(RowState) + (size_t)R * SR_LIST_ALL * sizeof(uint2) + (4 + AM_NT / TM_WAVE) * per_chunk +
           (size_t)R * (sizeof(RowKeep) + 12);
}

// stages: bit 0 = some row may use top-k, bit 1 = some row may use top-p (3 if the caller does not
// know: rows that use neither skip those launches' work); bit 2 = every row that is not greedy uses a top-k of at most tm_sample_list_k(V): the
// entries go through a list a row (a row that uses none, or more than its shares, is right all the same, worked out by one block: 0.5 to 0.9 ms at 151,936). Calls on one `work` must not overlap.
extern "C" int tm_sample_rows(const float* logits, int R, int V, const float* temperature, const int* top_k,
                              const float* top_p, const float* u, int* out, void* work, size_t work_bytes,
                              int stages, hipStream_t stream) {
    if (R <= 0) return TM_OK;
    if (V <= 0 || !work || ((uintptr_t)work % 16) || work_bytes < tm_sample_work_bytes(R, V)) return TM_ERR_ARG;
    const int NB = tm_argmax_work_chunks(V);
    const int chunk = (V + NB - 1) / NB;
    if (chunk > SR_MAX_ROWS * SR_NT || NB > SR_MAX_CHUNKS) return TM_ERR_ARG;      // more than 2^20 logits a row
    unsigned char* w = (unsigned char*)work;
    unsigned long long* hist = (unsigned long long*)w;
    w += sample_hist_bytes(R);
    RowState* state = (RowState*)w;     w += (size_t)R * sizeof(RowState);
    uint2* lists = (uint2*)w;           w += (size_t)R * SR_LIST_ALL * sizeof(uint2);
    float* part_v = (float*)w;          w += (size_t)R * NB * 4;
    int* part_i = (int*)w;              w += (size_t)R * NB * 4;
    float* wave_v = (float*)w;          w += (size_t)R * NB * (AM_NT / TM_WAVE) * 4;
    float* chunk_weight = (float*)w;    w += (size_t)R * NB * 4;
    int* chunk_ties = (int*)w;          w += (size_t)R * NB * 4;
    RowKeep* row_keep = (RowKeep*)w;    w += (size_t)R * sizeof(RowKeep);
    float* rowmax = (float*)w;          w += (size_t)R * 4;
    int* rowarg = (int*)w;              w += (size_t)R * 4;
    int* counts = (int*)w;
    const dim3 grid(R, NB);
    const bool listed = (stages & 4) && NB > 1;
    argmax_partial_kernel<<<grid, AM_NT, 0, stream>>>(logits, V, chunk, part_v, part_i, listed ? nullptr : hist, SR_HIST_PER_ROW, wave_v);
    TM_CHECK_LAUNCH();
    sample_bound_kernel<<<R, SR_NT, 0, stream>>>(part_v, part_i, wave_v, NB, V, temperature, top_k, top_p, rowmax, rowarg, state, counts);
    TM_CHECK_LAUNCH();
    if (listed) {
        sample_gather_kernel<<<grid, SR_NT, 0, stream>>>(logits, V, chunk, temperature, top_k, top_p, rowmax, wave_v, state, lists, counts, chunk_ties);
        TM_CHECK_LAUNCH();
        sample_select_kernel<<<R, SR_NT, 0, stream>>>(logits, V, chunk, NB, temperature, top_k, top_p, rowmax, wave_v, state, lists, counts, hist,
                                                      chunk_weight, chunk_ties, row_keep);
        TM_CHECK_LAUNCH();
        sample_pick_kernel<<<R, SR_NT, 0, stream>>>(logits, V, chunk, NB, temperature, top_k, top_p, rowmax, rowarg,
                                                    chunk_weight, chunk_ties, row_keep, u, out);
        TM_CHECK_LAUNCH();
        return TM_OK;
    }
    if (stages & 1)
        for (int level = 0; level < 3; ++level) {
            sample_hist_kernel<false><<<grid, SR_NT, 0, stream>>>(logits, V, chunk, temperature, top_k, top_p, rowmax,
                                                                 hist, level, wave_v, state, stages);
            TM_CHECK_LAUNCH();
        }
    if (stages & 2)
        for (int level = 0; level < 3; ++level) {
            sample_hist_kernel<true><<<grid, SR_NT, 0, stream>>>(logits, V, chunk, temperature, top_k, top_p, rowmax,
                                                                hist, level, wave_v, state, stages);
            TM_CHECK_LAUNCH();
        }
    sample_chunk_mass_kernel<<<grid, SR_NT, 0, stream>>>(logits, V, chunk, temperature, top_k, top_p, rowmax, hist,
                                                         chunk_weight, chunk_ties, row_keep, wave_v, state, stages);
    TM_CHECK_LAUNCH();
    sample_pick_kernel<<<R, SR_NT, 0, stream>>>(logits, V, chunk, NB, temperature, top_k, top_p, rowmax, rowarg,
                                                chunk_weight, chunk_ties, row_keep, u, out);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
