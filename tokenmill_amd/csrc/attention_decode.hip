// Paged attention for single decoded tokens on MFMA (bfloat16), split over the context.
//
//   One token per request; its G = H / KVH query heads that share a kv head are the 16 columns of
//   one MFMA tile, so the keys and values of a kv head are read once for all of them
//   (the reference folds the group into query rows the same way: src/infer/model/layers.py:110-124).
//   A wavefront always takes 64 consecutive keys, aligned to a multiple of 64 positions, and gets
//   their unnormalised partial (max, sum, weighted values) in 32-bit. Three ways to cover a context:
//
//   block kernel : one block of 8 (16 for head size 32) wavefronts per (request, kv head); wavefront
//                  w takes keys [64 (i W + w), +64) for i = 0, 1, ...; the partials are merged
//                  through LDS in wavefront order. One launch, no scratch memory: the way for large
//                  batches. Contexts of a few chunks (tm_decode_own_keys) a block takes as the whole kernel does.
//   split kernels: with few requests more blocks than (request, kv head) pairs are needed to pull
//                  the cache at speed: blocks of four wavefronts take chunks of 256 positions and
//                  write partials to scratch memory; a second kernel adds the partials of a request
//                  in ascending chunk order.
//   whole kernel : where contexts are a few chunks long: the split kernels' partials and their order of
//                  additions, in one block per (request, kv head).
//
//   Which keys meet in which partial and in which order partials are added depends on positions
//   only, and the split and the whole kernels have the same bits, so what a request gets does not depend on which other
//   requests are in the batch. It depends on how many there are: from 192 (request, kv head) pairs on, a context beyond
//   tm_decode_own_keys gets the block kernel's order (the two differ by rounding).
//
//   Operand layouts need no LDS: keys K[page][slot][kvh][d] give the A operand of S^T = K Q^T
//   (16 keys x 32 d per instruction), values V[page][kvh][d][slot] give the A operand of
//   O^T = V^T P^T (16 d x 32 keys), and P^T comes straight from the S^T accumulators.
#include "common.h"
#include "api.h"
#include "choose.h"
#include "ahead.h"
#include "attention_decode_keys.h"

// Load, then attend: the partial of 64 keys [wbase, wbase + 64).
template <int D>
__device__ __forceinline__ void wave_keys64(const Bf16x8Bits (&qreg)[D / 32], const bf16_t* __restrict__ k_pool,
                                            const bf16_t* __restrict__ v_pool, const int* __restrict__ table,
                                            int table_width, int wbase, int ctx, int keep, int lo, int kvh, int KVH,
                                            int page_shift, float scale_log2, float cap_in, float cap_out, int r, int g, float& m, float& l,
                                            f32x4_t (&o)[D / 16]) {
    int entry[4];
    load_table_entries(entry, table, table_width, wbase, page_shift);
    Keys64<D> kv;
    load_keys64<D, true>(kv, k_pool, v_pool, entry, wbase, ctx, keep, lo, kvh, KVH, page_shift, r, g);
    attend_keys64<D, true>(kv, qreg, wbase, ctx, keep, lo, scale_log2, cap_in, cap_out, g, m, l, o);
}

// ------------------------------------------------------------------------------------------------
// block kernel: grid (S, KVH), WAVES wavefronts
// ------------------------------------------------------------------------------------------------
template <int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attn_decode_block_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, int out_stride,
    const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool, const int* __restrict__ block_tables,
    int table_width, const int* __restrict__ context_lens, int whole_chunks, int H, int KVH, int page_shift, float scale_log2, float cap_in,
    float cap_out, int window, int keep, const float* __restrict__ sink, const bf16_t* __restrict__ cgate, int ldcg) {
    constexpr int NDT = D / 16;
    extern __shared__ __align__(16) float s_block[];
    const int s = blockIdx.x, kvh = blockIdx.y;
    const int G = H / KVH;
    const int ctx = context_lens[s];
    if (ctx <= whole_chunks * AD_CHUNK)                              // block-uniform
        return attend_whole<D, WAVES, false>(s_block, s, kvh, q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, whole_chunks,
                                      H, KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, sink, cgate, ldcg);
    float(*s_m)[16] = (float(*)[16])s_block, (*s_l)[16] = s_m + WAVES;
    float(*s_o)[16][16 + 1] = (float(*)[16][16 + 1])(s_l + WAVES);   // one 16-wide d tile at a time
    const int p = ctx - 1;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int* table = block_tables + (size_t)s * table_width;

    Bf16x8Bits qreg[D / 32];
    load_q_operand<D>(qreg, q + (size_t)s * q_stride, G, kvh, r, g);

    float m = -INFINITY, l = 0.f;
    f32x4_t o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // runs of 64 aligned positions: those of the kept first keys, then those of the window
    const int kept = lo > 0 ? (keep + AD_WKEYS - 1) / AD_WKEYS : 0;
    const int resume = lo / AD_WKEYS > kept ? lo / AD_WKEYS : kept;
    auto fold = [&](float mi, float li, const f32x4_t (&oi)[NDT]) {  // add a partial to the running one
        const float mn = fmaxf(m, mi);
        const float f0 = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        const float f1 = (mi == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mi - mn);
        l = l * f0 + li * f1;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[dt][i] = o[dt][i] * f0 + oi[dt][i] * f1;
        m = mn;
    };
    for (int run = wave;; run += WAVES) {
        const int wbase = (run < kept ? run : resume + run - kept) * AD_WKEYS;
        if (wbase >= ctx) break;
        float mi, li;
        f32x4_t oi[NDT];
        wave_keys64<D>(qreg, k_pool, v_pool, table, table_width, wbase, ctx, keep, lo, kvh, KVH, page_shift, scale_log2, cap_in, cap_out,
                       r, g, mi, li, oi);
        fold(mi, li, oi);
    }
    // merge the wavefronts in wavefront order; lane: head r, d = 16 dt + 4 g + i
    if (g == 0) {
        s_m[wave][r] = m;
        s_l[wave][r] = l;
    }
    __syncthreads();
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, s_m[w][r]);
    float ll = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        ll += s_l[w][r] * ((s_m[w][r] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(s_m[w][r] - mm));
    const float inv = 1.f / ll;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s_o[wave][r][4 * g + i] = o[dt][i];
        __syncthreads();
        // wavefront dt % WAVES writes this tile: thread -> (head n, 4 consecutive d)
        if (wave == dt % WAVES) {
            const int n = lane / 4, d4 = (lane % 4) * 4;
            if (n < G) {
                float mx = -INFINITY;
#pragma unroll
                for (int w = 0; w < WAVES; ++w) mx = fmaxf(mx, s_m[w][n]);
                float lsum = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < WAVES; ++w) {
                    const float f = (s_m[w][n] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(s_m[w][n] - mx);
                    lsum += s_l[w][n] * f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] += s_o[w][n][d4 + i] * f;
                }
                if (sink) lsum += __builtin_amdgcn_exp2f(sink[kvh * G + n] * 1.4426950408889634f - mx);     // a term of the denominator without a key
                const float iv = 1.f / lsum;
                if (cgate) {                                        // a gate per channel
                    const uint2 gp = *(const uint2*)(cgate + (size_t)s * ldcg + (size_t)(kvh * G + n) * D + 16 * dt + d4);
                    acc[0] *= sigmoid_fast(__uint_as_float(gp.x << 16));
                    acc[1] *= sigmoid_fast(__uint_as_float(gp.x & 0xffff0000u));
                    acc[2] *= sigmoid_fast(__uint_as_float(gp.y << 16));
                    acc[3] *= sigmoid_fast(__uint_as_float(gp.y & 0xffff0000u));
                }
                uint2 pk;
                pk.x = pack_bf16(acc[0] * iv, acc[1] * iv);
                pk.y = pack_bf16(acc[2] * iv, acc[3] * iv);
                *(uint2*)(out + (size_t)s * out_stride + (size_t)(kvh * G + n) * D + 16 * dt + d4) = pk;
            }
        }
        __syncthreads();
    }
    (void)inv;
}

// ------------------------------------------------------------------------------------------------
// split kernels: grid (S, KVH, chunks) with four wavefronts, then the merge
// ------------------------------------------------------------------------------------------------
// The split and the merge kernel begin at multiples of 8 KiB. The same instructions at other places took 796 to 817 us a step (4 requests of 16,000 keys)
// and 715 to 726 (8 of 2,048), and the kernels beside them were the slower ones: what fits is that a layer's kernels share the sets of the instruction
// cache, whose ways are 8 KiB, and drive each other out. Aligned: 796 to 802 and 719 to 721, whatever stands before them in this file.
template <int D, bool AHEAD>
__global__ __attribute__((aligned(8192))) __launch_bounds__(256) void attn_decode_split_kernel(
    const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ v_pool, const int* __restrict__ block_tables, int table_width,
    const int* __restrict__ context_lens, float* __restrict__ part_o, float* __restrict__ part_ml,
    int max_chunks, int H, int KVH, int page_shift, float scale_log2, float cap_in, float cap_out, int window, int keep,
    const TmAhead ahead) {
    constexpr int NDT = D / 16;
    __shared__ float s_m[4][16], s_l[4][16];
    __shared__ float s_o[4][16][D + 1];
    if constexpr (AHEAD) {
        ahead_with(q, q_stride, k_pool, v_pool, block_tables, table_width, context_lens, part_o, part_ml, H, KVH, page_shift, scale_log2, cap_in, cap_out,
                   window, keep);
        if ((int)blockIdx.z >= max_chunks) return tm_bring_ahead(ahead, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), 4);
    }
    const int s = blockIdx.x, kvh = blockIdx.y, chunk = blockIdx.z;
    const int G = H / KVH;
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int chunk_lo = chunk * AD_CHUNK, wbase = chunk_lo + wave * AD_WKEYS;
    // the context length, the block-table entries and the query are asked for together: one trip to
    // memory before the keys, not two
    const int ctx = context_lens[s];
    int entry[4];
    load_table_entries(entry, block_tables + (size_t)s * table_width, table_width, wbase, page_shift);
    Bf16x8Bits qreg[D / 32];
    load_q_operand<D>(qreg, q + (size_t)s * q_stride, G, kvh, r, g);
    const int p = ctx - 1;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    if (chunk_lo >= ctx || (chunk_lo + AD_CHUNK <= lo && chunk_lo >= keep)) return;       // nothing of this chunk is visible
    float m, l;
    f32x4_t o[NDT];
    {
        Keys64<D> kv;
        load_keys64<D, false>(kv, k_pool, v_pool, entry, wbase, ctx, keep, lo, kvh, KVH, page_shift, r, g);
        attend_keys64<D, false>(kv, qreg, wbase, ctx, keep, lo, scale_log2, cap_in, cap_out, g, m, l, o);
    }
    if (g == 0) {
        s_m[wave][r] = m;
        s_l[wave][r] = l;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_o[wave][r][16 * dt + 4 * g + i] = o[dt][i];
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * D; idx += 256) {
        const int n = idx / D, d = idx % D;
        float mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) mm = fmaxf(mm, s_m[w][n]);
        float ll = 0.f, oo = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = (s_m[w][n] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(s_m[w][n] - mm);
            ll += s_l[w][n] * f;
            oo += s_o[w][n][d] * f;
        }
        const size_t slot = ((size_t)s * H + kvh * G + n) * max_chunks + chunk;
        part_o[slot * D + d] = oo;
        if (d == 0) {
            part_ml[slot * 2 + 0] = mm;
            part_ml[slot * 2 + 1] = ll;
        }
    }
}

// out[s, h, :] = the partial values of the visible chunks, weighted and normalised. Four wavefronts
// share a (request, head): wavefront w adds the chunks w, w + 4, ... in ascending order and the four
// sums are added in wavefront order, so the order of additions depends on the context length and
// the window only. A lane holds elements d = lane and lane + 64 of the head.
// For up to 64 chunks: lane c of every wavefront holds (max, sum) of chunk c, and those and the
// values of the first 16 chunks are asked for together with the context length, before it is known
// which of them count (scratch memory beyond the context holds anything: it is dropped by selects,
// never multiplied): one trip to memory for contexts up to 4,096.
#define AD_MERGE_WAVES 4
__attribute__((aligned(8192))) __global__ __launch_bounds__(64 * AD_MERGE_WAVES) void attn_decode_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ context_lens,
    bf16_t* __restrict__ out, int out_stride, int max_chunks, int H, int D, int window, int keep, const float* __restrict__ sink,
    const bf16_t* __restrict__ cgate, int ldcg) {
    __shared__ float s_l[AD_MERGE_WAVES], s_o[AD_MERGE_WAVES][128];
    const int s = blockIdx.x, h = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const size_t base = ((size_t)s * H + h) * max_chunks;
    const int last = max_chunks - 1;
    const int ctx = context_lens[s];
    const f32x2_t ml = *(const f32x2_t*)(part_ml + (base + (lane < last ? lane : last)) * 2);
    const int d0 = lane < D ? lane : D - 1, d1 = lane + 64 < D ? lane + 64 : D - 1;
    float a0[4], a1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = wave + AD_MERGE_WAVES * i;
        const float* src = part_o + (base + (c < last ? c : last)) * D;
        a0[i] = src[d0];
        a1[i] = src[d1];
    }
    const int p = ctx - 1;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int c0 = lo / AD_CHUNK, c1 = (ctx - 1) / AD_CHUNK, ck = (keep + AD_CHUNK - 1) / AD_CHUNK;    // chunks c0 .. c1 and those before ck count
    const float mm = wave_max(((lane >= c0 || lane < ck) && lane <= c1) ? ml[0] : -INFINITY);
    float ll = 0.f, o0 = 0.f, o1 = 0.f;
    auto add_chunk = [&](int c, float v0, float v1) {               // c is the same in every lane
        const float mc = __shfl(ml[0], c, TM_WAVE), lc = __shfl(ml[1], c, TM_WAVE);
        const bool in = (c >= c0 || c < ck) && c <= c1 && mc != -INFINITY;
        const float f = in ? __builtin_amdgcn_exp2f(mc - mm) : 0.f;
        ll = fmaf(in ? lc : 0.f, f, ll);
        o0 = fmaf(in ? v0 : 0.f, f, o0);
        o1 = fmaf(in ? v1 : 0.f, f, o1);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) add_chunk(wave + AD_MERGE_WAVES * i, a0[i], a1[i]);
    // chunks from 16 on (contexts beyond 4,096), four to a wavefront at a time
    for (int cb = 4 * AD_MERGE_WAVES; cb <= c1; cb += 4 * AD_MERGE_WAVES) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = cb + wave + AD_MERGE_WAVES * i;
            const float* src = part_o + (base + (c < last ? c : last)) * D;
            a0[i] = src[d0];
            a1[i] = src[d1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) add_chunk(cb + wave + AD_MERGE_WAVES * i, a0[i], a1[i]);
    }
    if (lane == 0) s_l[wave] = ll;
    s_o[wave][lane] = o0;
    s_o[wave][lane + 64] = o1;
    __syncthreads();
    if (wave != 0) return;
    ll = s_l[0];
    o0 = s_o[0][lane];
    o1 = s_o[0][lane + 64];
#pragma unroll
    for (int w = 1; w < AD_MERGE_WAVES; ++w) {
        ll += s_l[w];
        o0 += s_o[w][lane];
        o1 += s_o[w][lane + 64];
    }
    if (sink) ll += __builtin_amdgcn_exp2f(sink[h] * 1.4426950408889634f - mm);      // a term of the denominator without a key
    bf16_t* orow = out + (size_t)s * out_stride + (size_t)h * D;
    if (cgate) {                                                    // a gate per channel
        const bf16_t* gp = cgate + (size_t)s * ldcg + (size_t)h * D;
        if (lane < D) o0 *= sigmoid_fast(bf16_to_f32(gp[lane]));
        if (lane + 64 < D) o1 *= sigmoid_fast(bf16_to_f32(gp[lane + 64]));
    }
    if (lane < D) orow[lane] = f32_to_bf16(o0 / ll);
    if (lane + 64 < D) orow[lane + 64] = f32_to_bf16(o1 / ll);
}

// The same for any number of chunks (contexts beyond 64 chunks): the maxima are found in a pass of
// their own, and wavefront w adds every fourth of those that count
__global__ __launch_bounds__(64 * AD_MERGE_WAVES) void attn_decode_merge_long_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ context_lens,
    bf16_t* __restrict__ out, int out_stride, int max_chunks, int H, int D, int window, int keep, const float* __restrict__ sink,
    const bf16_t* __restrict__ cgate, int ldcg) {
    __shared__ float s_m[AD_MERGE_WAVES], s_l[AD_MERGE_WAVES], s_o[AD_MERGE_WAVES][128];
    const int s = blockIdx.x, h = blockIdx.y;
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    const int ctx = context_lens[s];
    const int p = ctx - 1;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int c1 = (ctx - 1) / AD_CHUNK;
    // the chunks that count: those of the kept first keys, then those of the window
    const int kept = lo > 0 ? (keep + AD_CHUNK - 1) / AD_CHUNK : 0, resume = lo / AD_CHUNK > kept ? lo / AD_CHUNK : kept;
    const int runs = kept + c1 - resume + 1;
    auto chunk = [&](int i) { return i < kept ? i : resume + i - kept; };
    const size_t base = ((size_t)s * H + h) * max_chunks;
    float mm = -INFINITY;
    for (int i = (int)threadIdx.x; i < runs; i += 64 * AD_MERGE_WAVES) mm = fmaxf(mm, part_ml[(base + chunk(i)) * 2]);
    mm = wave_max(mm);
    if (lane == 0) s_m[wave] = mm;
    __syncthreads();
    mm = s_m[0];
#pragma unroll
    for (int w = 1; w < AD_MERGE_WAVES; ++w) mm = fmaxf(mm, s_m[w]);
    const bool two = lane + 64 < D;
    float ll = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll 4
    for (int i = wave; i < runs; i += AD_MERGE_WAVES) {
        const int c = chunk(i);
        const float mc = part_ml[(base + c) * 2];
        const float lc = part_ml[(base + c) * 2 + 1];
        const float a0 = lane < D ? part_o[(base + c) * D + lane] : 0.f;
        const float a1 = two ? part_o[(base + c) * D + lane + 64] : 0.f;
        const float f = (mc == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mc - mm);
        ll = fmaf(lc, f, ll);
        o0 = fmaf(a0, f, o0);
        o1 = fmaf(a1, f, o1);
    }
    if (lane == 0) s_l[wave] = ll;
    s_o[wave][lane] = o0;
    s_o[wave][lane + 64] = o1;
    __syncthreads();
    if (wave != 0) return;
    ll = s_l[0];
    o0 = s_o[0][lane];
    o1 = s_o[0][lane + 64];
#pragma unroll
    for (int w = 1; w < AD_MERGE_WAVES; ++w) {
        ll += s_l[w];
        o0 += s_o[w][lane];
        o1 += s_o[w][lane + 64];
    }
    if (sink) ll += __builtin_amdgcn_exp2f(sink[h] * 1.4426950408889634f - mm);      // a term of the denominator without a key
    bf16_t* orow = out + (size_t)s * out_stride + (size_t)h * D;
    if (cgate) {                                                    // a gate per channel
        const bf16_t* gp = cgate + (size_t)s * ldcg + (size_t)h * D;
        if (lane < D) o0 *= sigmoid_fast(bf16_to_f32(gp[lane]));
        if (lane + 64 < D) o1 *= sigmoid_fast(bf16_to_f32(gp[lane + 64]));
    }
    if (lane < D) orow[lane] = f32_to_bf16(o0 / ll);
    if (two) orow[lane + 64] = f32_to_bf16(o1 / ll);
}

// ------------------------------------------------------------------------------------------------
// whole kernel: the split kernels' work in one launch, grid (S, KVH), for contexts of a few chunks
// ------------------------------------------------------------------------------------------------
// A block takes all chunks of a (request, kv head): wavefront w the 64 keys of run w, w + WAVES, ...; the partials of the runs
// meet in LDS and are added as the split kernels add them (four runs to a chunk, every fourth chunk to a sum, the four sums in
// order), with the same bits.
//
// Short contexts are bound by the trips to memory that wait for each other, of which the split kernels have two more (partials out and
// in again, behind a launch); against that stands what one CU takes out of the caches, 55 to 60 GB/s whatever is asked for at once,
// where the split kernels use a CU a chunk. Hence one round of loads, as many wavefronts as the context has runs (at most 16, 88
// registers up to head size 64, 8 beyond and where pairs are so many that CUs hold two blocks). The partials meet in two passes of four elements a
// thread: with one element a thread in one pass head size 128 took 1.6 us longer, with four elements in one pass 16 wavefronts spilled.
// The rule and what it measured stand in choose.h (tm_decode_whole).
template <int D, int WAVES, bool AHEAD, bool TURN>
__global__ __launch_bounds__(64 * WAVES) void attn_decode_whole_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, int out_stride,
    const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool, const int* __restrict__ block_tables,
    int table_width, const int* __restrict__ context_lens, int chunks, int H, int KVH, int page_shift, float scale_log2,
    float cap_in, float cap_out, int window, int keep, const float* __restrict__ sink, const bf16_t* __restrict__ cgate, int ldcg,
    const TmAhead ahead) {
    extern __shared__ __align__(16) float s_whole[];
    if constexpr (AHEAD) {
        ahead_with(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, chunks, H, KVH, page_shift, scale_log2, cap_in,
                   cap_out, window, keep, sink, cgate, ldcg);
        if (blockIdx.z) return tm_bring_ahead(ahead, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), WAVES);
    }
    attend_whole<D, WAVES, TURN>(s_whole, blockIdx.x, blockIdx.y, q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, chunks, H,
                           KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, sink, cgate, ldcg);
}

// Layers of `pairs` blocks of a grid that has `own` of them, with those that bring matrices ahead.
static int ahead_layers(TmAhead& ahead, int pairs, int own) {
    const int more = ahead.n ? (ahead.blocks + pairs - 1) / pairs : 0;
    if (own + more > 65535) {                                       // (no room in the grid)
        ahead.n = 0;
        return own;
    }
    ahead.first = pairs * own;
    ahead.blocks = pairs * more;
    return own + more;
}

template <int D, int WAVES, bool AHEAD, bool TURN>
static int launch_whole(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                        const int* block_tables, int table_width, const int* context_lens, int chunks, int S, int H, int KVH,
                        int page_shift, float scale_log2, float cap_in, float cap_out, int window, int keep, const float* sink,
                        const bf16_t* cgate, int ldcg, TmAhead& ahead, hipStream_t stream) {
    static const hipError_t allowed = hipFuncSetAttribute((const void*)attn_decode_whole_kernel<D, WAVES, AHEAD, TURN>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)TM_DECODE_WHOLE_LDS);
    if (allowed != hipSuccess) return TM_ERR_LAUNCH;
    attn_decode_whole_kernel<D, WAVES, AHEAD, TURN><<<dim3(S, KVH, ahead_layers(ahead, S * KVH, 1)), 64 * WAVES, tm_decode_whole_lds(chunks, H / KVH, D), stream>>>(
        (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, (const bf16_t*)k_pool, (const bf16_t*)v_pool, block_tables,
        table_width, context_lens, chunks, H, KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, sink, cgate, ldcg, ahead);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

template <int D>
static int launch_decode(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                         const void* v_pool, const int* block_tables, int table_width, const int* context_lens,
                         float* part_o, float* part_ml, int max_chunks, int S, int H, int KVH, int page,
                         float scale, int window, int keep, float softcap, const float* sink, const bf16_t* cgate, int ldcg,
                         TmAhead& ahead, hipStream_t stream) {
    int page_shift = 0;
    while ((1 << page_shift) < page) ++page_shift;
    const float scale_log2 = scale * 1.4426950408889634f;
    const float cap_in = softcap > 0.f ? scale / softcap : 0.f, cap_out = softcap * 1.4426950408889634f;
    constexpr int WAVES = D <= 32 ? 16 : 8;       // 16 wavefronts leave 128 registers each: enough for D = 32 only
    // few (request, kv head) pairs: more blocks than pairs are needed to pull the cache at speed; the caller
    // asks for that by bringing the scratch memory
    const bool split = part_o && part_ml && max_chunks > 1;
    if (!split) {
        const int own = tm_decode_own_keys(H / KVH, D) / AD_CHUNK, whole_chunks = own < max_chunks ? own : max_chunks;
        const size_t block = (size_t)WAVES * 16 * (2 + 17) * sizeof(float), whole = tm_decode_whole_lds(whole_chunks, H / KVH, D);
        static const hipError_t allowed = hipFuncSetAttribute((const void*)attn_decode_block_kernel<D, WAVES>,
                                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)TM_DECODE_WHOLE_LDS);
        if (allowed != hipSuccess) return TM_ERR_LAUNCH;
        attn_decode_block_kernel<D, WAVES><<<dim3(S, KVH), 64 * WAVES, block > whole ? block : whole, stream>>>(
            (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, (const bf16_t*)k_pool, (const bf16_t*)v_pool,
            block_tables, table_width, context_lens, whole_chunks, H, KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, sink,
            cgate, ldcg);
        TM_CHECK_LAUNCH();
        return TM_OK;
    }
    const dim3 grid(S, KVH, ahead_layers(ahead, S * KVH, max_chunks));
    (ahead.n ? attn_decode_split_kernel<D, true> : attn_decode_split_kernel<D, false>)<<<grid, 256, 0, stream>>>(
        (const bf16_t*)q, q_stride, (const bf16_t*)k_pool, (const bf16_t*)v_pool, block_tables, table_width,
        context_lens, part_o, part_ml, max_chunks, H, KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, ahead);
    TM_CHECK_LAUNCH();
    if (max_chunks <= TM_WAVE)
        attn_decode_merge_kernel<<<dim3(S, H), 64 * AD_MERGE_WAVES, 0, stream>>>(
            part_o, part_ml, context_lens, (bf16_t*)out, out_stride, max_chunks, H, D, window, keep, sink, cgate, ldcg);
    else
        attn_decode_merge_long_kernel<<<dim3(S, H), 64 * AD_MERGE_WAVES, 0, stream>>>(
            part_o, part_ml, context_lens, (bf16_t*)out, out_stride, max_chunks, H, D, window, keep, sink, cgate, ldcg);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

bool decode_args_ok(const void* q, int q_stride, const void* out, int out_stride, int table_width, int max_chunks, int H, int KVH, int D,
                           int page, float scale, int window, int keep, float softcap, const void* cgate, int ldcg) {
    if (!(softcap >= 0.f) || keep < 0 || (cgate && (ldcg < H * D || ldcg % 4 || (uintptr_t)cgate % 8))) return false;
    return !(H <= 0 || KVH <= 0 || H % KVH || H / KVH > 16 || page < 16 || (page & (page - 1)) || max_chunks <= 0 ||
             !(scale > 0.f) || max_chunks > 65535 || KVH > 65535 || window < 0 || table_width <= 0 || (q_stride % 8) ||
             ((uintptr_t)q % 16) || (out_stride % 4) || ((uintptr_t)out % 8) || q_stride < H * D || out_stride < H * D);
}

// q: first decode row (one row per request, rows q_stride apart); out likewise; block_tables and
// context_lens: first decode request. part_o: float [S, H, max_chunks, D] and part_ml: [S, H, max_chunks, 2]
// are scratch for the split kernels, which run when both are given (the caller gives them when the
// (request, kv head) pairs alone are too few blocks for the chip); without them the block kernel runs.
// softcap > 0: a score s (scaled) becomes softcap * tanh(s / softcap) before the softmax; sink (float32 [H]) or null: one more term
// exp(sink[h]) in the denominator of head h's softmax, with no key behind it (added once, where a request's partials meet); with a window, `keep`: the first
// keys of a request that every token sees beside its window; cgate (rows ldcg apart, a row a request) or null: channel c of the result is
// multiplied by sigmoid(cgate[c]).
int attn_decode_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                       const void* v_pool, const int* block_tables, int table_width,
                                       const int* context_lens, float* part_o, float* part_ml, int max_chunks, int S,
                                       int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                       const float* sink, const void* cgate, int ldcg, TmAhead ahead, hipStream_t stream) {
    if (S <= 0) return TM_OK;
    if (!decode_args_ok(q, q_stride, out, out_stride, table_width, max_chunks, H, KVH, D, page, scale, window, keep, softcap, cgate, ldcg)) return TM_ERR_ARG;
    if (window == 0) keep = 0;
#define TM_DECODE_CASE(DD)                                                                                        \
    case DD:                                                                                                      \
        return launch_decode<DD>(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width,         \
                                 context_lens, part_o, part_ml, max_chunks, S, H, KVH, page, scale, window, keep, softcap, sink,  \
                                 (const bf16_t*)cgate, ldcg, ahead, stream)
    switch (D) {
        TM_DECODE_CASE(32);
        TM_DECODE_CASE(64);
        TM_DECODE_CASE(96);
        TM_DECODE_CASE(128);
        default:
            return TM_ERR_ARG;
    }
#undef TM_DECODE_CASE
}

extern "C" int tm_attn_decode_mfma_cap(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                       const void* v_pool, const int* block_tables, int table_width,
                                       const int* context_lens, float* part_o, float* part_ml, int max_chunks, int S,
                                       int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                       const float* sink, const void* cgate, int ldcg, hipStream_t stream) {
    return attn_decode_ahead(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, part_o, part_ml, max_chunks, S, H,
                             KVH, D, page, scale, window, keep, softcap, sink, cgate, ldcg, TmAhead{}, stream);
}

// The same by the whole kernel, for contexts of at most max_chunks chunks that its LDS holds (tm_decode_whole in choose.h says where it is
// the better one). No scratch memory; the bits of the split kernels.
template <int D>
static int launch_whole_waves(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                              const int* block_tables, int table_width, const int* context_lens, int chunks, int S, int H, int KVH, int page,
                              float scale, int window, int keep, float softcap, const float* sink, const bf16_t* cgate, int ldcg, TmAhead& ahead, hipStream_t stream) {
    int page_shift = 0;
    while ((1 << page_shift) < page) ++page_shift;
    const float cap_in = softcap > 0.f ? scale / softcap : 0.f;
#define TM_WHOLE(W, TURN)                                                                                                        \
    (ahead.n ? launch_whole<D, W, true, TURN> : launch_whole<D, W, false, TURN>)(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, chunks, S, H, KVH, \
                       page_shift, scale * 1.4426950408889634f, cap_in, softcap * 1.4426950408889634f, window, keep, sink, cgate, ldcg, ahead, stream)
    if constexpr (D > 64) {
        if (chunks > 1) return TM_WHOLE(8, true);           // (12 and 16 wavefronts do not have the registers)
        return tm_decode_whole_turns(D, chunks, S * KVH) ? TM_WHOLE(4, true) : TM_WHOLE(4, false);
    } else {
        constexpr bool turn = tm_decode_whole_turns(D, 2, 1);
        if (chunks == 1) return TM_WHOLE(4, false);
        return chunks == 2 || S * KVH > 256 ? TM_WHOLE(8, turn) : chunks == 3 ? TM_WHOLE(12, turn) : TM_WHOLE(16, turn);
    }
#undef TM_WHOLE
}

int attn_decode_whole_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                                    const int* block_tables, int table_width, const int* context_lens, int max_chunks, int S, int H, int KVH,
                                    int D, int page, float scale, int window, int keep, float softcap, const float* sink, const void* cgate,
                                    int ldcg, TmAhead ahead, hipStream_t stream) {
    if (S <= 0) return TM_OK;
    if (!decode_args_ok(q, q_stride, out, out_stride, table_width, max_chunks, H, KVH, D, page, scale, window, keep, softcap, cgate, ldcg) ||
        tm_decode_whole_lds(max_chunks, H / KVH, D) > TM_DECODE_WHOLE_LDS)
        return TM_ERR_ARG;
    if (window == 0) keep = 0;
#define TM_WHOLE_CASE(DD)                                                                                                                  \
    case DD:                                                                                                                               \
        return launch_whole_waves<DD>(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, max_chunks,  \
                                      S, H, KVH, page, scale, window, keep, softcap, sink, (const bf16_t*)cgate, ldcg, ahead, stream)
    switch (D) {
        TM_WHOLE_CASE(32);
        TM_WHOLE_CASE(64);
        TM_WHOLE_CASE(96);
        TM_WHOLE_CASE(128);
        default:
            return TM_ERR_ARG;
    }
#undef TM_WHOLE_CASE
}

extern "C" int tm_attn_decode_whole(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                                    const int* block_tables, int table_width, const int* context_lens, int max_chunks, int S, int H, int KVH,
                                    int D, int page, float scale, int window, int keep, float softcap, const float* sink, const void* cgate,
                                    int ldcg, hipStream_t stream) {
    return attn_decode_whole_ahead(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, max_chunks, S, H, KVH, D, page,
                                   scale, window, keep, softcap, sink, cgate, ldcg, TmAhead{}, stream);
}

extern "C" int tm_attn_decode_mfma(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                   const void* v_pool, const int* block_tables, int table_width,
                                   const int* context_lens, float* part_o, float* part_ml, int max_chunks, int S,
                                   int H, int KVH, int D, int page, float scale, int window, hipStream_t stream) {
    return tm_attn_decode_mfma_cap(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, context_lens, part_o, part_ml,
                                   max_chunks, S, H, KVH, D, page, scale, window, 0, 0.f, nullptr, nullptr, 0, stream);
}
