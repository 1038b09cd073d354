// What the kernels that attend single decoded tokens share (attention_decode.hip, and the kernel of prompt portions that has them beside it): the
// partial of 64 keys, and a whole context by one block.
#pragma once
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

#define AD_CHUNK 256        // keys per block
#define AD_WKEYS 64         // keys per wavefront

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// two floats -> packed bfloat16 (round to nearest even, one instruction on gfx950)
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const bf16x2_t v = __builtin_convertvector(f32x2_t{a, b}, bf16x2_t);
    return *(const uint32_t*)&v;
}

union Bf16x8Bits {
    u32x4_t u;
    bf16x8_t b;
};

// The keys and values of 64 positions [wbase, wbase + 64) of one kv head as a wavefront holds them
// between asking for them and using them: four tiles of 16 keys as MFMA operands.
//
// Which 16 keys make a tile is chosen for the loads of the values. A lane of the second product needs, for
// 32 keys at a time, 8 keys of one row d of V^T, and it must be the 8 keys whose probabilities the lane got
// from the first product's accumulators: 4 from each tile of a pair. With tiles of consecutive keys those are
// 4 + 4 keys 16 apart: two 8-byte loads, and an instruction of the wavefront touches 32 bytes of each of 16
// rows, which reads the pool at 3.9 TB/s at best. So the tiles of a pair (2b, 2b + 1) split their 32 keys in
// runs of four: row rho of tile t is key 32 (t / 2) + 8 (rho / 4) + 4 (t % 2) + rho % 4. The lane that holds
// rows 4g..4g+3 of both tiles then has the keys 32b + 8g .. + 7: one 16-byte load, 64 bytes of a row an
// instruction (4.7 TB/s), and half as many loads. The keys are whole rows of the pool either way.
//
// Neighbouring lanes of the first product's operand are in different rows: 64 addresses for a CU's address unit, one a cycle, where four lanes
// beside each other in a row are one. TURN: four lanes load 64 bytes of a row (lane (4 q + p, g) row 4 q + g, piece p) and the pieces change
// lanes in front of the product by ds_bpermute, four a load, which a wavefront waits for. So it pays where a CU has many keys to load: in the kernel of a whole
// context with more than one chunk and more than 32 channels a head, with one chunk of more than 64 channels and fewer than 128 pairs. us without / with: 1 request of
// two heads, D 64 of 300 / 600 / 1,100 keys 5.6 / 5.2, 7.3 / 6.4, 10.3 / 8.5, D 128 of 200 / 600 6.6 / 5.9, 11.1 / 9.2, 32 requests, D 64 of 320 / 768 6.5 / 6.1, 8.9 / 8.2; 64,
// of 600 9.0 / 8.7. Where it does not: D 64 of 64 / 128 / 200 keys, 1 request 4.4 / 4.6, 4.5 / 4.7, 4.9 / 4.9; D 32, of 128 / 512 keys 1 and 64 requests
// 4.2 / 4.3, 5.0 / 4.9, 5.0 / 5.0, 6.0 / 6.0; D 128, 64 and 90 requests of 256 keys 8.4 / 8.6, 8.8 / 9.1. The block kernel takes its requests beyond the
// whole kernel's order so (200 of 2,500 keys, D 64 56.2 / 53.4, D 96 and D 128 100 of 40 heads over 8 171 / 168, 217 / 204) and those of the whole kernel's order without (128 and 200 of 200
// keys, D 128 9.4 / 9.9, 15.5 / 16.1). The split kernel, whose wavefronts have 64 keys and no more, has the exchange in its one chain: 8 of 2,048, D 128, 12.7 / 13.1, 64
// level. It goes without. The same bits.
constexpr bool tm_decode_whole_turns(int D, int chunks, int pairs) { return D > 32 && (chunks > 1 || (D > 64 && pairs < 128)); }
__device__ __forceinline__ int tile_key(int t, int rho) { return 32 * (t / 2) + 8 * (rho / 4) + 4 * (t % 2) + rho % 4; }

template <int D>
struct Keys64 {
    int group_page[4];                      // page of the 16 positions [wbase + 16 q, + 16), -1 if no query may see them (wave-uniform)
    Bf16x8Bits k[4][D / 32];                // [tile][32 d], rows and pieces as loaded
    u32x4_t v[D / 16][2];                   // [16 d][32 keys]: keys 32 b + 8 g .. + 7 of row d = 16 dt + r
};

// The block-table entries of the four 16-key tiles of [wbase, wbase + 64), read without a test at an
// index inside the row (what lies beyond the context is dropped by load_keys64): they depend on
// nothing but the request, so a kernel can ask for them before it knows the context length.
__device__ __forceinline__ void load_table_entries(int (&entry)[4], const int* __restrict__ table, int table_width,
                                                   int wbase, int page_shift) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int at = (wbase + 16 * t) >> page_shift;
        entry[t] = table[at < table_width ? at : table_width - 1];
    }
}

// Ask for the keys and values of [wbase, wbase + 64): every load is issued, nothing is waited for.
template <int D, bool TURN>
__device__ __forceinline__ void load_keys64(Keys64<D>& kv, const bf16_t* __restrict__ k_pool,
                                            const bf16_t* __restrict__ v_pool, const int (&entry)[4], int wbase,
                                            int ctx, int keep, int lo, int kvh, int KVH, int page_shift, int r, int g) {
    constexpr int NDC = D / 32, NDT = D / 16;
    const int page_mask = (1 << page_shift) - 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int first = wbase + 16 * q;
        kv.group_page[q] = (first < ctx && (first + 16 > lo || first < keep)) ? entry[q] : -1;                        // wave-uniform
    }
    // Every load is unconditional, so that none of them has to be waited for before the next is
    // issued: positions nobody may see read page 0 instead, and keys beyond the context read the rest of
    // their page. What such loads bring is never used: their scores are replaced by -inf and their
    // values are masked bit by bit.
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        // the 16 positions of a row's key: the pair's first 16 for rows 0..7, its second 16 for rows 8..15
        const int row = TURN ? 4 * (r / 4) + g : r, piece = TURN ? r % 4 : g, key = wbase + tile_key(t, row);
        const int page = row < 8 ? kv.group_page[2 * (t / 2)] : kv.group_page[2 * (t / 2) + 1];
        const size_t pg = page >= 0 ? (size_t)page : 0;
        const bf16_t* kr = k_pool + (((pg << page_shift) + (key & page_mask)) * KVH + kvh) * D + 8 * piece;
#pragma unroll
        for (int c = 0; c < NDC; ++c) kv.k[t][c].u = *(const u32x4_t*)(kr + 32 * c);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int key = wbase + 32 * b + 8 * g;                      // this lane's 8 keys of the pair
        const int page = g < 2 ? kv.group_page[2 * b] : kv.group_page[2 * b + 1];
        const size_t pg = page >= 0 ? (size_t)page : 0;
        const bf16_t* vr = v_pool + (((pg * KVH + kvh) * D + r) << page_shift) + (key & page_mask);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) kv.v[dt][b] = *(const u32x4_t*)(vr + ((size_t)(16 * dt) << page_shift));
    }
    // nothing that uses the keys may be scheduled above the loads of the values: both are on their
    // way before the first wait
    __builtin_amdgcn_sched_barrier(0);
}

// The partial of the 64 keys in kv for the (up to 16) query heads of one kv head.
// m is in units of score * scale * log2(e).
template <int D, bool TURN>
__device__ __forceinline__ void attend_keys64(const Keys64<D>& kv, const Bf16x8Bits (&qreg)[D / 32], int wbase, int ctx,
                                              int keep, int lo, float scale_log2, float cap_in, float cap_out, int g, float& m, float& l,
                                              f32x4_t (&o)[D / 16]) {
    constexpr int NDC = D / 32, NDT = D / 16;
    float sc[4][4];                                                 // [tile][row 4g+i of the tile] for head r
    const int r = threadIdx.x % 16, from = 4 * (16 * (r % 4) + 4 * (r / 4) + g);       // the lane, in bytes, that has row r's piece g
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NDC; ++c) {
            Bf16x8Bits kf = kv.k[t][c];
            if constexpr (TURN) {
#pragma unroll
                for (int e = 0; e < 4; ++e) kf.u[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)kf.u[e]);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.b, qreg[c].b, acc, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kj = wbase + tile_key(t, 4 * g + i);
            // cap_in > 0: capped scores, cap * tanh(score * scale / cap), in units of log2 like the plain ones
            const float sv = cap_in > 0.f ? cap_out * tanh_fast(acc[i] * cap_in) : acc[i] * scale_log2;
            sc[t][i] = (kj < ctx && (kj >= lo || kj < keep)) ? sv : -INFINITY;
        }
    }
    m = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) m = fmaxf(m, sc[t][i]);
    m = lane_max<16>(m);
    m = lane_max<32>(m);
    const float neg_m = (m == -INFINITY) ? 0.f : -m;
    l = 0.f;
    float pr[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            pr[t][i] = __builtin_amdgcn_exp2f(sc[t][i] + neg_m);
            l += pr[t][i];
        }
    l = lane_sum<16>(l);
    l = lane_sum<32>(l);
    // O^T[d][head] = V^T[d][keys] P^T[keys][head], 32 keys (tiles 2b, 2b+1) per instruction
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        Bf16x8Bits pt;
        pt.u = u32x4_t{pack_bf16(pr[2 * b][0], pr[2 * b][1]), pack_bf16(pr[2 * b][2], pr[2 * b][3]),
                       pack_bf16(pr[2 * b + 1][0], pr[2 * b + 1][1]), pack_bf16(pr[2 * b + 1][2], pr[2 * b + 1][3])};
        // which of this lane's 8 keys exist (a value beyond the context may hold anything)
        uint32_t mask[4];
#pragma unroll
        for (int w2 = 0; w2 < 4; ++w2) {
            const int ka = wbase + 32 * b + 8 * g + 2 * w2, kb = ka + 1;
            mask[w2] = ((ka < ctx && (ka >= lo || ka < keep)) ? 0x0000ffffu : 0u) | ((kb < ctx && (kb >= lo || kb < keep)) ? 0xffff0000u : 0u);
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            Bf16x8Bits vf;
            vf.u = u32x4_t{kv.v[dt][b][0] & mask[0], kv.v[dt][b][1] & mask[1], kv.v[dt][b][2] & mask[2],
                           kv.v[dt][b][3] & mask[3]};
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.b, pt.b, o[dt], 0, 0, 0);
        }
    }
}

template <int D>
__device__ __forceinline__ void load_q_operand(Bf16x8Bits (&qreg)[D / 32], const bf16_t* __restrict__ q, int G,
                                               int kvh, int r, int g) {
    // Q^T operand: column r = query head kvh*G + r, rows d = 32c + 8g .. +7
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
        if (r < G)
            qreg[c].u = *(const u32x4_t*)(q + (size_t)(kvh * G + r) * D + 32 * c + 8 * g);
        else
            qreg[c].u = u32x4_t{0, 0, 0, 0};
    }
}

// All chunks of a (request, kv head) by one block of WAVES wavefronts (the whole kernel of attention_decode.hip); lds: tm_decode_whole_lds bytes, 16 byte aligned.
template <int D, int WAVES, bool TURN>
__device__ __forceinline__ void attend_whole(float* lds, int s, int kvh, const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out,
                                             int out_stride, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool,
                                             const int* __restrict__ block_tables, int table_width, const int* __restrict__ context_lens, int chunks,
                                             int H, int KVH, int page_shift, float scale_log2, float cap_in, float cap_out, int window, int keep,
                                             const float* __restrict__ sink, const bf16_t* __restrict__ cgate, int ldcg) {
    constexpr int NDT = D / 16, ROW = D + 4;
    const int G = H / KVH;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int runs = 4 * chunks;
    f32x2_t* s_ml = (f32x2_t*)lds;                                   // [runs][16]: maximum and sum
    f32x2_t* s_chunk = s_ml + runs * 16;                             // [chunks][16]: the same of a chunk
    float* s_o = (float*)(s_chunk + chunks * 16);                    // [runs][G][ROW]
    const int* table = block_tables + (size_t)s * table_width;
    const int ctx = context_lens[s];
    int entry[4];
    load_table_entries(entry, table, table_width, wave * AD_WKEYS, page_shift);
    Bf16x8Bits qreg[D / 32];
    load_q_operand<D>(qreg, q + (size_t)s * q_stride, G, kvh, r, g);
    const int p = ctx - 1;
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    for (int run = wave; run < runs; run += WAVES) {
        const int wbase = run * AD_WKEYS;
        float m = -INFINITY, l = 0.f;
        if (wbase < ctx && (wbase + AD_WKEYS > lo || wbase < keep)) {       // else nothing of the run is visible
            f32x4_t o[NDT];
            Keys64<D> kv;
            load_keys64<D, TURN>(kv, k_pool, v_pool, entry, wbase, ctx, keep, lo, kvh, KVH, page_shift, r, g);
            attend_keys64<D, TURN>(kv, qreg, wbase, ctx, keep, lo, scale_log2, cap_in, cap_out, g, m, l, o);
            if (r < G) {
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) *(f32x4_t*)(s_o + ((size_t)run * G + r) * ROW + 16 * dt + 4 * g) = o[dt];
            }
        }
        if (g == 0) s_ml[run * 16 + r] = f32x2_t{m, l};
        if (run + WAVES < runs) load_table_entries(entry, table, table_width, wbase + WAVES * AD_WKEYS, page_shift);
    }
    __syncthreads();
    const int c1 = ctx <= chunks * AD_CHUNK ? (ctx - 1) / AD_CHUNK : chunks - 1;      // the last chunk that counts
    // the runs of a chunk, four elements of a head a thread (what a chunk has takes the place of its first run's)
    constexpr int PIECES = D / 4;
    for (int idx = threadIdx.x; idx < (c1 + 1) * G * PIECES; idx += 64 * WAVES) {
        const int cn = idx / PIECES, d = idx % PIECES * 4, c = cn / G, n = cn - c * G;
        f32x2_t ml[4];
        f32x4_t v[4], oc = {0.f, 0.f, 0.f, 0.f};
        float* at = s_o + ((size_t)4 * c * G + n) * ROW + d;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            ml[w] = s_ml[(4 * c + w) * 16 + n];
            v[w] = *(const f32x4_t*)(at + (size_t)w * G * ROW);
        }
        float mc = -INFINITY, lc = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) mc = fmaxf(mc, ml[w][0]);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const bool in = ml[w][0] != -INFINITY;                   // (nothing was stored where nothing is visible)
            const float f = in ? __builtin_amdgcn_exp2f(ml[w][0] - mc) : 0.f;
            lc = fmaf(ml[w][1], f, lc);
#pragma unroll
            for (int i = 0; i < 4; ++i) oc[i] = fmaf(in ? v[w][i] : 0.f, f, oc[i]);
        }
        *(f32x4_t*)at = oc;
        if (d == 0) s_chunk[c * 16 + n] = f32x2_t{mc, lc};
    }
    __syncthreads();
    // the chunks
    for (int idx = threadIdx.x; idx < G * PIECES; idx += 64 * WAVES) {
        const int n = idx / PIECES, d = idx % PIECES * 4;
        float mm = -INFINITY;
        for (int c = 0; c <= c1; ++c) mm = fmaxf(mm, s_chunk[c * 16 + n][0]);
        float ll[4] = {0.f, 0.f, 0.f, 0.f};
        f32x4_t oo[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) oo[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int cb = 0; cb <= c1; cb += 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = cb + j < c1 ? cb + j : c1;
                const f32x2_t ml = s_chunk[c * 16 + n];
                const f32x4_t oc = *(const f32x4_t*)(s_o + ((size_t)4 * c * G + n) * ROW + d);
                const float f = cb + j > c1 || ml[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[0] - mm);
                ll[j] = fmaf(ml[1], f, ll[j]);
#pragma unroll
                for (int i = 0; i < 4; ++i) oo[j][i] = fmaf(oc[i], f, oo[j][i]);
            }
        }
        float lsum = ll[0];
        f32x4_t osum = oo[0];
#pragma unroll
        for (int j = 1; j < 4; ++j) {
            lsum += ll[j];
            osum += oo[j];
        }
        if (sink) lsum += __builtin_amdgcn_exp2f(sink[kvh * G + n] * 1.4426950408889634f - mm);     // a term of the denominator without a key
        const size_t at = (size_t)(kvh * G + n) * D + d;
        if (cgate) {                                                 // a gate per channel
            const uint2 gp = *(const uint2*)(cgate + (size_t)s * ldcg + at);
            osum[0] *= sigmoid_fast(__uint_as_float(gp.x << 16));
            osum[1] *= sigmoid_fast(__uint_as_float(gp.x & 0xffff0000u));
            osum[2] *= sigmoid_fast(__uint_as_float(gp.y << 16));
            osum[3] *= sigmoid_fast(__uint_as_float(gp.y & 0xffff0000u));
        }
        *(uint2*)(out + (size_t)s * out_stride + at) = uint2{pack_bf16(osum[0] / lsum, osum[1] / lsum), pack_bf16(osum[2] / lsum, osum[3] / lsum)};
    }
}
