// Paged attention for portions of prompts in true 32-bit, flash style on the 32-bit MFMA
// (v_mfma_f32_16x16x4_f32: 32-bit inputs, 32-bit products and sums; no reduced-precision mode).
//
//   A block takes 16 consecutive query tokens of one request (a "tile") and one query head. The keys
//   the tile may see are cut into blocks of 16 at absolute positions; the block's four wavefronts take
//   every fourth key block each (key block kb goes to wavefront kb % 4), in ascending position with an
//   online softmax of their own, and their four partial results are merged through LDS in the order of
//   the wavefronts: a query at position p sees keys lo..p, lo = 0 or p - window + 1, and with a window also the first `keep`
//                               (reference src/infer/kv/context.py:70-75, src/infer/model/layers.py:100-107).
//   Which wavefront takes a key block hangs on the key's position only, so a token's result depends
//   on its request only. The longest tile of a 2,048-token prompt walks 32 key blocks a wavefront
//   instead of 128; the heads of a kv head run in blocks of their own and share its keys through the
//   second-level cache (two heads a wavefront were no faster).
//   The matrix instructions of a 1,000-token prompt of the 0.5B shape (14 heads of 64) take 12 us a layer. What stood beside them: the newest
//   tiles' blocks met on the same CUs (52 us; 38 dealt out as below), accumulators that the vector unit had to fetch back and a
//   branch for a cap (35), and sums rescaled at every block, expf, loads without a scalar base (30). The next block's keys and
//   values are on their way while a block is multiplied (but in short windows).
//
//   S^T = K Q^T   A = keys  [16 keys x 4 d]   B = Q^T [4 d x 16 tokens]   (D / 4 steps; which d a step
//                 multiplies is free as long as keys and queries agree: the lanes of group g = lane / 16
//                 hold d = 16 c + 4 g .. + 3 for c = 0 .. D/16 - 1 of their key / token, so one 16-byte
//                 load of the four groups of a key is one run of 64 bytes)
//   O^T = V^T P^T A = V^T   [16 d x 4 keys]   B = P^T [4 keys x 16 tokens]: in step i the lanes of
//                 group g hold key 4 g + i, which is where the S^T accumulators already have it
//                 (register i of the same lane) and what one 16-byte load of V[d][4 g .. 4 g + 3] gives.
#include "common.h"
#include "api.h"
#include "fused_common.h"

#define AF_SPLIT 4          // wavefronts of a block; each takes every fourth key block
// Keys a token sees at most where a wavefront's walk is two or three blocks: the block ahead is one that nobody wants then, and without its
// registers a CU holds more blocks (14 heads of 64, a window of 64 / 128, 1,000 tokens, with it 12.2 / 14.9 us, without 10.5 / 13.1; 3,000
// 25.9 / 33.4 and 22.9 / 29.9; at 256 keys 44.9 with it)
#define AF_SHORT_WALK 128
// TURN: neighbouring lanes of the operands are in different rows, 64 addresses for a CU's address unit, one a clock, and four wavefronts
// ask for twice what it can take while they multiply. So four lanes load 64 bytes of a row (lane (4 q + p, g) row 4 q + g, piece p) and the
// pieces change lanes by ds_bpermute, four a load. us without / with: 28 heads over 4 of 128, 300 / 512 / 1,000 tokens 18.7 / 18.0, 38.2 / 35.4, 103 / 94;
// 12 over 2 of 96, 800 / 1,500 26.5 / 25.2, 74.6 / 63.4; 14 over 2 of 64, 1,000 / 1,500 / 3,000 31.3 / 28.5, 59.7 / 54.3, 189 / 173. A launch of few blocks or of small heads
// waits for the exchange instead: 14 of 64, 600 / 800 tokens 15.4 / 16.6, 22.0 / 22.0, 8 over 8 of 64, 1,000 20.3 / 22.5, 5 of 80, 2,500 59.8 / 63.0, 8 over 2
// of 32, 3,000 56.4 / 55.9, 12 over 2 of 96, 300 10.9 / 11.8, 9 over 3 of 112, 1,500 56 / 60: head size 64 takes it from three blocks a CU, 96 and 128 from
// two. The same bits.
constexpr bool AF_TURNS(int D) { return D == 64 || D == 96 || D == 128; }
constexpr int AF_TURN_BLOCKS(int D) { return D == 64 ? 768 : 512; }
#define AF_ROUND 256        // blocks that come to rest on CUs of their own before the first CU gets a second one

// A column's reference moves only when its maximum has grown by more than this (weights up to e^8 cost 32-bit sums nothing), so
// most blocks rescale no sums.
#define AF_GROWTH 8.f

// e^x for x <= AF_GROWTH, -inf (a key not to be seen) and what is no number: two to the fraction of x log2(e), which one fused operation
// leaves exact and a second one corrects by what the 32-bit log2(e) lacks, times two to its whole part. Off 64 bits by 0.44 units of
// 2^-24 (root mean square; 1.4 at most) throughout, as expf is, without its look after overflow.
__device__ __forceinline__ float exp_weight(float x) {
    const float whole = __builtin_rintf(x * 1.44269504f);
    const float part = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, 1.44269504f, -whole));
    return x < -104.f ? 0.f : __builtin_ldexpf(__builtin_amdgcn_exp2f(part), (int)whole);
}

// What a wavefront loads of a block of 16 keys. AHEAD (below): the next block's are on their way while a block is multiplied.
template <int D>
struct KVBlock32 {
    f32x4_t k[D / 16], v[D / 16];
};

template <int D, bool CAP, bool AHEAD, bool TURN>
__global__ __launch_bounds__(64 * AF_SPLIT, AHEAD ? 2 : 1) void attn_prefill_f32_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
    const float* __restrict__ k_pool, const float* __restrict__ v_pool, const int* __restrict__ block_tables,
    int table_width, const int* __restrict__ tiles, int H, int KVH, int page_shift, float scale, int window, int keep, float softcap,
    const float* __restrict__ sink, const float* __restrict__ cgate, int ldcg) {
    constexpr int NDT = D / 16;         // 16-row tiles of d
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE);
    const int lane = threadIdx.x % TM_WAVE, r = lane % 16, g = lane / 16;
    // The newest tile walks the most keys, and a prompt's blocks are mostly all on the chip at once, so it is where they lie that balances
    // them: the tiles (newest first) go over the CUs, and in every second round of the CUs the other way round.
    const int round = blockIdx.x / AF_ROUND, in_round = blockIdx.x % AF_ROUND;
    const int left = (int)gridDim.x - round * AF_ROUND, items = left < AF_ROUND ? left : AF_ROUND;
    const int item = round * AF_ROUND + (round & 1 ? items - 1 - in_round : in_round);
    const int tile = item / H, h = item % H, kvh = h / (H / KVH);
    const int* tl = tiles + (size_t)tile * 4;
    const int s = tl[0], row0 = tl[1], valid = tl[2], pos0 = tl[3];
    const int* table = block_tables + (size_t)s * table_width;
    const int page = 1 << page_shift;
    const int last_key = pos0 + valid - 1;
    const int my_pos = pos0 + r < last_key ? pos0 + r : last_key;       // position of this lane's query column
    const int my_lo = (window > 0 && my_pos - window + 1 > 0) ? my_pos - window + 1 : 0;
    const int first_key = (window > 0 && pos0 - window + 1 > 0) ? pos0 - window + 1 : 0;
    const int last_lo = (window > 0 && last_key - window + 1 > 0) ? last_key - window + 1 : 0;

    // (columns beyond the tile's tokens: its last one again, not stored)
    const float* qrow = q + (size_t)(row0 + (r < valid ? r : valid - 1)) * q_stride + (size_t)h * D + 4 * g;
    f32x4_t qf[NDT];
#pragma unroll
    for (int c = 0; c < NDT; ++c) qf[c] = *(const f32x4_t*)(qrow + 16 * c);
    float m = -3.402823466e38f, l = 0.f; // the reference of the weights of this lane's column; this lane's share of their sum
    f32x4_t o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // key blocks: those of the kept first keys, then those from the oldest window's start on
    const int kb_first = first_key >> 4, kb_last = last_key >> 4;
    const int kb_kept = keep > 0 && first_key > 0 ? (keep + 15) >> 4 : 0;
    auto behind_gap = [&](int b) { return (b >= kb_kept && b < kb_first) ? kb_first + ((wave - kb_first) & (AF_SPLIT - 1)) : b; };
    // (behind the wavefront's last block the newest one there is again, unused: always at an entry this tile may see)
    auto page_of = [&](int b) { return table[((b <= kb_last ? b : kb_last) << 4) >> page_shift]; };
    const uint32_t row = TURN ? 4 * (r / 4) + g : r, piece = TURN ? r % 4 : g;
    const uint32_t k_lane = (row * KVH * D + 4 * piece) * 4, v_lane = ((row << page_shift) + 4 * piece) * 4;
    const int from = 4 * (16 * (r % 4) + 4 * (r / 4) + g);             // the lane, in bytes, that has row r's piece g
    auto turn = [&](f32x4_t& v) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(v[e])));
    };
    auto load = [&](KVBlock32<D>& blk, int b, int pg) {
        const int in_page = ((b <= kb_last ? b : kb_last) << 4) & (page - 1);
        // keys: lane (r, g) loads K[key0 + row][16 c + 4 piece .. + 3]; values: V[d = 16 dt + row][key0 + 4 piece .. + 3]. With TURN lane (r, g) holds
        // row r's piece g behind `turn`, without from the load on
        // (the page's and the key's place by the scalar unit, a lane's own place in them all along the same)
        const auto kr = fd_buffer(k_pool + ((((size_t)pg << page_shift) + in_page) * KVH + kvh) * D, 0x7fffffff);
        const auto vr = fd_buffer(v_pool + ((((size_t)pg * KVH + kvh) * D) << page_shift) + in_page, 0x7fffffff);
#pragma unroll
        for (int c = 0; c < NDT; ++c) blk.k[c] = as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(kr, k_lane + 64 * c, 0, 0));
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) blk.v[dt] = as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(vr, v_lane, (64 * dt) << page_shift, 0));
    };
    int kb = behind_gap(wave), next = behind_gap(kb + AF_SPLIT);
    int pg = page_of(kb), pg_next = page_of(next);
    auto attend = [&](KVBlock32<D>& now, KVBlock32<D>& then) {
        const int key0 = kb << 4;
        const int after = behind_gap(next + AF_SPLIT);
        if constexpr (AHEAD) {
            load(then, next, pg_next);                  // the next block, and the page of the one behind it
            pg_next = page_of(after);
        } else {
            load(now, kb, pg);
            pg = pg_next;
            pg_next = page_of(after);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TURN) {
#pragma unroll
            for (int c = 0; c < NDT; ++c) turn(now.k[c]);
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) turn(now.v[dt]);
        }
        // values of keys nobody may see yet (beyond the newest key) can hold anything: clear them
        if (key0 + 15 > last_key) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (key0 + 4 * g + i > last_key) now.v[dt][i] = 0.f;
        }
        f32x4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NDT; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[c][e], qf[c][e], sc, 0, 0, 0);
        // sc[i] = score of key key0 + 4 g + i for this lane's token
        bool hidden[4] = {false, false, false, false};
        if (key0 + 15 > pos0 || key0 < last_lo)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int kj = key0 + 4 * g + i;
                hidden[i] = kj > my_pos || (kj < my_lo && kj >= keep);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sc[i] *= scale;
            if (CAP) sc[i] = softcap * tanhf(sc[i] / softcap);
            sc[i] = hidden[i] ? -INFINITY : sc[i];
        }
        float bm = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        bm = lane_max<16>(bm);
        bm = lane_max<32>(bm);
        // (a column that has seen no key yet keeps the lowest number: -inf scores less that are -inf, their weights zeros. Whether a
        // column's reference moves hangs on that column alone)
        const bool grew = bm > m + AF_GROWTH;
        if (__builtin_expect(__any(grew), 0)) {
            const float corr = grew ? exp_weight(m - bm) : 1.f;
            m = grew ? bm : m;
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[dt][i] *= corr;
        }
        f32x4_t pr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            pr[i] = exp_weight(sc[i] - m);
            l += pr[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.v[dt][i], pr[i], o[dt], 0, 0, 0);
        kb = next;
        next = after;
    };
    KVBlock32<D> ba, bb;
    if constexpr (AHEAD) {
        load(ba, kb, pg);
        while (kb <= kb_last) {
            attend(ba, bb);
            if (kb > kb_last) break;
            attend(bb, ba);
        }
    } else {
        while (kb <= kb_last) attend(ba, ba);
    }
    // o[dt][i] = sum for d = 16 dt + 4 g + i of token r; the column's sum is spread over its four lanes.
    // The four wavefronts' partial results meet in LDS; a wavefront that had no key block brings the lowest number as its reference, l = 0, o = 0
    __shared__ float m_s[AF_SPLIT][16], l_s[AF_SPLIT][16];
    __shared__ __attribute__((aligned(16))) float o_s[AF_SPLIT][16][D + 4];
    const float own = lane_sum<32>(lane_sum<16>(l));
    if (g == 0) {
        m_s[wave][r] = m;
        l_s[wave][r] = own;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) *(f32x4_t*)&o_s[wave][r][16 * dt + 4 * g] = o[dt];
    __syncthreads();
    const int tok = threadIdx.x >> 4;
    if (tok >= valid) return;
    float mw[AF_SPLIT], sw[AF_SPLIT], top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < AF_SPLIT; ++w) {
        mw[w] = m_s[w][tok];
        top = fmaxf(top, mw[w]);
    }
#pragma unroll
    for (int w = 0; w < AF_SPLIT; ++w) {
        sw[w] = expf(mw[w] - top);                                      // a token always sees its own key: top is finite
        sum += l_s[w][tok] * sw[w];
    }
    if (sink) sum += expf(sink[h] - top);                                 // a term of the denominator without a key
    const float inv = 1.f / sum;
    float* orow = out + (size_t)(row0 + tok) * out_stride + (size_t)h * D;
    for (int d = (threadIdx.x & 15) * 4; d < D; d += 64) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < AF_SPLIT; ++w) {
            const f32x4_t part = *(const f32x4_t*)&o_s[w][tok][d];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += part[i] * sw[w];
        }
        if (cgate)                                                      // a gate per channel
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] *= 1.f / (1.f + expf(-cgate[(size_t)(row0 + tok) * ldcg + (size_t)h * D + d + i]));
        *(f32x4_t*)(orow + d) = f32x4_t{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    }
}

// q float32 [T, >= H*D] rows, out float32 [T, >= H*D]; pools float32, K [pages, page, KVH, D], V [pages, KVH, D, page];
// tiles int32 [n_tiles][4] = (request index, first row, tokens (1..16), position of the first token).
// Needs D % 16 == 0 (at most 128), page a power of two >= 16, 16-byte aligned q, out and pools, strides % 4 == 0.
// softcap > 0: a score s (scaled) becomes softcap * tanh(s / softcap) before the softmax; sink (float32 [H]) or null: one more term
// exp(sink[h]) in the denominator of head h's softmax, with no key behind it; with a window, `keep`: the first keys of a request
// that every token sees beside its window; cgate (rows of the flat batch, ldcg apart) or null: channel c of the result is multiplied by
// sigmoid(cgate[c]).
extern "C" int tm_attn_prefill_f32_cap(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                       const void* v_pool, const int* block_tables, int table_width, const int* tiles,
                                       int n_tiles, int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                       const float* sink, const void* cgate, int ldcg, hipStream_t stream) {
    if (n_tiles <= 0) return TM_OK;
    if (!(softcap >= 0.f) || keep < 0 || (cgate && ldcg < H * D)) return TM_ERR_ARG;
    if (H <= 0 || KVH <= 0 || H % KVH || page < 16 || (page & (page - 1)) || window < 0 || table_width <= 0 ||
        (q_stride % 4) || (out_stride % 4) || ((uintptr_t)q % 16) || ((uintptr_t)out % 16) || ((uintptr_t)k_pool % 16) ||
        ((uintptr_t)v_pool % 16) || q_stride < H * D || out_stride < H * D || !(scale > 0.f))
        return TM_ERR_ARG;
    if (H > 65535) return TM_ERR_ARG;
    int page_shift = 0;
    while ((1 << page_shift) < page) ++page_shift;
    // (a launch has fewer than 2^32 threads: tables beyond that go in pieces)
    const int most = (1 << 23) / H;
    const bool short_walk = window > 0 && (long long)window + keep <= AF_SHORT_WALK;
    const bool turn = AF_TURNS(D) && (long long)n_tiles * H >= AF_TURN_BLOCKS(D);
#define TM_PREFILL_F32_GO(DD, CAP, AHEAD, TURN)                                                                   \
    for (int t = 0; t < n_tiles; t += most)                                                                       \
        attn_prefill_f32_kernel<DD, CAP, AHEAD, TURN><<<(n_tiles - t < most ? n_tiles - t : most) * H, 64 * AF_SPLIT, 0, stream>>>( \
            (const float*)q, q_stride, (float*)out, out_stride, (const float*)k_pool, (const float*)v_pool,       \
            block_tables, table_width, tiles + (size_t)t * 4, H, KVH, page_shift, scale, window, keep, softcap, sink, (const float*)cgate, ldcg)
#define TM_PREFILL_F32_CASE(DD)                                                                                   \
    case DD:                                                                                                      \
        if (short_walk) {                                                                                         \
            if (softcap > 0.f) { TM_PREFILL_F32_GO(DD, true, false, false); } else { TM_PREFILL_F32_GO(DD, false, false, false); } \
        } else if (!turn) {                                                                                       \
            if (softcap > 0.f) { TM_PREFILL_F32_GO(DD, true, true, false); } else { TM_PREFILL_F32_GO(DD, false, true, false); } \
        } else {                                                                                                  \
            if (softcap > 0.f) { TM_PREFILL_F32_GO(DD, true, true, AF_TURNS(DD)); } else { TM_PREFILL_F32_GO(DD, false, true, AF_TURNS(DD)); } \
        }                                                                                                         \
        break
    switch (D) {
        TM_PREFILL_F32_CASE(16);
        TM_PREFILL_F32_CASE(32);
        TM_PREFILL_F32_CASE(48);
        TM_PREFILL_F32_CASE(64);
        TM_PREFILL_F32_CASE(80);
        TM_PREFILL_F32_CASE(96);
        TM_PREFILL_F32_CASE(112);
        TM_PREFILL_F32_CASE(128);
        default:
            return TM_ERR_ARG;
    }
#undef TM_PREFILL_F32_CASE
#undef TM_PREFILL_F32_GO
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_attn_prefill_f32(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                   const void* v_pool, const int* block_tables, int table_width, const int* tiles,
                                   int n_tiles, int H, int KVH, int D, int page, float scale, int window,
                                   hipStream_t stream) {
    return tm_attn_prefill_f32_cap(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, tiles, n_tiles, H, KVH, D,
                                   page, scale, window, 0, 0.f, nullptr, nullptr, 0, stream);
}
