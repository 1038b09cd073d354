// Paged attention for portions of prompts on MFMA (bfloat16), flash style: online softmax over
// blocks of 32 keys, nothing but registers between the two products.
//
//   A wavefront takes 16 consecutive query tokens of one request (a "tile"), one kv head and up to
//   four of the query heads that share it, so that every key and value fragment it loads feeds up
//   to four heads. Keys and values are read in place through the block table, this step's own
//   tokens included (they were stored before this kernel runs). A query at position p sees keys
//   lo..p, lo = 0 or p - window + 1, and with a window also the first `keep` (reference src/infer/kv/context.py:70-75,
//                                                   src/infer/model/layers.py:100-107).
//   Key blocks are aligned to absolute positions (multiples of 32) and visited in ascending order,
//   so a token's result does not depend on how its prompt was cut into portions nor on the rest of
//   the batch.
//
//   S^T = K Q^T      A = keys  [16 keys x 32 d]   from K[page][slot][kvh][d]
//                    B = Q^T   [32 d x 16 tokens]
//   O^T = V^T P^T    A = V^T   [16 d x 32 keys]   from V[page][kvh][d][slot]
//                    B = P^T   [32 keys x 16 tokens] straight from the S^T accumulators
#include "common.h"
#include "api.h"
#include "attention_prefill_common.h"
#include "choose.h"
#include "ahead.h"
#include "attention_decode_keys.h"

#include <algorithm>

// A block of 32 keys as a wavefront holds it between asking for it and using it. Row rho of operand tile t is key 16 t + rho: the lane which holds
// rows 4 g .. 4 g + 3 of both tiles of the scores has the keys 4 g .. + 3 of either, and wants the same of a row of V^T.
//
// What bounds a long prompt is the address unit of a CU, beside its vector units: it takes 64 bytes a cycle where four neighbouring lanes ask for a
// piece of one line, and one lane a cycle where they are in different keys, as the lanes of a score operand are (a key a lane). So keys are
// loaded as whole rows, eight lanes a row of 64, and change lanes through LDS (attend_block). At 8,000 tokens of the 0.5B shape the first-level
// caches had 112 million accesses in 443,000 cycles, one a cycle and CU, and have 43 million in 385,000. (Keys by loads of half rows that lanes exchange in
// registers ask for as many places: 2,048 / 8,000 tokens 26.1 and 215 us. The next block's keys through LDS behind this block's last score products, a
// wait less: spills, 27.0 and 197.)
//
// HALVES: values come as two loads of eight bytes a lane. In pages of 16 keys, whose rows of V^T lie side by side, that is the better way where a
// wavefront has two heads of more than 64 channels or four; else they come 16 bytes a lane, half of which belong to the lane 16 on (turn_values). us a launch, keys a
// lane and eight bytes / keys by rows and 16 bytes / by rows and eight bytes: 14 heads over 2 of 64, pages of 16, 77 / 512 / 2,048 / 8,000 tokens
// 4.87 / 4.58 / 4.68, 7.9 / 6.4 / 6.7, 24.2 / 22.3 / 21.7, 209 / 195 / 186, pages of 64, 77 / 3,001 6.5 / 4.8 / 5.6, 87 / 49 / 60; 16 over 16, 1,500
// 40.6 / 27.0 / 29.3; 12 over 2 of 96, 600 / 2,500 10.1 / 10.4 / 9.5, 56.7 / 57.6 / 50.7; 32 over 8 of 128, 1,500 78.2 / 78.2 / 67.6; 12 over 2 of 96, pages of 64, 700
// 16.6 / 11.8 / 13.9. The same bits.
template <int D>
struct KVBlock {
    static constexpr int PIECES = D / 8, ROW = 2 * D + 16, TILE = 16 * ROW;       // 16-byte pieces of a key; bytes of a key and of a tile in LDS
    u32x4_t k[2][D / 32];   // [16 keys][c]: piece 64 c + lane of the keys as they lie
    PFrag v[D / 16];        // [d tile]: of row d = r, keys 4 g .. + 3 of both tiles (HALVES), or 8 (g / 2) .. + 7 of tile g % 2
};

// Floats of LDS that a wavefront has: its partials of all heads, and before that a block's keys.
template <int D, int HPW>
constexpr int wave_floats() { return HPW * 16 * (D + 4) > KVBlock<D>::TILE / 2 ? HPW * 16 * (D + 4) : KVBlock<D>::TILE / 2; }

// What a lane adds to a tile's (wave-uniform) base address: constant for the whole kernel.
template <int D>
struct LaneOffsets {
    uint32_t k[D / 32];     // bytes: piece 64 c + lane of the tile's keys
    uint32_t v;             // bytes: d = r, and the keys (KVBlock)
    uint32_t turn[D / 32];  // bytes in LDS: where a tile's keys go
    uint32_t row;           // bytes in LDS: piece g of row r
};

// A raw buffer descriptor over memory that starts at a wave-uniform address: loads through it take
// the base from scalar registers and a 32-bit offset per lane, so no lane computes a 64-bit address.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_buffer(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}

// The key blocks of a wavefront: blocks `kept` and up are left out until `resume` (the gap between the kept first keys and the
// windows; without one kept = 0 and resume is the first block there is).
struct BlockWalk {
    int kept, resume;
    // block b of the walk that goes on by steps of KS from a block of it as if there were no gap
    template <int KS>
    __device__ __forceinline__ int at(int from, int b) const { return from < kept && b >= kept ? resume + (b - kept) / KS * KS : b; }
};

// Where the next 32 key blocks of a wavefront (blocks kb, kb + KS, ... of its walk) lie, one 16-key tile per
// lane: lane 2 i + t holds the places of tile t of the i-th of them, of its keys in units of 64 bytes of the key pool and of its
// values in units of 32 bytes of the value pool (a tile is whole runs of both). 64 lanes work them out at once; the scalar
// unit needed 47 instructions a tile, in a loop that waits for its results. A tile that holds no key any
// query of this wavefront may see (beyond the newest key, or wholly behind the window) is replaced
// by the nearest tile that does: its table entry may name no page. The caller masks every score of
// such a tile by the key's real position and clears its values (the tile in its place may hold keys beyond the newest one).
struct TilePlaces {
    uint32_t k, v;
};
template <int D, int KS>
__device__ __forceinline__ TilePlaces lane_pages(int kb, const BlockWalk& walk, int lane, int kept_tiles, int first_tile, int last_tile,
                                                 const int* __restrict__ table, int kvh, int KVH, int page_shift) {
    int tile = 2 * walk.at<KS>(kb, kb + (lane >> 1) * KS) + (lane & 1);
    tile = (tile < first_tile && tile >= kept_tiles) ? first_tile : (tile > last_tile ? last_tile : tile);
    const int tile0 = 16 * tile;
    const uint32_t page = (uint32_t)table[tile0 >> page_shift], in_page = (uint32_t)(tile0 & ((1 << page_shift) - 1));
    return TilePlaces{(((page << page_shift) + in_page) * KVH + kvh) * (D / 32), ((page * KVH + kvh) * D << (page_shift - 4)) + in_page / 16};
}

// Loads one block of 32 keys (two tiles of 16); slot = which of the 32 blocks held in `places`.
template <int D, bool HALVES>
__device__ __forceinline__ void load_kv_block(KVBlock<D>& blk, const TilePlaces& places, int slot, const bf16_t* __restrict__ k_pool,
                                              const bf16_t* __restrict__ v_pool, int page_shift, const LaneOffsets<D>& off) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t k_at = __builtin_amdgcn_readlane(places.k, 2 * slot + t);
        const __amdgpu_buffer_rsrc_t kbuf = uniform_buffer((const char*)k_pool + ((uint64_t)k_at << 6));
#pragma unroll
        for (int c = 0; c < D / 32; ++c) blk.k[t][c] = __builtin_amdgcn_raw_buffer_load_b128(kbuf, off.k[c], 0, 0);
    }
    const uint32_t v0 = __builtin_amdgcn_readlane(places.v, 2 * slot), v1 = __builtin_amdgcn_readlane(places.v, 2 * slot + 1);
    if constexpr (HALVES) {
        const __amdgpu_buffer_rsrc_t b0 = uniform_buffer((const char*)v_pool + ((uint64_t)v0 << 5)), b1 = uniform_buffer((const char*)v_pool + ((uint64_t)v1 << 5));
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            const u32x2_t lo = __builtin_amdgcn_raw_buffer_load_b64(b0, off.v, (32 * dt) << page_shift, 0);
            const u32x2_t hi = __builtin_amdgcn_raw_buffer_load_b64(b1, off.v, (32 * dt) << page_shift, 0);
            blk.v[dt].u = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
    } else {
        const char* vp = (const char*)v_pool + ((uint64_t)(threadIdx.x & 16 ? v1 : v0) << 5) + off.v;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) blk.v[dt].u = *(const u32x4_t*)(vp + ((size_t)(32 * dt) << page_shift));
    }
}

// Lane (r, g) has keys 4 g .. + 3 of one tile and the lane 16 on those of the other, each beside four that the other wants: an instruction a word
// changes them (rows of 16 lanes: the odd ones of the first operand with the even ones of the second).
template <int D>
__device__ __forceinline__ void turn_values(KVBlock<D>& blk) {
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const auto both = __builtin_amdgcn_permlane16_swap(blk.v[dt].u[w], blk.v[dt].u[w + 2], false, false);
            blk.v[dt].u[w] = both[0];
            blk.v[dt].u[w + 2] = both[1];
        }
}

// One block of 32 keys against the wavefront's heads.
template <int D, int HPW, bool CAP, bool HALVES>
__device__ __forceinline__ void attend_block(KVBlock<D>& blk, unsigned char* turn, const LaneOffsets<D>& off, HeadState<D, HPW>& st, const PFrag (&qf)[HPW][D / 32],
                                             int key0, int nh, const TileView& tv, int g, float scale_log2, float cap_in, float cap_out) {
    constexpr int NDC = D / 32, NDT = D / 16;
    // values of keys nobody may see (beyond the newest key, or behind every window: see lane_pages) can hold anything: clear them
    if (key0 + 31 > tv.last_key || key0 < tv.first_key) {
        uint32_t seen[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int k0 = key0 + (HALVES ? 4 * g + 16 * (w / 2) + 2 * (w % 2) : 16 * (g % 2) + 8 * (g / 2) + 2 * w);
            seen[w] = (tv.seen(k0) ? 0x0000ffffu : 0u) | (tv.seen(k0 + 1) ? 0xffff0000u : 0u);
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int w = 0; w < 4; ++w) blk.v[dt].u[w] &= seen[w];
    }
    if constexpr (!HALVES && D <= 64) turn_values(blk);
    // the keys change lanes: whole rows as they were loaded, a row a lane as the matrix unit takes them (rows 16 bytes more than their values
    // apart meet no bank twice)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < NDC; ++c) *(u32x4_t*)(turn + t * KVBlock<D>::TILE + off.turn[c]) = blk.k[t][c];
    // (a wavefront's LDS instructions are done in their order; this holds the compiler to it)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    PFrag kf[2][NDC];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < NDC; ++c) kf[t][c].u = *(const u32x4_t*)(turn + off.row + t * KVBlock<D>::TILE + 64 * c);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // does any (query, key) pair of this block fall outside the causal / window limits?
    const bool edge = (key0 + 31 > tv.pos0) || (key0 < tv.last_lo);
    // the score products of two heads first: the matrix unit works on the next head's while the vector unit does the softmax of this
    // one. (Of all four at once the registers do not hold the scores beside a block's keys in both orders.)
    auto heads = [&](auto FIRST, auto COUNT) {
        constexpr int h0 = decltype(FIRST)::value, AT_ONCE = decltype(COUNT)::value;
        __builtin_amdgcn_sched_barrier(0);
        f32x4_t sc[AT_ONCE][2];
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < NDC; ++c)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][c].b, qf[h0 + j][c].b, acc, 0, 0, 0);
                // capped scores: cap * tanh(score * scale / cap), kept in units of 1 / scale like the plain ones
                if constexpr (CAP) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = cap_out * tanh_fast(acc[i] * cap_in);
                }
                sc[j][t] = acc;
            }
        if (edge) {                                              // (which keys a column sees is worked out once for both heads)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int kj = key0 + 16 * t + 4 * g + i;
                    const bool mine = (kj <= tv.my_pos) & ((kj >= tv.my_lo) | (kj < tv.keep));
#pragma unroll
                    for (int j = 0; j < AT_ONCE; ++j) sc[j][t][i] = mine ? sc[j][t][i] : -INFINITY;
                }
        }
        // this lane's largest scores of the block (scale > 0: the maximum commutes with it)
        float lm[AT_ONCE];
        bool grows = false;
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            lm[j] = max3(-INFINITY, sc[j][0][0], sc[j][0][1]);
            lm[j] = max3(lm[j], sc[j][0][2], sc[j][0][3]);
            lm[j] = max3(lm[j], sc[j][1][0], sc[j][1][1]);
            lm[j] = max3(lm[j], sc[j][1][2], sc[j][1][3]);
            grows |= lm[j] * scale_log2 > st.m[h0 + j] + PF_SLACK;   // (true for a column that has seen no key: m = -inf)
        }
        // The running reference m of a column moves only when the block's maximum exceeds it by more
        // than PF_SLACK (in units of log2): until then the weights are exp2(s - m) <= 2^PF_SLACK instead of
        // <= 1, which changes nothing but their common scale (it cancels against the sum), and the
        // rescaling of the accumulators, the expensive part of a block on the vector unit, becomes rare.
        // Each column decides for itself and one that stays multiplies by exactly 1, so a query's result
        // does not depend on the other queries of its tile. Whether any column moves is asked of the lanes'
        // own maxima first (a column's maximum exceeds the limit exactly when one of its four lanes' does), so
        // the exchange between the lanes of a column is as rare as the rescaling.
        if (__any(grows)) {
#pragma unroll
            for (int j = 0; j < AT_ONCE; ++j) {
                const int hh = h0 + j;
                const float bm = column_max(lm[j]) * scale_log2;
                const bool grow = bm > st.m[hh] + PF_SLACK;
                const float m_new = grow ? bm : st.m[hh];
                const float corr = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(st.m[hh] - m_new);
                st.m[hh] = m_new;
                st.l[hh] *= corr;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st.o[hh][dt][i] *= corr;
            }
        }
        if constexpr (!HALVES && D > 64 && h0 == 0) turn_values(blk);      // (behind the scores up to 64 channels the registers do not hold it: 22.3 to 25.2 us at 2,048)
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            const int hh = h0 + j;
            // a column that has seen no key yet (m = -inf) gets zeros: exp2(-inf - 0)
            const float neg_m = (st.m[hh] == -INFINITY) ? 0.f : -st.m[hh];
            float pr[2][4];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pr[t][i] = __builtin_amdgcn_exp2f(fmaf(sc[j][t][i], scale_log2, neg_m));
                    st.l[hh] += pr[t][i];
                }
            PFrag pt;
            pt.u = u32x4_t{pk_bf16(pr[0][0], pr[0][1]), pk_bf16(pr[0][2], pr[0][3]), pk_bf16(pr[1][0], pr[1][1]),
                           pk_bf16(pr[1][2], pr[1][3])};
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                st.o[hh][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk.v[dt].b, pt.b, st.o[hh][dt], 0, 0, 0);
            }
        }
    };
    using std::integral_constant;
    if constexpr (HPW == 1) {
        heads(integral_constant<int, 0>{}, integral_constant<int, 1>{});
    } else {
        if (nh >= 2) heads(integral_constant<int, 0>{}, integral_constant<int, 2>{});        // (nh is the same in every lane)
        else heads(integral_constant<int, 0>{}, integral_constant<int, 1>{});
        if constexpr (HPW > 2) {
            if (nh >= 4) heads(integral_constant<int, 2>{}, integral_constant<int, 2>{});
            else if (nh == 3) heads(integral_constant<int, 2>{}, integral_constant<int, 1>{});
        }
    }
}

enum { PF_PLAIN, PF_PAIRS, PF_DEALT };

// tiles: int32 [n_tiles][4] = (request index in the step, first row of the tile in the flat batch,
//                              tokens in the tile (1..16), position of its first token)
// A block is KS wavefronts on the same tile and heads; wavefront j takes the key blocks kb with
// kb % KS == j and the partial results are merged through LDS in wavefront order. Which blocks a
// wavefront takes depends on absolute positions only, and a block in which a token sees no key
// changes nothing for it, so a token's bits do not depend on the tile it falls into.
// order: a block takes a tile and heads by its place in the grid (PF_PLAIN); tile b and then tile n_tiles - 1 - b (PF_PAIRS: in
// a table sorted by the number of keys a tile sees, the longest goes with the shortest and every block has the same
// work, the lower triangle of a prompt, folded); or the pieces of all heads in the order of the table (PF_DEALT).
// DECODES: `decodes.layers` layers of the grid in front attend single decoded tokens, a (request, kv head) a block (attend_whole). On its own that
// is a launch, or two, that waits for its trips to memory, behind one that leaves CUs without a block or their matrix units idle; the blocks in front
// are the first to get a CU, so a launch that does not fit the chip at once has its long blocks last. Prompt portions, tokens decoded beside them, us of
// both launches and of one (0.5B shape): 2 of 241 tokens behind 482, 30 of contexts to 1,000 17.2 to 12.1; 1 of 100, 4 of 300 10.2 to 5.9; 1 of 400 behind
// 1,000, 60 of 1,500 25.4 to 15.2; 4 of 400, 60 of 1,000 26.2 to 20.1; 2 of 256, 100 of 800 16.7 to 16.3.
struct KernelDecodes {
    const bf16_t* q;
    bf16_t* out;
    const int* tables;
    const int* context_lens;
    const bf16_t* cgate;
    int n, pairs, layers, chunks;
    float cap_out;
};
struct NoDecodes {};
template <bool DECODES>
using DecodesArg = std::conditional_t<DECODES, KernelDecodes, NoDecodes>;

template <int D, int HPW, int KS, bool CAP, bool AHEAD, bool DECODES, bool HALVES>
__global__ __launch_bounds__(64 * KS) void attn_prefill_mfma_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, int out_stride,
    const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool, const int* __restrict__ block_tables,
    int table_width, const int* __restrict__ tiles, int n_tiles, int order, int H, int KVH, int page_shift,
    float scale_log2, float cap_in, float cap_out, int window, int keep, const float* __restrict__ sink,
    const bf16_t* __restrict__ cgate, int ldcg, const TmAheadArg<AHEAD> ahead, const DecodesArg<DECODES> decodes) {
    constexpr int NDC = D / 32, NDT = D / 16;
    // the wavefronts' partials of all heads: rows of d four floats apart from a multiple of 64, so that 16 lanes of a store or load
    // of 16 bytes meet no bank twice
    __shared__ float s_m[KS][HPW][16], s_l[KS][HPW][16];
    extern __shared__ __align__(16) float s_o[];                     // [KS][wave_floats]: [HPW][16][D + 4]
    int layer = blockIdx.z;
    if constexpr (DECODES) {
        if (layer < decodes.layers) {
            const int pair = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * layer), of = pair / decodes.n;
            if (pair >= decodes.pairs) return;
            return attend_whole<D, KS, (D > 32)>(s_o, pair - of * decodes.n, of, decodes.q, q_stride, decodes.out, out_stride, k_pool, v_pool, decodes.tables,
                                       table_width, decodes.context_lens, decodes.chunks, H, KVH, page_shift, scale_log2, cap_in, decodes.cap_out, window,
                                       keep, sink, decodes.cgate, ldcg);
        }
        layer -= decodes.layers;
    }
    if constexpr (AHEAD) {
        if (layer) return tm_bring_ahead(ahead, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), KS);
    }
    auto partial_at = [&](int w, int hh, int col, int d) { return s_o + w * wave_floats<D, HPW>() + (hh * 16 + col) * (D + 4) + d; };
    // the wavefront index in a scalar register: everything derived from it (its key blocks, their
    // pages, the branches on them) stays wave-uniform
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE);
    const int lane = threadIdx.x % TM_WAVE, r = lane % 16, g = lane / 16;
    const int G = H / KVH;
    const int splits = (G + HPW - 1) / HPW;
    int tile0 = blockIdx.x, heads = blockIdx.y;
    if (order == PF_DEALT) {
        heads = tile0 % (KVH * splits);
        tile0 /= KVH * splits;
    }
    const int kvh = heads / splits, split = heads % splits;
    const int h0 = kvh * G + split * HPW;
    const int nh = (G - split * HPW) < HPW ? (G - split * HPW) : HPW;
    LaneOffsets<D> off;
    using Block = KVBlock<D>;
#pragma unroll
    for (int c = 0; c < NDC; ++c) {
        const int key = (64 * c + lane) / Block::PIECES, piece = (64 * c + lane) % Block::PIECES;
        off.k[c] = (uint32_t)(((size_t)key * KVH * D + 8 * piece) * sizeof(bf16_t));
        off.turn[c] = (uint32_t)(key * Block::ROW + 16 * piece);
    }
    off.v = (uint32_t)((((size_t)r << page_shift) + (HALVES ? 4 * g : 8 * (g / 2))) * sizeof(bf16_t));
    off.row = (uint32_t)(r * Block::ROW + 16 * g);
    unsigned char* turn = (unsigned char*)partial_at(wave, 0, 0, 0);         // (the place of this wavefront's partials, which are stored behind the last block)
    const int other = n_tiles - 1 - tile0;
    const int n_mine = (order == PF_PAIRS && other > tile0) ? 2 : 1;

    // A tile begins with three trips to memory (its entry in the table, its queries and pages, its first keys). Those of the second
    // tile are made while the first one's partials meet.
    int row0, valid, pos0, kb, kb1, kept_tiles, first_tile, last_tile;
    const int* table;
    TileView tv;
    BlockWalk walk;
    PFrag qf[HPW][NDC];
    KVBlock<D> ba, bb;
    TilePlaces pages;
    auto begin = [&](int tile) {                                     // up to the queries and the pages
        const int* tl = tiles + (size_t)tile * 4;
        const int s = tl[0];
        row0 = tl[1], valid = tl[2], pos0 = tl[3];
        table = block_tables + (size_t)s * table_width;
        tv = tile_view(pos0, valid, r, window, keep);
        const int kb0 = tv.first_key / 32;
        kb1 = tv.last_key / 32;
        first_tile = tv.first_key / 16, last_tile = tv.last_key / 16;
        walk.kept = tv.first_key > 0 ? (tv.keep + 31) / 32 : 0;
        kept_tiles = tv.first_key > 0 ? (tv.keep + 15) / 16 : 0;
        const int behind = kb0 > walk.kept ? kb0 : walk.kept;        // the first block >= behind of this wavefront:
        walk.resume = behind + ((wave - behind) & (KS - 1));
        kb = wave < walk.kept ? wave : walk.resume;
        pages = lane_pages<D, KS>(kb, walk, lane, kept_tiles, first_tile, last_tile, table, kvh, KVH, page_shift);
        // (columns beyond the tile's tokens are its last token again, heads beyond the group its last head: nobody reads their results)
        const bf16_t* qrow = q + (size_t)(row0 + (r < valid ? r : valid - 1)) * q_stride + 8 * g;
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh)
#pragma unroll
            for (int c = 0; c < NDC; ++c) qf[hh][c].u = *(const u32x4_t*)(qrow + (size_t)(h0 + (hh < nh ? hh : nh - 1)) * D + 32 * c);
    };
    begin(tile0);
    load_kv_block<D, HALVES>(ba, pages, 0, k_pool, v_pool, page_shift, off);

#pragma unroll 1
    for (int which = 0; which < n_mine; ++which) {
        HeadState<D, HPW> st;
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            st.m[hh] = -INFINITY;
            st.l[hh] = 0.f;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) st.o[hh][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }

        // Two register sets take turns: one is worked on while the other's loads are in flight. The
        // load after the last block repeats it, unused, so that no load hides behind a branch.
        int slot = 0;                                                // block kb is slot `slot` of `pages`
        while (kb <= kb1) {
            if (slot == 31) {                                        // the next block starts a new set of pages
                pages = lane_pages<D, KS>(walk.at<KS>(kb, kb + KS), walk, lane, kept_tiles, first_tile, last_tile, table, kvh, KVH, page_shift);
                slot = -1;
            }
            load_kv_block<D, HALVES>(bb, pages, slot + 1, k_pool, v_pool, page_shift, off);
            attend_block<D, HPW, CAP, HALVES>(ba, turn, off, st, qf, kb * 32, nh, tv, g, scale_log2, cap_in, cap_out);
            kb = walk.at<KS>(kb, kb + KS);
            ++slot;
            if (kb > kb1) break;
            if (slot == 31) {
                pages = lane_pages<D, KS>(walk.at<KS>(kb, kb + KS), walk, lane, kept_tiles, first_tile, last_tile, table, kvh, KVH, page_shift);
                slot = -1;
            }
            load_kv_block<D, HALVES>(ba, pages, slot + 1, k_pool, v_pool, page_shift, off);
            attend_block<D, HPW, CAP, HALVES>(bb, turn, off, st, qf, kb * 32, nh, tv, g, scale_log2, cap_in, cap_out);
            kb = walk.at<KS>(kb, kb + KS);
            ++slot;
        }

        // The wavefronts' partials meet in LDS, all heads at once, and are added in wavefront order. (A head at a time, 17 KB of LDS and two
        // barriers each, this took 5 of a tile's 13 to 15 us at 2,048 tokens.)
        const int done_row0 = row0, done_valid = valid;
        const bool more = which + 1 < n_mine;
        if (more) begin(other);
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            if (hh >= nh) continue;                                  // block-uniform
            const float lsum = lane_sum<32>(lane_sum<16>(st.l[hh]));
            if (g == 0) {
                s_m[wave][hh][r] = st.m[hh];
                s_l[wave][hh][r] = lsum;
            }
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) *(f32x4_t*)partial_at(wave, hh, r, 16 * dt + 4 * g) = st.o[hh][dt];    // lane: d = 16 dt + 4 g + i of token r
        }
        if (more) load_kv_block<D, HALVES>(ba, pages, 0, k_pool, v_pool, page_shift, off);
        __syncthreads();
        // a thread: four channels of a token and head
        for (int idx = threadIdx.x; idx < nh * 16 * (D / 4); idx += 64 * KS) {
            const int d = 4 * (idx % (D / 4)), col = idx / (D / 4) % 16, hh = idx / (16 * (D / 4));
            if (col >= done_valid) continue;
            uint2 gp = {0u, 0u};
            if (cgate) {                                             // a gate per channel
                const bf16_t* gate = cgate + (size_t)(done_row0 + col) * ldcg + (size_t)(h0 + hh) * D + d;
                gp = uint2{*(const uint32_t*)gate, *(const uint32_t*)(gate + 2)};
            }
            float mm = s_m[0][hh][col];
#pragma unroll
            for (int w = 1; w < KS; ++w) mm = fmaxf(mm, s_m[w][hh][col]);
            float ll = 0.f;
            f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < KS; ++w) {
                const float mw = s_m[w][hh][col];
                const float f = (mw == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mw - mm);
                const f32x4_t ow = *(const f32x4_t*)partial_at(w, hh, col, d);
                ll = fmaf(s_l[w][hh][col], f, ll);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = fmaf(ow[i], f, o[i]);
            }
            if (sink) ll += __builtin_amdgcn_exp2f(sink[h0 + hh] * 1.4426950408889634f - mm);      // a term of the denominator without a key
            const float inv = 1.f / ll;
            if (cgate) {
                o[0] *= sigmoid_fast(__uint_as_float(gp.x << 16));
                o[1] *= sigmoid_fast(__uint_as_float(gp.x & 0xffff0000u));
                o[2] *= sigmoid_fast(__uint_as_float(gp.y << 16));
                o[3] *= sigmoid_fast(__uint_as_float(gp.y & 0xffff0000u));
            }
            uint32_t* dst = (uint32_t*)(out + (size_t)(done_row0 + col) * out_stride + (size_t)(h0 + hh) * D + d);
            dst[0] = pk_bf16(o[0] * inv, o[1] * inv);                // (the rows are 4-byte aligned, no more)
            dst[1] = pk_bf16(o[2] * inv, o[3] * inv);
        }
        if (more) __syncthreads();                                   // the partials have been read
    }
}

// Heads a wavefront takes and wavefronts a block has, by head size (registers decide). Up to head size 64 a
// wavefront can hold four heads, which quarters the loads of a long prompt's keys; a short step, whose blocks of
// two heads a wavefront still fit the chip in one round, takes those instead: twice the blocks, half as long
// (512 tokens at the 0.5B shape: 13.4 to 9.8 us; one a CU with the blocks of decoded tokens too, or those of four heads: 482 tokens beside 30 of
// 1,000 keys 16.5 to 12.1). A kv head of one or two heads takes no more than it has: places that stand empty cost
// queries, room for partials in LDS and with it blocks a CU (8 heads of 64 and as many kv heads, 17 / 512 / 2,048 tokens, four places 5.9 / 9.2 /
// 40.6 us, one 4.1 / 7.0 / 34.8). A head's arithmetic is the same either way, so its bits are.
template <int D> struct PrefillShape { static constexpr int HPW = D <= 64 ? 4 : 2, KS = D <= 64 ? 8 : 4; };

// The order of a launch's pieces of work (a tile and the heads a wavefront takes of one kv head), of which a CU mostly holds one.
// Two tiles a block save a block its beginning: the second tile's trips to memory are made while the first one's partials
// meet. But a pair is as long as the longest tile, and where the pairs do not fill their last round of the 256 CUs, pieces of
// their own, handed out longest first over all heads, are better balanced by the CUs that come free. us on an MI355X, pairs (below 256 of them:
// tiles by heads) / dealt: 14 heads over 2 of 64, 1,040 tokens (a fill of 0.52) 13.2 / 13.3, 1,100 (0.55) 12.9 / 13.5, 1,200 (0.59) 16.2 / 15.2, 1,500 (0.73) 20.9 / 18.2,
// 2,100 (0.52) 37.3 / 29.2, 3,001 (0.73) 48.0 / 43.9, 3,400 (0.84) 52.3 / 53.2, 3,700 (0.91) 55.6 / 58.4, 4,096 (1) 60.9 / 67.9; 32 over 8 of 128, 600
// (0.59) 30.6 / 24.0, 800 (0.78) 34.2 / 33.8, 900 (0.91) 36.4 / 37.9; 8 over 8 of 64, 1,500 (0.73) 18.5 / 14.9; 12 over 2 of 96, 1,500 (0.55) 36.4 / 27.2.
// From 218 pairs (0.85) on pairs are better than tiles by heads too (1,740 and 1,900 tokens of the first 24.1 / 20.5, 24.8 / 21.9), with fewer they are not (1,100
// tokens, as the kernel was before, 14.6 / 18.8). Head size 32, where a CU holds two blocks, stays with tiles by heads and pairs from 256 on (2,500 tokens of 12
// heads over 2, as it was, 26.4 / 28.5 dealt), and up to 256 pieces there is nothing to choose. Pieces that do not fit the grid's x are not dealt.
static int prefill_order(int D, int threads, long long pieces, long long folded) {
    if (D < 64 || pieces <= 256 || !fits_a_dimension(pieces, threads)) return folded >= 256 ? PF_PAIRS : PF_PLAIN;
    return 100 * folded < 85 * 256 * ((folded + 255) / 256) ? PF_DEALT : PF_PAIRS;
}

// ... of a launch (for tests), with `heads` query heads of a kv head a wavefront
extern "C" int tm_attn_prefill_order(int H, int KVH, int D, int heads, int n_tiles) {
    if (H <= 0 || KVH <= 0 || H % KVH || heads <= 0 || n_tiles <= 0) return -1;
    const long long columns = (long long)KVH * ((H / KVH + heads - 1) / heads);
    return prefill_order(D, 64 * (D <= 64 ? PrefillShape<64>::KS : PrefillShape<128>::KS), n_tiles * columns, (n_tiles / 2 + n_tiles % 2) * columns);
}

template <int D, int HPW, bool CAP>
static int launch_split_keys(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                              const int* block_tables, int table_width, const int* tiles, int n_tiles, int H, int KVH,
                              int page_shift, float scale_log2, float cap_in, float cap_out, int window, int keep, const float* sink,
                              const bf16_t* cgate, int ldcg, TmAhead& ahead, const TmDecodes* beside, hipStream_t stream) {
    constexpr int KS = PrefillShape<D>::KS;
    const int splits = (H / KVH + HPW - 1) / HPW;
    const long long pieces = (long long)n_tiles * KVH * splits, folded = (long long)(n_tiles / 2 + n_tiles % 2) * KVH * splits;
    const int order = prefill_order(D, 64 * KS, pieces, folded);
    dim3 grid = order == PF_DEALT ? dim3((unsigned)pieces) : dim3(order == PF_PAIRS ? n_tiles / 2 + n_tiles % 2 : n_tiles, KVH * splits);
    constexpr int lds = KS * wave_floats<D, HPW>() * (int)sizeof(float);          // at most 139,264 bytes
    const long long layer = (long long)grid.x * grid.y;
    const int pairs = beside ? beside->n * KVH : 0, front = beside ? (int)((pairs + layer - 1) / layer) : 0;
    const bool far = layer + pairs >= 256;                           // (more blocks than CUs: none to spare)
    if (far) ahead.n = 0;
    grid.z = 1 + front + (far ? 0 : ahead_spare_layers(ahead, layer, layer + pairs));
    if (front) ahead.first = (int)layer * (1 + front);
    auto go = [&](auto AHEAD, auto DECODES, auto PIECES) {
        constexpr bool with = decltype(AHEAD)::value, decode = decltype(DECODES)::value, halves = decltype(PIECES)::value;
        DecodesArg<decode> decodes;
        int bytes = lds;
        if constexpr (decode) {
            decodes = {(const bf16_t*)beside->q, (bf16_t*)beside->out, beside->tables, beside->context_lens, (const bf16_t*)beside->cgate, beside->n, pairs,
                       front, beside->chunks, beside->cap_out};
            bytes = std::max(bytes, (int)tm_decode_whole_lds(beside->chunks, H / KVH, D));
        }
        constexpr int most = decode ? std::max(lds, TM_DECODE_BESIDE_LDS) : lds;
        if (most > 64 * 1024) {
            static const hipError_t raised = hipFuncSetAttribute((const void*)attn_prefill_mfma_kernel<D, HPW, KS, CAP, with, decode, halves>,
                                                                 hipFuncAttributeMaxDynamicSharedMemorySize, most);
            if (raised != hipSuccess) return TM_ERR_LAUNCH;
        }
        attn_prefill_mfma_kernel<D, HPW, KS, CAP, with, decode, halves><<<grid, 64 * KS, bytes, stream>>>(
            (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, (const bf16_t*)k_pool, (const bf16_t*)v_pool, block_tables,
            table_width, tiles, n_tiles, order, H, KVH, page_shift, scale_log2, cap_in, cap_out, window, keep, sink, cgate, ldcg, ahead_arg<with>(ahead), decodes);
        return TM_OK;
    };
    auto with_values = [&](auto PIECES) {
        if constexpr (D <= 64) {
            if (beside) return ahead.n ? go(std::true_type{}, std::true_type{}, PIECES) : go(std::false_type{}, std::true_type{}, PIECES);
        }
        return ahead.n ? go(std::true_type{}, std::false_type{}, PIECES) : go(std::false_type{}, std::false_type{}, PIECES);
    };
    if constexpr (D <= 64 ? HPW > 2 : HPW > 1) {
        if (page_shift == 4) return with_values(std::true_type{});
    }
    return with_values(std::false_type{});
}

// softcap > 0: a score s (scaled) becomes softcap * tanh(s / softcap) before the softmax; sink (float32 [H]) or null: one more term
// exp(sink[h]) in the denominator of head h's softmax, with no key behind it; with a window, `keep`: the first keys of a request that
// every query sees beside its window; cgate (rows of the flat batch, ldcg apart) or null: channel c of the result is multiplied by
// sigmoid(cgate[c])
int attn_prefill_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                        const void* v_pool, const int* block_tables, int table_width, const int* tiles,
                                        int n_tiles, int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                        const float* sink, const void* cgate, int ldcg, TmAhead& ahead, hipStream_t stream, TmDecodes* beside) {
    if (beside) {
        if (n_tiles <= 0 || beside->n <= 0 || D > 64 ||
            !decode_args_ok(beside->q, q_stride, beside->out, out_stride, table_width, beside->chunks, H, KVH, D, page, scale, window, keep, softcap, beside->cgate, ldcg) ||
            tm_decode_whole_lds(beside->chunks, H / KVH, D) > TM_DECODE_BESIDE_LDS || (long long)beside->n * KVH > 32768)
            return TM_ERR_ARG;
        beside->cap_out = softcap * 1.4426950408889634f;
    }
    if (n_tiles <= 0) return TM_OK;
    if (!(softcap >= 0.f) || keep < 0 || (cgate && (ldcg < H * D || ldcg % 2 || (uintptr_t)cgate % 4))) return TM_ERR_ARG;
    const float cap_in = softcap > 0.f ? scale / softcap : 0.f, cap_out = softcap > 0.f ? softcap / scale : 0.f;
    if (H <= 0 || KVH <= 0 || H % KVH || page < 16 || (page & (page - 1)) || window < 0 || table_width <= 0 ||
        (q_stride % 8) || ((uintptr_t)q % 16) || (out_stride % 2) || ((uintptr_t)out % 4) || q_stride < H * D ||
        out_stride < H * D || !(scale > 0.f))
        return TM_ERR_ARG;
    const int G = H / KVH;
    int page_shift = 0;
    while ((1 << page_shift) < page) ++page_shift;
    const float scale_log2 = scale * 1.4426950408889634f;
    if ((long long)KVH * ((G + 1) / 2) > 65535) return TM_ERR_ARG;
    int rc = TM_OK;
#define TM_SPLIT_ARGS q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, tiles, n_tiles, H, KVH, \
                      page_shift, scale_log2, cap_in, cap_out, window, keep, sink, (const bf16_t*)cgate, ldcg, ahead, beside, stream
#define TM_PREFILL_CASE(DD)                                                                                       \
    case DD: {                                                                                                    \
        constexpr int HPW = PrefillShape<DD>::HPW;                                                                \
        if (G == 1)                                                                                               \
            rc = softcap > 0.f ? launch_split_keys<DD, 1, true>(TM_SPLIT_ARGS) : launch_split_keys<DD, 1, false>(TM_SPLIT_ARGS); \
        else if (HPW > 2 && (G == 2 || ((long long)n_tiles * ((G + 1) / 2) + (beside ? beside->n : 0)) * KVH <= TM_PREFILL_ONE_ROUND)) \
            rc = softcap > 0.f ? launch_split_keys<DD, 2, true>(TM_SPLIT_ARGS) : launch_split_keys<DD, 2, false>(TM_SPLIT_ARGS); \
        else                                                                                                      \
            rc = softcap > 0.f ? launch_split_keys<DD, HPW, true>(TM_SPLIT_ARGS) : launch_split_keys<DD, HPW, false>(TM_SPLIT_ARGS); \
        break;                                                                                                    \
    }
    switch (D) {
        TM_PREFILL_CASE(32)
        TM_PREFILL_CASE(64)
        TM_PREFILL_CASE(96)
        TM_PREFILL_CASE(128)
        default:
            return TM_ERR_ARG;
    }
#undef TM_PREFILL_CASE
#undef TM_SPLIT_ARGS
    if (rc) return rc;
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_attn_prefill_mfma_cap(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                        const void* v_pool, const int* block_tables, int table_width, const int* tiles,
                                        int n_tiles, int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                        const float* sink, const void* cgate, int ldcg, hipStream_t stream) {
    TmAhead none;
    return attn_prefill_ahead(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, tiles, n_tiles, H, KVH, D, page, scale, window, keep,
                              softcap, sink, cgate, ldcg, none, stream);
}

extern "C" int tm_attn_prefill_mfma(const void* q, int q_stride, void* out, int out_stride, const void* k_pool,
                                    const void* v_pool, const int* block_tables, int table_width, const int* tiles,
                                    int n_tiles, int H, int KVH, int D, int page, float scale, int window,
                                    hipStream_t stream) {
    return tm_attn_prefill_mfma_cap(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, tiles, n_tiles, H, KVH, D,
                                    page, scale, window, 0, 0.f, nullptr, nullptr, 0, stream);
}

// The same with single decoded tokens beside them: qd their queries and outd their results (a row a request, in the strides of q and out), of requests with
// block tables `tables`, context_lens and contexts of at most `chunks` chunks of 256.
extern "C" int tm_attn_prefill_decodes(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                                       const int* block_tables, int table_width, const int* tiles, int n_tiles, const void* qd, void* outd, const int* tables,
                                       const int* context_lens, int chunks, int n, int H, int KVH, int D, int page, float scale, int window, int keep,
                                       float softcap, const float* sink, const void* cgate, const void* cgated, int ldcg, hipStream_t stream) {
    TmAhead none;
    TmDecodes decodes{qd, outd, tables, context_lens, cgated, n, chunks, 0.f};
    return attn_prefill_ahead(q, q_stride, out, out_stride, k_pool, v_pool, block_tables, table_width, tiles, n_tiles, H, KVH, D, page, scale, window, keep,
                              softcap, sink, cgate, ldcg, none, stream, &decodes);
}
