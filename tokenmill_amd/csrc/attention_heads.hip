// Attention of prompt portions over a shared latent with keys and values per head (bfloat16): the portions' visible rows of the cache
// are gathered, the per-head matrices move them to keys and values once (plain products, gemm_tile.hip), and a flash-style
// kernel multiplies queries of Dn + Dr channels by them. Against the attention over the latent itself (latent_mfma.hip: a
// query of Lk + Dr channels, a result of Lk, each row of the cache read by every head) a (query, key) pair costs Dn + Dr + Dv in
// place of 2 Lk + Dr products, 320 for 1,088 at Lk 512, and moving a row costs once what moving a query and its result onto the
// latent did. Few queries gain most: over the latent a tile of them has four blocks that walk all rows one after the other (2 tokens behind
// 4,000 rows at 2k sizes 611 to 119 us a layer).
//
// A block: 64 queries of a head; its four wavefronts are two groups of 32 queries by two halves of every 64 keys. Keys (64 rows of
// Dn + Dr, the last Dr shared by the heads) and transposed values (Dv rows of 64) come straight into LDS, 16 bytes a lane, two buffers
// that take turns; 40 KB a buffer at 192 + 128 channels, so that a CU holds two blocks, whose waits and arithmetic interleave.
// Pieces of 16 bytes lie where an XOR by the row puts them, so operand loads meet no bank twice.
//   S^T = K Q^T      A = keys [32 x 16 channels], lane (r, half): row key_of(r), B = Q^T in registers
//   O^T = V^T P^T    A = V^T [32 channels x 16 keys], B = P^T straight from the S^T accumulators: rows of K are taken in the order
//                    that gives a lane eight consecutive keys
// The halves' results meet in LDS at the end. Keys are visited in blocks aligned to absolute positions, in ascending order, so a
// token's result depends on its request's cache and its position only. The softmax's reference moves as in attention_prefill.hip.
#include "common.h"
#include "api.h"
#include "attention_prefill_common.h"
#include "fused_common.h"

typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct HeadsArgs {
    const bf16_t* q;            // [T, H (DN + DR)], rows ldq apart
    const bf16_t* qr;           // [T, H DR]: the queries' last DR channels, rotated
    const bf16_t* kv;           // keys [R, H DN], behind them (rope_at bytes) the shared channels [R, DR]
    const bf16_t* vt;           // [H DV, R]
    bf16_t* out;                // [T, H DV]
    const int* blocks;          // [n][4]: first row of q, queries (1..64), position of the first, row of position 0 in kv and vt
    const float* gate;          // [T, >= H], rows ldg apart, or null
    const float* sink;          // [H] or null
    uint32_t rope_at;
    int ldq, ldg, H, R, window;
    float scale_log2;
};

// Rows of K (DK channels) in LDS: where piece p of row r lies. 384-byte rows start at one of two places of the 64 banks, 192-byte
// rows at one of four; the XOR spreads the rest of 16 consecutive rows.
template <int DK>
__device__ __forceinline__ int heads_key_piece(int p, int r) {
    return DK * 2 % 256 == 128 ? p ^ ((r >> 1) & 7) : p ^ ((r >> 2) & 3);
}

template <int DN, int DR, int DV>
__global__ __launch_bounds__(256, 2) void attn_heads_kernel(const HeadsArgs a) {
    constexpr int DK = DN + DR, KP = DK / 8, NC = DK / 16, ND = DV / 32;
    constexpr int KBYTES = 64 * DK * 2, VBYTES = DV * 128, STAGE = KBYTES + VBYTES;
    constexpr int KL = KP / 4, VL = DV / 32;                        // loads a wavefront makes for a buffer
    static_assert(KP % 4 == 0 && DV % 32 == 0 && DN % 16 == 0 && DR % 16 == 0 && (DK * 2 % 256 == 128 || DK * 2 % 128 == 64), "");
    extern __shared__ __align__(16) unsigned char ah_smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)ah_smem;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int col = lane % 32, half = lane / 32;
    const int qg = wave / 2, kg = wave % 2;
    const int head = blockIdx.x % a.H;                              // (a head's blocks on one or two XCDs: its keys stay in their L2)
    const int* e = a.blocks + 4 * (blockIdx.x / a.H);
    const int row0 = e[0], valid = e[1], pos0 = e[2], kv0 = e[3];

    // queries: column `col` of this wavefront's group; beyond the last one: that again, never stored
    const int query = 32 * qg + col < valid ? 32 * qg + col : valid - 1;
    const int token = row0 + query, my_pos = pos0 + query;
    const int my_lo = (a.window > 0 && my_pos - a.window + 1 > 0) ? my_pos - a.window + 1 : 0;
    PFrag qf[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        qf[c].u = *(const u32x4_t*)(c < DN / 16 ? a.q + (size_t)token * a.ldq + head * DK + 16 * c + 8 * half
                                                : a.qr + (size_t)token * a.H * DR + head * DR + 16 * c - DN + 8 * half);
    // what the wavefront's queries see (the same in every lane)
    const bool any = 32 * qg < valid;
    const int first_pos = pos0 + (any ? 32 * qg : 0), last_pos = pos0 + (valid < 32 * qg + 32 ? valid : 32 * qg + 32) - 1;
    const int first_lo = (a.window > 0 && first_pos - a.window + 1 > 0) ? first_pos - a.window + 1 : 0;
    const int last_lo = (a.window > 0 && last_pos - a.window + 1 > 0) ? last_pos - a.window + 1 : 0;

    // blocks of 64 keys of the whole block of queries
    const int block_lo = (a.window > 0 && pos0 - a.window + 1 > 0) ? pos0 - a.window + 1 : 0;
    const int t0 = block_lo / 64, t1 = (pos0 + valid - 1) / 64;
    uint32_t koff[KL], kinc[KL], voff[VL];
    const int kv_row = 64 * t0 + kv0;
#pragma unroll
    for (int i = 0; i < KL; ++i) {
        const int idx = (wave + 4 * i) * 64 + lane, r = idx / KP, p = heads_key_piece<DK>(idx % KP, r);
        const bool own = p < DN / 8;
        kinc[i] = 64u * (own ? a.H * DN * 2 : DR * 2);
        koff[i] = own ? (uint32_t)(kv_row + r) * (a.H * DN * 2) + head * DN * 2 + p * 16
                      : a.rope_at + (uint32_t)(kv_row + r) * (DR * 2) + (p - DN / 8) * 16;
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
        const int idx = (wave + 4 * i) * 64 + lane, ch = idx / 8, p = (idx % 8) ^ ((ch >> 1) & 7);
        voff[i] = (uint32_t)(head * DV + ch) * (a.R * 2) + kv_row * 2 + p * 16;
    }
    auto issue = [&](int buf) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + wave * 1024);
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            fd_load_lds(dst + i * 4096, koff[i], a.kv);
            koff[i] += kinc[i];
        }
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            fd_load_lds(dst + KBYTES + i * 4096, voff[i], a.vt);
            voff[i] += 128;
        }
    };

    // where this lane's operands lie in a buffer: row `col` of a tile of 32 keys is the key that makes the products' results eight
    // consecutive keys a lane (bits 2 and 3 of a run of 16 change places)
    const int key_row = 32 * kg + (col & 19) + ((col & 4) << 1) + ((col & 8) >> 1);
    const unsigned char* k_row = ah_smem + key_row * (DK * 2);
    const unsigned char* v_row = ah_smem + KBYTES + col * 128;
    const int v_swz = (col >> 1) & 7;

    float neg = 0.f, limit = -INFINITY, l = 0.f;                    // the softmax's reference m as -m and m + PF_SLACK
    f32x16_t o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.f;

    issue(0);
    int buf = 0;
    for (int t = t0; t <= t1; ++t) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this wavefront's part of the buffer is there ...
        __builtin_amdgcn_s_barrier();                               // ... and everybody's, and the other buffer has been read
        asm volatile("" ::: "memory");
        if (t < t1) issue(buf ^ 1);
        const int key0 = 64 * t + 32 * kg;
        if (any && key0 <= last_pos && key0 + 31 >= first_lo) {     // (the same in every lane)
            const unsigned char *kr = k_row + buf * STAGE, *vr = v_row + buf * STAGE;
            f32x16_t sc;
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[i] = 0.f;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                PFrag kf;
                kf.u = *(const u32x4_t*)(kr + heads_key_piece<DK>(2 * c + half, key_row) * 16);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf.b, qf[c].b, sc, 0, 0, 0);
            }
            if (key0 + 31 > first_pos || key0 < last_lo) {          // a pair outside the limits
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int kj = key0 + 16 * (i / 8) + 8 * half + i % 8;
                    sc[i] = (kj <= my_pos) & (kj >= my_lo) ? sc[i] : -INFINITY;
                }
            }
            float lm = max3(-INFINITY, sc[0], sc[1]);
#pragma unroll
            for (int i = 2; i < 16; i += 2) lm = max3(lm, sc[i], sc[i + 1]);
            if (__any(lm * a.scale_log2 > limit)) {                 // (true for a column that has seen no key)
                const float bm = lane_max<32>(lm) * a.scale_log2;
                const bool grow = bm > limit;
                const float m = limit == -INFINITY ? -INFINITY : -neg, m_new = grow ? bm : m;
                const float corr = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
                neg = m_new == -INFINITY ? 0.f : -m_new;
                limit = m_new + PF_SLACK;
                l *= corr;
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[d][i] *= corr;
            }
            float pr[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                pr[i] = __builtin_amdgcn_exp2f(fmaf(sc[i], a.scale_log2, neg));
                l += pr[i];
            }
            PFrag pt[2];
#pragma unroll
            for (int s = 0; s < 2; ++s)
                pt[s].u = u32x4_t{pk_bf16(pr[8 * s], pr[8 * s + 1]), pk_bf16(pr[8 * s + 2], pr[8 * s + 3]), pk_bf16(pr[8 * s + 4], pr[8 * s + 5]),
                                  pk_bf16(pr[8 * s + 6], pr[8 * s + 7])};
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    PFrag vf;
                    vf.u = *(const u32x4_t*)(vr + d * 4096 + ((4 * kg + 2 * s + half) ^ v_swz) * 16);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.b, pt[s].b, o[d], 0, 0, 0);
                }
        }
        buf ^= 1;
    }
    // the second half's results to the first, through LDS
    l = lane_sum<32>(l);
    float m = limit == -INFINITY ? -INFINITY : -neg;
    float* ml = (float*)(ah_smem + qg * (ND * 4096 + 512)) + lane;
    f32x4_t* parts = (f32x4_t*)(ah_smem + qg * (ND * 4096 + 512) + 512) + lane;
    __syncthreads();
    if (kg == 1) {
        ml[0] = m;
        ml[64] = l;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) parts[(d * 4 + i) * 64] = f32x4_t{o[d][4 * i], o[d][4 * i + 1], o[d][4 * i + 2], o[d][4 * i + 3]};
    }
    __syncthreads();
    if (kg == 1 || 32 * qg + col >= valid) return;
    const float m1 = ml[0], l1 = ml[64], top = fmaxf(m, m1);        // (a query sees itself: top is a number)
    const float f0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - top), f1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - top);
    float total = l * f0 + l1 * f1;
    if (a.sink) total += __builtin_amdgcn_exp2f(a.sink[head] * 1.4426950408889634f - top);      // a term of the denominator without a key
    float inv = 1.f / total;
    if (a.gate) inv *= sigmoid_fast(a.gate[(size_t)token * a.ldg + head]);
    bf16_t* dst = a.out + (size_t)token * a.H * DV + head * DV + 4 * half;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) {                               // channels 32 d + 8 i + 4 half .. + 3
            const f32x4_t p = parts[(d * 4 + i) * 64];
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (o[d][4 * i + j] * f0 + p[j] * f1) * inv;
            *(uint2*)(dst + 32 * d + 8 * i) = uint2{pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3])};
        }
}

// Rows first .. first + count - 1 of request s (positions), of which those from `lo` to `hi` are in the cache; the others, and what
// count leaves over, are zeros: latent [count, Lk] and shared channels [count, Dr] of the rows of the pool [slots, Lk + Dr].
__global__ __launch_bounds__(256) void latent_rows_kernel(const bf16_t* __restrict__ pool, const int* __restrict__ table, int page, int first,
                                                          int count, int lo, int hi, int Lk, int Dr, bf16_t* __restrict__ latent,
                                                          bf16_t* __restrict__ shared) {
    const int pieces = (Lk + Dr) / 8;
    const int idx = blockIdx.x * 256 + threadIdx.x, row = idx / pieces, p = idx - row * pieces;
    if (row >= count) return;
    const int pos = first + row;
    u32x4_t v = {0, 0, 0, 0};
    if (pos >= lo && pos <= hi) v = *(const u32x4_t*)(pool + ((size_t)table[pos / page] * page + pos % page) * (Lk + Dr) + 8 * p);
    *(u32x4_t*)(8 * p < Lk ? latent + (size_t)row * Lk + 8 * p : shared + (size_t)row * Dr + 8 * p - Lk) = v;
}

static bool ah_aligned(const void* p) { return p && ((uintptr_t)p % 16) == 0; }

extern "C" int tm_latent_rows(const void* pool, const int* table, int table_width, int page, int first, int count, int lo, int hi, int Lk, int Dr,
                              void* latent, void* shared, hipStream_t stream) {
    if (count <= 0) return TM_OK;
    if (!ah_aligned(pool) || !table || page <= 0 || first < 0 || lo < 0 || (hi >= lo && hi / page >= table_width) || Lk <= 0 || Lk % 8 || Dr < 0 || Dr % 8 ||
        !ah_aligned(latent) || (Dr && !ah_aligned(shared)) || (long long)count * ((Lk + Dr) / 8) > 0x7fffff00LL)
        return TM_ERR_ARG;
    const unsigned blocks = (unsigned)(((long long)count * ((Lk + Dr) / 8) + 255) / 256);
    latent_rows_kernel<<<blocks, 256, 0, stream>>>((const bf16_t*)pool, table, page, first, count, lo, hi, Lk, Dr, (bf16_t*)latent, (bf16_t*)shared);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// Head sizes there are kernels for: 128 + 64 (shared) and 128, 64 + 32 and 64.
extern "C" int tm_attn_heads_takes(int Dn, int Dr, int Dv) { return (Dn == 128 && Dr == 64 && Dv == 128) || (Dn == 64 && Dr == 32 && Dv == 64); }

template <int DN, int DR, int DV>
static int ah_launch(const HeadsArgs& a, int n_blocks, hipStream_t stream) {
    constexpr int lds = 2 * (64 * (DN + DR) * 2 + DV * 128);        // two buffers: 81,920 or 40,960 bytes
    static_assert(2 * (DV / 32 * 4096 + 512) <= lds, "");
    static const hipError_t raised = hipFuncSetAttribute((const void*)attn_heads_kernel<DN, DR, DV>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (raised != hipSuccess) return TM_ERR_LAUNCH;
    attn_heads_kernel<DN, DR, DV><<<n_blocks * a.H, 256, lds, stream>>>(a);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// out[t, h DV + c] (times sigmoid(gate[t, h])) for the queries that `blocks` names: entries (first row, queries, position of the first, kv
// row of position 0). kv: keys [R, H Dn] and behind them the shared channels [R, Dr]; vt [H Dv, R]; R a multiple of 64, rows that
// exist for every block of 64 keys a query's window touches.
extern "C" int tm_attn_heads(const void* q, int ldq, const void* qr, const void* kv, const void* vt, void* out, const int* blocks, int n_blocks,
                             const float* gate, int ldg, const float* sink, int H, int Dn, int Dr, int Dv, int R, float scale, int window,
                             hipStream_t stream) {
    if (n_blocks <= 0) return TM_OK;
    if (!tm_attn_heads_takes(Dn, Dr, Dv) || H <= 0 || R <= 0 || R % 64 || window < 0 || !(scale > 0.f) || !blocks || ldq < H * (Dn + Dr) || ldq % 8 ||
        !ah_aligned(q) || !ah_aligned(qr) || !ah_aligned(kv) || !ah_aligned(vt) || !ah_aligned(out) || (gate && ldg < H) ||
        (long long)R * (H * Dn + Dr) * 2 >= (1ll << 32) || (long long)H * Dv * R * 2 >= (1ll << 32) || (long long)n_blocks * H > 0xffffff)
        return TM_ERR_ARG;
    HeadsArgs a{(const bf16_t*)q, (const bf16_t*)qr, (const bf16_t*)kv, (const bf16_t*)vt, (bf16_t*)out, blocks, gate, sink,
                (uint32_t)((long long)R * H * Dn * 2), ldq, ldg, H, R, window, scale * 1.4426950408889634f};
    return Dn == 128 ? ah_launch<128, 64, 128>(a, n_blocks, stream) : ah_launch<64, 32, 64>(a, n_blocks, stream);
}
