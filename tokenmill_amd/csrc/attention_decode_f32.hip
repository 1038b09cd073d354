// Attention of single tokens of the true 32-bit path, on the 32-bit matrix unit: a block takes one request, one kv head and, one
// after the other, every gridDim.z-th chunk of TM_DECODE_F32_CHUNK keys, its four wavefronts every fourth block of 16 keys; the query heads of the kv head are the columns of the matrix
// instruction, so a key and a value are read once for all of them. The chunks' partial results (maximum, sum, weighted values)
// meet in a second kernel, in the order of the chunks.
//   scores S^T = K q^T: lane (r, g) holds K[key r][16 c + 4 g .. + 3] and q[head r][the same]; the result has key 4 g + i of head r
//   values O^T = V^T P^T: lane (r, g) holds V[d = 16 dt + r][key 4 g .. + 3]; the weights are where the scores were
//                               (formulas as in attention_generic.hip)
// The generic kernel gave a block a (token, head) pair, which read the 0.5B shape's keys once for each of the seven heads and
// walked 64 of them a wavefront: 29.9 us a layer for eight requests of 700 keys; this pair 10 us.
// The grid is bounded (tm_attn_decode_f32_blocks): a captured step asks for the longest context there can be, and of a block for
// each of its chunks next to all end at once. 64 / 95 requests of 300 keys under a limit of 32,768 tokens: 13.2 / 19.3 us with
// 32,768 / 48,640 blocks, 10.1 / 13.0 with 2,048 (a limit of 2,048: 10.1 / 13.2 either way); where every chunk has keys it is level
// (64 x 2,000 keys 26.5 and 26.9, 16 requests of 8 kv heads x 4,000 113.5 and 113.9; with 512 blocks 27.8 and 115.7).
#include "common.h"
#include "api.h"
#include "choose.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define DF_WAVES 4
#define DF_GRID 2048        // blocks a launch has at most, beyond one a (request, kv head) pair

template <int D>
__global__ __launch_bounds__(64 * DF_WAVES) void attn_decode_f32_kernel(const float* __restrict__ q, int q_stride,
                                                                        const float* __restrict__ k_pool, const float* __restrict__ v_pool,
                                                                        const int* __restrict__ block_tables, int table_width,
                                                                        const int* __restrict__ context_lens, float* __restrict__ part_o,
                                                                        float* __restrict__ part_ml, int max_chunks, int H, int KVH,
                                                                        int page_shift, float scale, int window, int keep, float softcap) {
    constexpr int DQ = D / 4, NDT = D / 16;
    __shared__ float m_s[DF_WAVES][16], l_s[DF_WAVES][16];
    __shared__ __attribute__((aligned(16))) float o_s[DF_WAVES][16][D + 4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int s = blockIdx.x, kvh = blockIdx.y, G = H / KVH;
    const int last = context_lens[s] - 1;                               // the token's own position, the newest key
    const int lo = (window > 0 && last - window + 1 > 0) ? last - window + 1 : 0;
    if ((int)blockIdx.z * TM_DECODE_F32_CHUNK > last) return;
    const int* table = block_tables + (size_t)s * table_width;
    const int page = 1 << page_shift;
    const float* qrow = q + (size_t)s * q_stride + (size_t)(kvh * G + (r < G ? r : G - 1)) * D + 4 * g;
    f32x4_t qf[NDT];
#pragma unroll
    for (int c = 0; c < NDT; ++c) qf[c] = *(const f32x4_t*)(qrow + 16 * c);
    constexpr int BLOCKS = TM_DECODE_F32_CHUNK / 16 / DF_WAVES;         // blocks of 16 keys a wavefront has: all asked for at once
    for (int chunk = blockIdx.z; chunk < max_chunks; chunk += gridDim.z) {      // (the same for the whole block)
        const int first = chunk * TM_DECODE_F32_CHUNK;
        if (first > last) return;
        // chunks without a key that is seen are not looked at by the second kernel either
        if (first + TM_DECODE_F32_CHUNK <= lo && first >= keep) continue;
        f32x4_t kf[BLOCKS][NDT], vf[BLOCKS][NDT];
        int key0[BLOCKS];
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            key0[b] = first + 16 * (wave + DF_WAVES * b);
            const int at = key0[b] <= last ? key0[b] : (last & ~15);        // (beyond the newest key: its own block again, all masked)
            const int pg = table[at >> page_shift], in_page = at & (page - 1);
            const float* kr = k_pool + ((((size_t)pg << page_shift) + in_page + r) * KVH + kvh) * D + 4 * g;
            const float* vr = v_pool + ((((size_t)pg * KVH + kvh) * D + r) << page_shift) + in_page + 4 * g;
#pragma unroll
            for (int c = 0; c < NDT; ++c) kf[b][c] = *(const f32x4_t*)(kr + 16 * c);
#pragma unroll
            for (int c = 0; c < NDT; ++c) vf[b][c] = *(const f32x4_t*)(vr + ((size_t)(16 * c) << page_shift));
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x4_t sc[BLOCKS];
        float m = -INFINITY;
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            sc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NDT; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][c][e], qf[c][e], sc[b], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = key0[b] + 4 * g + i;
                float v = sc[b][i] * scale;
                if (softcap > 0.f) v = softcap * tanhf(v / softcap);
                const bool seen = k <= last && (k >= lo || k < keep);
                sc[b][i] = seen ? v : -INFINITY;
                m = fmaxf(m, sc[b][i]);
                if (!seen)                                                  // values of keys nobody sees can hold anything
#pragma unroll
                    for (int c = 0; c < NDT; ++c) vf[b][c][i] = 0.f;
            }
        }
        m = lane_max<16>(m);
        m = lane_max<32>(m);
        const float ref = m == -INFINITY ? 0.f : m;                         // (a wavefront whose keys nobody sees: weights of zero)
        float l = 0.f;
        f32x4_t o[NDT];
#pragma unroll
        for (int c = 0; c < NDT; ++c) o[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < BLOCKS; ++b) {
            f32x4_t pr;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pr[i] = expf(sc[b][i] - ref);
                l += pr[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < NDT; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][c][i], pr[i], o[c], 0, 0, 0);
        }
        l = lane_sum<16>(l);
        l = lane_sum<32>(l);
        __syncthreads();                                                // (the sums of the chunk before have been read)
        if (g == 0) {
            m_s[wave][r] = m;
            l_s[wave][r] = l;
        }
#pragma unroll
        for (int c = 0; c < NDT; ++c) *(f32x4_t*)&o_s[wave][r][16 * c + 4 * g] = o[c];
        __syncthreads();
        const int col = threadIdx.x >> 4, part = threadIdx.x & 15;          // sixteen threads a head
        if (col >= G) continue;
        float top = -INFINITY, w[DF_WAVES], sum = 0.f;
#pragma unroll
        for (int v = 0; v < DF_WAVES; ++v) top = fmaxf(top, m_s[v][col]);
#pragma unroll
        for (int v = 0; v < DF_WAVES; ++v) {
            w[v] = m_s[v][col] == -INFINITY ? 0.f : expf(m_s[v][col] - top);
            sum += l_s[v][col] * w[v];
        }
        const size_t at = ((size_t)s * H + kvh * G + col) * max_chunks + chunk;
        if (part == 0) {
            part_ml[2 * at] = top;
            part_ml[2 * at + 1] = sum;
        }
        for (int d = 4 * part; d < D; d += 64) {
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < DF_WAVES; ++v) acc += *(const f32x4_t*)&o_s[v][col][d] * w[v];
            *(f32x4_t*)(part_o + at * D + d) = acc;
        }
    }
}

__global__ __launch_bounds__(64 * DF_WAVES) void attn_decode_f32_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                              const int* __restrict__ context_lens, float* __restrict__ out,
                                                                              int out_stride, int max_chunks, int H, int D, int window, int keep,
                                                                              const float* __restrict__ sink, const float* __restrict__ cgate,
                                                                              int ldcg) {
    __shared__ float s_l[DF_WAVES], s_o[DF_WAVES][128];
    const int s = blockIdx.x, h = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const size_t base = ((size_t)s * H + h) * max_chunks;
    const int last = context_lens[s] - 1;
    const int lo = (window > 0 && last - window + 1 > 0) ? last - window + 1 : 0;
    const int n = last / TM_DECODE_F32_CHUNK + 1 < max_chunks ? last / TM_DECODE_F32_CHUNK + 1 : max_chunks;
    auto seen = [&](int c) { return c < n && ((c + 1) * TM_DECODE_F32_CHUNK > lo || c * TM_DECODE_F32_CHUNK < keep); };
    float mm = -INFINITY;
    for (int c = lane; c < n; c += TM_WAVE)
        if (seen(c)) mm = fmaxf(mm, part_ml[2 * (base + c)]);
    mm = wave_max(mm);
    const int d0 = lane < D ? lane : D - 1, d1 = lane + 64 < D ? lane + 64 : D - 1;
    float ll = 0.f, o0 = 0.f, o1 = 0.f;
    for (int c0 = wave; c0 < n; c0 += 4 * DF_WAVES) {                   // four chunks asked for at a time
        float mc[4], lc[4], a0[4], a1[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = c0 + DF_WAVES * i < n ? c0 + DF_WAVES * i : n - 1;
            mc[i] = part_ml[2 * (base + c)];
            lc[i] = part_ml[2 * (base + c) + 1];
            a0[i] = part_o[(base + c) * D + d0];
            a1[i] = part_o[(base + c) * D + d1];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!seen(c0 + DF_WAVES * i)) continue;                     // (what was read there is whatever the memory held)
            const float f = expf(mc[i] - mm);
            ll = fmaf(lc[i], f, ll);
            o0 = fmaf(a0[i], f, o0);
            o1 = fmaf(a1[i], f, o1);
        }
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
    for (int w = 1; w < DF_WAVES; ++w) {
        ll += s_l[w];
        o0 += s_o[w][lane];
        o1 += s_o[w][lane + 64];
    }
    if (sink) ll += expf(sink[h] - mm);                                 // a term of the denominator without a key
    const float* gp = cgate ? cgate + (size_t)s * ldcg + (size_t)h * D : nullptr;      // a gate per channel
    auto gated = [&](float v, int d) { return gp ? v / (1.f + expf(-gp[d])) : v; };
    float* orow = out + (size_t)s * out_stride + (size_t)h * D;
    if (lane < D) orow[lane] = gated(o0 / ll, lane);
    if (lane + 64 < D) orow[lane + 64] = gated(o1 / ll, lane + 64);
}

// Blocks of the grid for a (request, kv head) pair: the chunks there can be, at most as many as give the chip eight blocks a CU.
extern "C" int tm_attn_decode_f32_blocks(int S, int KVH, int max_chunks) {
    const long long pairs = (long long)S * KVH;
    const long long most = (DF_GRID + pairs - 1) / pairs;
    return most < max_chunks ? (int)most : max_chunks;
}

// As tm_attn_decode_mfma_cap, in 32-bit: q, out and pools float32; head sizes 32, 64 and 128, at most 16 query heads a kv
// head; part_o [S, H, max_chunks, D] and part_ml [S, H, max_chunks, 2] are scratch, chunks of TM_DECODE_F32_CHUNK keys.
extern "C" int tm_attn_decode_f32_takes(const void* q, int q_stride, const void* k_pool, const void* v_pool, int H, int KVH, int D, int page) {
    auto whole = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
    return H > 0 && KVH > 0 && H % KVH == 0 && H / KVH <= 16 && KVH <= 65535 && (D == 32 || D == 64 || D == 128) && page >= 16 && (page & (page - 1)) == 0 &&
           q_stride % 4 == 0 && q_stride >= H * D && whole(q) && whole(k_pool) && whole(v_pool);
}

extern "C" int tm_attn_decode_f32(const float* q, int q_stride, float* out, int out_stride, const float* k_pool, const float* v_pool,
                                  const int* block_tables, int table_width, const int* context_lens, float* part_o, float* part_ml,
                                  int max_chunks, int S, int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                                  const float* sink, const float* cgate, int ldcg, hipStream_t stream) {
    if (S <= 0) return TM_OK;
    if (window == 0) keep = 0;
    if (!tm_attn_decode_f32_takes(q, q_stride, k_pool, v_pool, H, KVH, D, page) || !out || out_stride < H * D || !part_o || !part_ml ||
        ((uintptr_t)part_o % 16) || max_chunks <= 0 || max_chunks > 65535 || table_width <= 0 || window < 0 || keep < 0 || !(softcap >= 0.f) ||
        (cgate && ldcg < H * D))
        return TM_ERR_ARG;
    int shift = 0;
    while ((1 << shift) < page) ++shift;
    const dim3 grid(S, KVH, tm_attn_decode_f32_blocks(S, KVH, max_chunks));
#define DF_GO(D_)                                                                                                                          \
    case D_:                                                                                                                               \
        attn_decode_f32_kernel<D_><<<grid, 64 * DF_WAVES, 0, stream>>>(q, q_stride, k_pool, v_pool, block_tables, table_width, context_lens, part_o, \
                                                                       part_ml, max_chunks, H, KVH, shift, scale, window, keep, softcap);   \
        break
    switch (D) {
        DF_GO(32);
        DF_GO(64);
        DF_GO(128);
    }
#undef DF_GO
    TM_CHECK_LAUNCH();
    attn_decode_f32_merge_kernel<<<dim3(S, H), 64 * DF_WAVES, 0, stream>>>(part_o, part_ml, context_lens, out, out_stride, max_chunks, H, D, window,
                                                                           keep, sink, cgate, ldcg);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
