// Layer norm with weight and bias behind a gated, scaled residual add; a short causal convolution over time with
// per-request state; and the PolyNorm activation. Everything is computed in 32-bit and rounded once where stored.
//
//   tm_layer_norm      v = resid[r] + mult * y[r] * sigmoid(gate[r])    (gate null: no gate; y null: v = resid[r])
//                      resid[r] = v                                     (only with y, and only when every row is run)
//                      out[r] = (v - mean(v)) / sqrt(mean((v - mean(v))^2) + eps) * w + b      (out null: the add alone)
//                      rows != null: row rows[r] of resid, y and gate is read, nothing is written back, out row r.
//   tm_short_conv      out[t] = h[t] + sum_j w[:, j] * h[t - taps + 1 + j], the rows before a request's first row of the
//                      step taken from its state [taps - 1, width] (zeros at a sequence's start);
//   tm_short_conv_state  then the state becomes the last taps - 1 rows the request has seen.
//   tm_short_conv_walk   both in one launch, for steps whose requests bring few rows each; the same bits.
//   tm_poly_norm       out = a N(z) + b N(z^2) + c N(z^3) + e, N(v) = v / sqrt(mean(v^2) + eps) over a row, powers by element.
#include "common.h"
#include "api.h"

#define LN_THREADS 256

template <typename T>
__global__ __launch_bounds__(LN_THREADS) void layer_norm_kernel(float* __restrict__ resid, const T* __restrict__ y,
                                                                const T* __restrict__ gate, float mult,
                                                                const int* __restrict__ rows, const float* __restrict__ w,
                                                                const float* __restrict__ b, T* __restrict__ out, int hidden,
                                                                float eps) {
    extern __shared__ float row_s[];
    __shared__ float red[LN_THREADS / TM_WAVE];
    const int r = blockIdx.x;
    const size_t src = (size_t)(rows ? rows[r] : r) * hidden;
    float sum = 0.f;
    for (int c = threadIdx.x; c < hidden; c += LN_THREADS) {
        float v = resid[src + c];
        if (y) {
            float d = Elem<T>::load(y + src + c);
            if (gate) d *= 1.0f / (1.0f + __expf(-Elem<T>::load(gate + src + c)));
            v += mult * d;
            if (!rows) resid[src + c] = v;
        }
        row_s[c] = v;
        sum += v;
    }
    if (!out) return;
    const float mean = block_sum<LN_THREADS>(sum, red) / (float)hidden;
    float ss = 0.f;
    for (int c = threadIdx.x; c < hidden; c += LN_THREADS) {
        const float d = row_s[c] - mean;
        ss += d * d;
    }
    const float inv = 1.0f / sqrtf(block_sum<LN_THREADS>(ss, red) / (float)hidden + eps);
    T* o = out + (size_t)r * hidden;
    for (int c = threadIdx.x; c < hidden; c += LN_THREADS)
        Elem<T>::store(o + c, (row_s[c] - mean) * inv * w[c] + b[c]);
}

// eight values, 16-byte aligned, as 32-bit floats
__device__ __forceinline__ void ln_load8(const float* p, float* v) {
    Piece<float>::unpack(*(const uint4*)p, v);
    Piece<float>::unpack(*(const uint4*)(p + 4), v + 4);
}
__device__ __forceinline__ void ln_load8(const bf16_t* p, float* v) { Piece<bf16_t>::unpack(*(const uint4*)p, v); }
__device__ __forceinline__ void ln_store8(float* p, const float* v) {
    *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void ln_store8(bf16_t* p, const float* v) {
    uint4 u;
    u.x = (uint32_t)f32_to_bf16(v[0]) | (uint32_t)f32_to_bf16(v[1]) << 16;
    u.y = (uint32_t)f32_to_bf16(v[2]) | (uint32_t)f32_to_bf16(v[3]) << 16;
    u.z = (uint32_t)f32_to_bf16(v[4]) | (uint32_t)f32_to_bf16(v[5]) << 16;
    u.w = (uint32_t)f32_to_bf16(v[6]) | (uint32_t)f32_to_bf16(v[7]) << 16;
    *(uint4*)p = u;
}

// The same with rows of whole pieces of eight, all of a row in registers (PIECES of a thread, 256 apart) and every load of it in
// flight at once, weight and bias among them: bound by memory (rows of 2,048 with a gate move 18 KB each).
template <typename T, int PIECES>
__global__ __launch_bounds__(LN_THREADS) void layer_norm_pieces_kernel(float* __restrict__ resid, const T* __restrict__ y,
                                                                       const T* __restrict__ gate, float mult,
                                                                       const int* __restrict__ rows, const float* __restrict__ w,
                                                                       const float* __restrict__ b, T* __restrict__ out, int hidden,
                                                                       float eps) {
    __shared__ float red[LN_THREADS / TM_WAVE];
    const int r = blockIdx.x;
    const size_t src = (size_t)(rows ? rows[r] : r) * hidden;
    float v[PIECES][8];
    float sum = 0.f;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int c = (p * LN_THREADS + (int)threadIdx.x) * 8;
        if (c >= hidden) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[p][e] = 0.f;
            continue;
        }
        ln_load8(resid + src + c, v[p]);
        if (y) {
            float d[8], g[8];
            ln_load8(y + src + c, d);
            if (gate) {
                ln_load8(gate + src + c, g);
#pragma unroll
                for (int e = 0; e < 8; ++e) d[e] *= 1.0f / (1.0f + __expf(-g[e]));
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[p][e] += mult * d[e];
            if (!rows) ln_store8(resid + src + c, v[p]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += v[p][e];
    }
    if (!out) return;
    const float mean = block_sum<LN_THREADS>(sum, red) / (float)hidden;
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
        if ((p * LN_THREADS + (int)threadIdx.x) * 8 < hidden)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float d = v[p][e] - mean;
                ss += d * d;
            }
    const float inv = 1.0f / sqrtf(block_sum<LN_THREADS>(ss, red) / (float)hidden + eps);
    T* o = out + (size_t)r * hidden;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int c = (p * LN_THREADS + (int)threadIdx.x) * 8;
        if (c >= hidden) continue;
        float wv[8], bv[8];
        ln_load8(w + c, wv);
        ln_load8(b + c, bv);
#pragma unroll
        for (int e = 0; e < 8; ++e) wv[e] = (v[p][e] - mean) * inv * wv[e] + bv[e];
        ln_store8(o + c, wv);
    }
}

// Rows of whole pieces on 16-byte boundaries take the kernel above, of up to 8,192 values (four pieces of a thread in registers);
// the rest keep their row in LDS, a value at a time. 1,500 rows of 2,048 in bfloat16 behind a gated add: 16.7 us a value at a
// time, 10.4 us in pieces.
template <typename T>
static void layer_norm_go(float* resid, const T* y, const T* gate, float mult, const int* rows, const float* w, const float* b, T* out,
                          int R, int hidden, float eps, hipStream_t stream) {
    auto whole = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
    if (hidden % 8 == 0 && hidden <= 4 * LN_THREADS * 8 && whole(resid) && whole(y) && whole(gate) && whole(w) && whole(b) && whole(out)) {
        if (hidden <= LN_THREADS * 8)
            layer_norm_pieces_kernel<T, 1><<<R, LN_THREADS, 0, stream>>>(resid, y, gate, mult, rows, w, b, out, hidden, eps);
        else if (hidden <= 2 * LN_THREADS * 8)
            layer_norm_pieces_kernel<T, 2><<<R, LN_THREADS, 0, stream>>>(resid, y, gate, mult, rows, w, b, out, hidden, eps);
        else
            layer_norm_pieces_kernel<T, 4><<<R, LN_THREADS, 0, stream>>>(resid, y, gate, mult, rows, w, b, out, hidden, eps);
        return;
    }
    layer_norm_kernel<T><<<R, LN_THREADS, (size_t)hidden * sizeof(float), stream>>>(resid, y, gate, mult, rows, w, b, out, hidden, eps);
}

extern "C" int tm_layer_norm(float* resid, const void* y, const void* gate, float mult, const int* rows, const float* w,
                             const float* b, void* out, int dtype, int R, int hidden, float eps, hipStream_t stream) {
    if (!resid || R < 0 || hidden <= 0 || hidden > 16384 || (gate && !y) || (out && (!w || !b)) || !(eps > 0.f)) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (R == 0 || (!y && !out)) return TM_OK;
    if (dtype == TM_F32)
        layer_norm_go<float>(resid, (const float*)y, (const float*)gate, mult, rows, w, b, (float*)out, R, hidden, eps, stream);
    else
        layer_norm_go<bf16_t>(resid, (const bf16_t*)y, (const bf16_t*)gate, mult, rows, w, b, (bf16_t*)out, R, hidden, eps, stream);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ------------------------------------------------------------------------------------------------ short convolution

#define SC_THREADS 256
#define SC_MAX_TAPS 16

// sum_j w[j] * x[j], j ascending, every product and sum rounded on its own: the two kernels below give the same bits
// (MAXT: the most taps the instantiation takes; the sum is the same sequence of operations at every MAXT)
template <int MAXT>
__device__ __forceinline__ float tap_sum(const float (&wv)[MAXT], const float (&xv)[MAXT], int taps) {
#pragma clang fp contract(off)
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < MAXT; ++j)
        if (j < taps) acc += wv[j] * xv[j];
    return acc;
}

template <typename T, int MAXT>
__global__ __launch_bounds__(SC_THREADS) void short_conv_kernel(const T* __restrict__ h, T* __restrict__ out,
                                                                const T* __restrict__ w, const T* __restrict__ state,
                                                                const int* __restrict__ cu, const int* __restrict__ slots,
                                                                const int* __restrict__ seq_of_token, int width, int taps) {
    const int t = blockIdx.x;
    const int s = seq_of_token[t];
    const int first = cu[s];
    const int i = t - first;                                 // the token's place among its request's rows of this step
    const T* st = state + (size_t)slots[s] * (taps - 1) * width;
    for (int c = blockIdx.y * SC_THREADS + threadIdx.x; c < width; c += gridDim.y * SC_THREADS) {
        float wv[MAXT], xv[MAXT];
#pragma unroll
        for (int j = 0; j < MAXT; ++j) {
            wv[j] = xv[j] = 0.f;
            if (j < taps) {
                const int at = i - (taps - 1) + j;           // < 0: before this step's rows, in the state
                xv[j] = at >= 0 ? Elem<T>::load(h + (size_t)(first + at) * width + c)
                                : Elem<T>::load(st + (size_t)(taps - 1 + at) * width + c);
                wv[j] = Elem<T>::load(w + (size_t)c * taps + j);
            }
        }
        Elem<T>::store(out + (size_t)t * width + c, Elem<T>::load(h + (size_t)t * width + c) + tap_sum<MAXT>(wv, xv, taps));
    }
}

// The same for up to four taps over rows of whole pieces of eight on 16-byte boundaries: a thread takes eight channels of a token,
// a wavefront's rows and weights come in whole lines. 1,500 rows of 2,048 in bfloat16, four taps: 17.1 us a channel at a time,
// 7.4 us in pieces (12 MB to read and write; the rows before a token come out of the caches). More taps stay
// a channel a thread. The same bits.
template <typename T, int TAPS>
__global__ __launch_bounds__(SC_THREADS) void short_conv_pieces_kernel(const T* __restrict__ h, T* __restrict__ out,
                                                                       const T* __restrict__ w, const T* __restrict__ state,
                                                                       const int* __restrict__ cu, const int* __restrict__ slots,
                                                                       const int* __restrict__ seq_of_token, int tokens, int width) {
    const int pieces = width / 8;
    const long long at = (long long)blockIdx.x * SC_THREADS + threadIdx.x;
    const int t = (int)(at / pieces), c = (int)(at % pieces) * 8;
    if (t >= tokens) return;
    const int s = seq_of_token[t], first = cu[s], i = t - first;
    const T* st = TAPS > 1 ? state + (size_t)slots[s] * (TAPS - 1) * width : state;
    float x[TAPS][8], wv[8 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        const int from = i - (TAPS - 1) + j;                 // < 0: before this step's rows, in the state
        ln_load8((from >= 0 ? h + (size_t)(first + from) * width : st + (size_t)(TAPS - 1 + from) * width) + c, x[j]);
        ln_load8(w + (size_t)c * TAPS + 8 * j, wv + 8 * j);
    }
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float we[TAPS], xe[TAPS];
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            we[j] = wv[e * TAPS + j];
            xe[j] = x[j][e];
        }
        o[e] = x[TAPS - 1][e] + tap_sum<TAPS>(we, xe, TAPS);
    }
    ln_store8(out + (size_t)t * width + c, o);
}

// The same for steps whose requests bring few rows each (single tokens): a thread takes a channel of a request, walks the
// request's rows with the window of the last taps rows in registers, and leaves the new state behind: one launch.
template <typename T, int MAXT>
__global__ __launch_bounds__(SC_THREADS) void short_conv_walk_kernel(const T* __restrict__ h, T* __restrict__ out,
                                                                     const T* __restrict__ w, T* __restrict__ state,
                                                                     const int* __restrict__ cu, const int* __restrict__ slots,
                                                                     int width, int taps) {
    const int s = blockIdx.x;
    const int first = cu[s], n = cu[s + 1] - first;
    if (n <= 0) return;
    T* st = state + (size_t)slots[s] * (taps - 1) * width;
    for (int c = blockIdx.y * SC_THREADS + threadIdx.x; c < width; c += gridDim.y * SC_THREADS) {
        float wv[MAXT], xv[MAXT];
#pragma unroll
        for (int j = 0; j < MAXT; ++j) {
            wv[j] = j < taps ? Elem<T>::load(w + (size_t)c * taps + j) : 0.f;
            xv[j] = j < taps - 1 ? Elem<T>::load(st + (size_t)j * width + c) : 0.f;
        }
        for (int i = 0; i < n; ++i) {
            const float cur = Elem<T>::load(h + (size_t)(first + i) * width + c);
#pragma unroll
            for (int j = 0; j < MAXT; ++j)
                if (j == taps - 1) xv[j] = cur;
            Elem<T>::store(out + (size_t)(first + i) * width + c, cur + tap_sum<MAXT>(wv, xv, taps));
#pragma unroll
            for (int j = 0; j + 1 < MAXT; ++j)
                if (j < taps - 1) xv[j] = xv[j + 1];
        }
#pragma unroll
        for (int j = 0; j < MAXT; ++j)
            if (j < taps - 1) Elem<T>::store(st + (size_t)j * width + c, xv[j]);
    }
}

template <typename T>
__global__ __launch_bounds__(SC_THREADS) void short_conv_state_kernel(const T* __restrict__ h, T* __restrict__ state,
                                                                      const int* __restrict__ cu, const int* __restrict__ slots,
                                                                      int width, int taps) {
    const int s = blockIdx.x;
    const int first = cu[s], n = cu[s + 1] - first;
    if (n <= 0) return;
    T* st = state + (size_t)slots[s] * (taps - 1) * width;
    const int keep = taps - 1;
    for (int c = blockIdx.y * SC_THREADS + threadIdx.x; c < width; c += gridDim.y * SC_THREADS) {
        T next[SC_MAX_TAPS - 1];
        for (int k = 0; k < keep; ++k) {
            const int at = n - keep + k;                     // the row that becomes state row k
            next[k] = at >= 0 ? h[(size_t)(first + at) * width + c] : st[(size_t)(keep + at) * width + c];
        }
        for (int k = 0; k < keep; ++k) st[(size_t)k * width + c] = next[k];
    }
}

extern "C" int tm_short_conv(const void* h, void* out, const void* w, const void* state, const int* cu_q_lens,
                             const int* state_slots, const int* seq_of_token, int T, int width, int taps, int dtype,
                             hipStream_t stream) {
    if (!h || !out || !w || T < 0 || width <= 0 || taps < 1 || taps > SC_MAX_TAPS || (taps > 1 && !state)) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (T == 0) return TM_OK;
    auto whole = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
    const long long blocks = ((long long)T * (width / 8) + SC_THREADS - 1) / SC_THREADS;
    if (taps <= 4 && width % 8 == 0 && blocks < (1ll << 31) && whole(h) && whole(out) && whole(w) && whole(state)) {
#define SC_GO(T_, TAPS_)                                                                                                  \
    short_conv_pieces_kernel<T_, TAPS_><<<(int)blocks, SC_THREADS, 0, stream>>>((const T_*)h, (T_*)out, (const T_*)w, (const T_*)state, \
                                                                                cu_q_lens, state_slots, seq_of_token, T, width)
        if (dtype == TM_F32) {
            if (taps == 1) SC_GO(float, 1); else if (taps == 2) SC_GO(float, 2); else if (taps == 3) SC_GO(float, 3); else SC_GO(float, 4);
        } else {
            if (taps == 1) SC_GO(bf16_t, 1); else if (taps == 2) SC_GO(bf16_t, 2); else if (taps == 3) SC_GO(bf16_t, 3); else SC_GO(bf16_t, 4);
        }
#undef SC_GO
        TM_CHECK_LAUNCH();
        return TM_OK;
    }
    dim3 grid(T, (width + SC_THREADS - 1) / SC_THREADS > 8 ? 8 : (width + SC_THREADS - 1) / SC_THREADS);
#define SC_GO(T_, MAXT_)                                                                                                  \
    short_conv_kernel<T_, MAXT_><<<grid, SC_THREADS, 0, stream>>>((const T_*)h, (T_*)out, (const T_*)w, (const T_*)state, cu_q_lens, \
                                                                  state_slots, seq_of_token, width, taps)
    if (dtype == TM_F32) {
        if (taps <= 4) SC_GO(float, 4); else if (taps <= 8) SC_GO(float, 8); else SC_GO(float, SC_MAX_TAPS);
    } else {
        if (taps <= 4) SC_GO(bf16_t, 4); else if (taps <= 8) SC_GO(bf16_t, 8); else SC_GO(bf16_t, SC_MAX_TAPS);
    }
#undef SC_GO
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// tm_short_conv and tm_short_conv_state in one launch, for steps whose requests bring few rows each: the same bits.
extern "C" int tm_short_conv_walk(const void* h, void* out, const void* w, void* state, const int* cu_q_lens, const int* state_slots,
                                  int S, int width, int taps, int dtype, hipStream_t stream) {
    if (!h || !out || !w || S < 0 || width <= 0 || taps < 2 || taps > SC_MAX_TAPS || !state) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (S == 0) return TM_OK;
    dim3 grid(S, (width + SC_THREADS - 1) / SC_THREADS > 8 ? 8 : (width + SC_THREADS - 1) / SC_THREADS);
#define SC_GO(T_, MAXT_)                                                                                                       \
    short_conv_walk_kernel<T_, MAXT_><<<grid, SC_THREADS, 0, stream>>>((const T_*)h, (T_*)out, (const T_*)w, (T_*)state, cu_q_lens,     \
                                                                       state_slots, width, taps)
    if (dtype == TM_F32) {
        if (taps <= 4) SC_GO(float, 4); else if (taps <= 8) SC_GO(float, 8); else SC_GO(float, SC_MAX_TAPS);
    } else {
        if (taps <= 4) SC_GO(bf16_t, 4); else if (taps <= 8) SC_GO(bf16_t, 8); else SC_GO(bf16_t, SC_MAX_TAPS);
    }
#undef SC_GO
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_short_conv_state(const void* h, void* state, const int* cu_q_lens, const int* state_slots, int S, int width,
                                   int taps, int dtype, hipStream_t stream) {
    if (!h || S < 0 || width <= 0 || taps < 1 || taps > SC_MAX_TAPS || (taps > 1 && !state)) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (S == 0 || taps == 1) return TM_OK;
    dim3 grid(S, (width + SC_THREADS - 1) / SC_THREADS > 8 ? 8 : (width + SC_THREADS - 1) / SC_THREADS);
    if (dtype == TM_F32)
        short_conv_state_kernel<float><<<grid, SC_THREADS, 0, stream>>>((const float*)h, (float*)state, cu_q_lens, state_slots, width, taps);
    else
        short_conv_state_kernel<bf16_t><<<grid, SC_THREADS, 0, stream>>>((const bf16_t*)h, (bf16_t*)state, cu_q_lens, state_slots, width, taps);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ------------------------------------------------------------------------------------------------ PolyNorm

template <typename T>
__global__ __launch_bounds__(LN_THREADS) void poly_norm_kernel(const float* __restrict__ z, const float* __restrict__ coef,
                                                               T* __restrict__ out, int F, float eps) {
    __shared__ float red[LN_THREADS / TM_WAVE];
    const float* zr = z + (size_t)blockIdx.x * F;
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
    for (int c = threadIdx.x; c < F; c += LN_THREADS) {
        const float v = zr[c], v2 = v * v, v3 = v2 * v;
        s2 += v2;
        s4 += v2 * v2;
        s6 += v3 * v3;
    }
    const float r1 = 1.0f / sqrtf(block_sum<LN_THREADS>(s2, red) / (float)F + eps);
    const float r2 = 1.0f / sqrtf(block_sum<LN_THREADS>(s4, red) / (float)F + eps);
    const float r3 = 1.0f / sqrtf(block_sum<LN_THREADS>(s6, red) / (float)F + eps);
    const float a = coef[0], b = coef[1], c3 = coef[2], e = coef[3];
    T* o = out + (size_t)blockIdx.x * F;
    for (int c = threadIdx.x; c < F; c += LN_THREADS) {
        const float v = zr[c], v2 = v * v;
        Elem<T>::store(o + c, a * (v * r1) + b * (v2 * r2) + c3 * (v2 * v * r3) + e);
    }
}

extern "C" int tm_poly_norm(const float* z, const float* coef, void* out, int dtype, int T, int F, float eps,
                            hipStream_t stream) {
    if (!z || !coef || !out || T < 0 || F <= 0 || !(eps > 0.f)) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (T == 0) return TM_OK;
    if (dtype == TM_F32)
        poly_norm_kernel<float><<<T, LN_THREADS, 0, stream>>>(z, coef, (float*)out, F, eps);
    else
        poly_norm_kernel<bf16_t><<<T, LN_THREADS, 0, stream>>>(z, coef, (bf16_t*)out, F, eps);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
