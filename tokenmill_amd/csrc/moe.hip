// A feed-forward of many small experts of which every token uses a few, chosen by a table row of its token id or by a
// router.
//
//   pair p = (token t = p / top, choice k = p % top) goes to expert e(p) = table[id[t] * top + k]  (ids null: table[p])
//   tm_moe_router    z [T, E] (32-bit router outputs) -> s = softmax(z); the `top` largest of s + correction are chosen
//                    (ties: the lower index), chosen[t, k] in descending order, weight[t, k] = s / (sum of the chosen s + 1e-20);
//                    with `over_chosen` the `top` largest z are chosen and the weights are the softmax over the chosen z only;
//                    with `sigmoid` s = sigmoid(z), and the chosen s are the weights as they are
//   tm_moe_route     sorts the pairs by expert: slot_pair[slot] = p, pair_slot[p] = slot, and cuts every expert's run of
//                    slots into tiles of `tile_rows` rows: tiles[i] = (expert, first slot, rows), n_tiles[0] = their number
//   tm_moe_gate_up   act[slot] = silu(x[t] . Wg[e]^T) * (x[t] . Wu[e]^T)          W [E, 2F, K]: gate rows, then up rows
//   tm_moe_down      part[slot] = act[slot] . Wd[e]^T  (32-bit)                    Wd [E, N, F]
//   tm_moe_combine   y[t] = sum_k weight * part[pair_slot[t * top + k]], k ascending, rounded once
//   tm_moe_up_act    act[slot] = relu(x[t] . Wu[e]^T)^2                           W [E, F, K]: experts without a gate
//   tm_moe_clamped   act[slot] = g sigmoid(alpha g) (u + 1), g = min(z Wg[e] x[t], limit), u = z Wu[e] x[t] held to +-limit, with z the
//                    pair's weight (null: 1): an expert on its weighted input                 W [E, 2F, K]
//   tm_moe_combine_weighted   y[t] = sum_k weight[t, k] * (part[slot of the pair], or x[t] for a pair that has no slot: an
//                    expert >= `real` stands for the input itself; weight null: 1) + sigmoid(shared_gate[t]) * shared[t]
//
// All of it runs from device data (no count crosses to the host), so a step can be recorded into a graph. Which slot a
// pair gets inside its expert's run may differ from run to run (the cursor is an atomic counter); a row's result does not
// depend on its slot: every element is summed over k in ascending order by one thread.
#include "common.h"
#include "api.h"

#define MR_THREADS 1024
#define MOE_MAX_EXPERTS 1024
#define MR_FEW_EXPERTS 16

// One block, bound by its trips to memory (the token, its table row) and to LDS. A pair's expert and its place in the expert's run come
// from one pass: a thread asks for four pairs' tokens and then for their rows at once, the counter that counts a pair says its place,
// and both stay in registers (beyond 4,096 pairs: the place waits in pair_slot and the expert is read again). The runs are
// laid out by a scan with a thread an expert, the tiles written with a thread a tile. us where every pair was read and counted twice and one
// thread laid out runs and tiles / now: 1,500 tokens, 16 experts, top 2 7.7 / 5.3 (with the table out of HBM 10.3); 2,048, 64, 6
// 20.4 / 9.9; 64, 512, 8 38.0 / 4.8; 4,096, 1,000, 8 111 / 28.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void moe_route_kernel(const int* __restrict__ ids, const int* __restrict__ table, int T,
                                                               int top, int E, int real, int tile_rows, int* __restrict__ slot_pair,
                                                               int* __restrict__ pair_slot, int* __restrict__ tiles,
                                                               int* __restrict__ n_tiles) {
    constexpr int HOLD = 4, WAVES = THREADS / TM_WAVE;
    static_assert(THREADS % TM_WAVE == 0, "");
    __shared__ int cnt[THREADS], off[THREADS], tile0[THREADS + 1];
    __shared__ int wave_pairs[WAVES], wave_tiles[WAVES];
    const int P = T * top, tid = threadIdx.x, lane = tid % TM_WAVE, wave = tid / TM_WAVE;
    if (tid < E) cnt[tid] = 0;
    __syncthreads();
    auto experts = [&](int base, int (&e)[HOLD]) {                   // of pairs base + tid + i THREADS; beyond the last pair: none
        size_t row[HOLD];
#pragma unroll
        for (int i = 0; i < HOLD; ++i) {
            const int p = base + tid + i * THREADS, at = p < P ? p : 0;
            row[i] = ids ? (size_t)ids[at / top] * top + at % top : at;
        }
#pragma unroll
        for (int i = 0; i < HOLD; ++i) {
            const int p = base + tid + i * THREADS;
            e[i] = p < P ? table[row[i]] : MOE_MAX_EXPERTS;
        }
    };
    int held[HOLD], place[HOLD];
    for (int base = 0; base < P; base += HOLD * THREADS) {
        int e[HOLD];
        experts(base, e);
#pragma unroll
        for (int i = 0; i < HOLD; ++i) {
            const int p = base + tid + i * THREADS, at = e[i] < real ? atomicAdd(&cnt[e[i]], 1) : -1;
            if (base == 0) {
                held[i] = e[i];
                place[i] = at;
            } else if (p < P) {
                pair_slot[p] = at;
            }
        }
    }
    __syncthreads();
    const int pairs = tid < real ? cnt[tid] : 0, mine = (pairs + tile_rows - 1) / tile_rows;
    int pairs_to = pairs, tiles_to = mine;                           // inclusive sums over the experts
#pragma unroll
    for (int o = 1; o < TM_WAVE; o *= 2) {
        if (o >= real) break;                                        // (what lies beyond the last expert is not used)
        const int a = __shfl_up(pairs_to, o, TM_WAVE), b = __shfl_up(tiles_to, o, TM_WAVE);
        if (lane >= o) {
            pairs_to += a;
            tiles_to += b;
        }
    }
    if (lane == TM_WAVE - 1) {
        wave_pairs[wave] = pairs_to;
        wave_tiles[wave] = tiles_to;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
        pairs_to += wave_pairs[w];
        tiles_to += wave_tiles[w];
    }
    if (tid < real) {
        off[tid] = pairs_to - pairs;
        tile0[tid] = tiles_to - mine;
    }
    if (tid == (real > 0 ? real - 1 : 0)) tile0[real] = n_tiles[0] = tiles_to;
    __syncthreads();
    const int total = tile0[real];
    for (int i = tid; i < total; i += THREADS) {
        int e = 0, end = real;                                       // the last expert whose tiles start at or before tile i: it has tile i
        while (end - e > 1) {
            const int mid = (e + end) / 2;
            if (tile0[mid] <= i) e = mid;
            else end = mid;
        }
        const int from = (i - tile0[e]) * tile_rows;
        tiles[3 * i] = e;
        tiles[3 * i + 1] = off[e] + from;
        tiles[3 * i + 2] = min(tile_rows, cnt[e] - from);
    }
    for (int base = 0; base < P; base += HOLD * THREADS) {
        if (base != 0) {
            experts(base, held);
#pragma unroll
            for (int i = 0; i < HOLD; ++i) {
                const int p = base + tid + i * THREADS;
                place[i] = p < P ? pair_slot[p] : -1;                // (this thread's own store)
            }
        }
#pragma unroll
        for (int i = 0; i < HOLD; ++i) {
            const int p = base + tid + i * THREADS;
            if (p >= P) continue;
            if (held[i] >= real) {                                   // an expert without matrices: the pair has no slot
                pair_slot[p] = -1;
                continue;
            }
            const int slot = off[held[i]] + place[i];
            slot_pair[slot] = p;
            pair_slot[p] = slot;
        }
    }
}

// The same for few experts and pairs: in a step the launch finds its code out of the instruction cache, and this is a quarter of it (16 experts,
// top 2, 90 / 400 / 900 tokens between a layer's other launches, us: 4.2 / 5.2 / 7.3, the kernel above 5.2 / 6.0 / 7.4; at 1,500 10.3 / 9.3).
__global__ __launch_bounds__(MR_THREADS) void moe_route_few_kernel(const int* __restrict__ ids, const int* __restrict__ table, int T,
                                                                   int top, int E, int real, int tile_rows, int* __restrict__ slot_pair,
                                                                   int* __restrict__ pair_slot, int* __restrict__ tiles,
                                                                   int* __restrict__ n_tiles) {
    __shared__ int cnt[MR_FEW_EXPERTS];
    __shared__ int off[MR_FEW_EXPERTS + 1];
    const int P = T * top;
    for (int e = threadIdx.x; e < E; e += MR_THREADS) cnt[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < P; p += MR_THREADS) {
        const int e = ids ? table[(size_t)ids[p / top] * top + p % top] : table[p];
        if (e < real) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int at = 0, n = 0;
        for (int e = 0; e < real; ++e) {
            off[e] = at;
            for (int r = 0; r < cnt[e]; r += tile_rows) {
                tiles[3 * n] = e;
                tiles[3 * n + 1] = at + r;
                tiles[3 * n + 2] = min(tile_rows, cnt[e] - r);
                ++n;
            }
            at += cnt[e];
            cnt[e] = 0;
        }
        off[real] = at;
        n_tiles[0] = n;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < P; p += MR_THREADS) {
        const int e = ids ? table[(size_t)ids[p / top] * top + p % top] : table[p];
        if (e >= real) {                        // an expert without matrices: the pair has no slot
            pair_slot[p] = -1;
            continue;
        }
        const int slot = off[e] + atomicAdd(&cnt[e], 1);
        slot_pair[slot] = p;
        pair_slot[p] = slot;
    }
}

// Otherwise the fewest wavefronts that have a lane an expert and hold the pairs (8 tokens, 64 experts, top 8 in one 3.1 us, in 16 4.4; the one thread's runs and
// tiles 6.6, launched again and again). Between fifteen launches of other kernels, the code out of the second-level cache, the one thread's / this, us at 8 / 90 / 400
// tokens: 17 experts, top 2, 3.0 / 3.2, 3.5 / 3.4, 4.4 / 3.7, 24, 4, 4.1 / 3.2, 4.1 / 3.9, 6.6 / 4.1, 32, 2, 4.0 / 3.1, 4.7 / 3.1, 4.8 / 3.8, 64, 6, 6.6 / 3.2, 7.8 / 3.7, 10.9 / 4.6.
static int launch_moe_route(const int* ids, const int* table, int T, int top, int E, int real, int tile_rows, int* slot_pair, int* pair_slot,
                            int* tiles, int* n_tiles, hipStream_t stream) {
    static_assert(MOE_MAX_EXPERTS <= MR_THREADS, "");
    if (E <= MR_FEW_EXPERTS && T * top <= 2 * MR_THREADS)
        moe_route_few_kernel<<<1, MR_THREADS, 0, stream>>>(ids, table, T, top, E, real, tile_rows, slot_pair, pair_slot, tiles, n_tiles);
    else if (E <= TM_WAVE && T * top <= 4 * TM_WAVE)
        moe_route_kernel<TM_WAVE><<<1, TM_WAVE, 0, stream>>>(ids, table, T, top, E, real, tile_rows, slot_pair, pair_slot, tiles, n_tiles);
    else if (E <= 4 * TM_WAVE && T * top <= 16 * TM_WAVE)
        moe_route_kernel<4 * TM_WAVE><<<1, 4 * TM_WAVE, 0, stream>>>(ids, table, T, top, E, real, tile_rows, slot_pair, pair_slot, tiles, n_tiles);
    else
        moe_route_kernel<MR_THREADS><<<1, MR_THREADS, 0, stream>>>(ids, table, T, top, E, real, tile_rows, slot_pair, pair_slot, tiles, n_tiles);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ids null: table is [T, top], the experts of every pair as a router chose them. real: experts real .. E - 1 have no matrices.
extern "C" int tm_moe_route_chosen(const int* ids, const int* table, int T, int top, int E, int real, int tile_rows, int* slot_pair,
                                   int* pair_slot, int* tiles, int* n_tiles, hipStream_t stream) {
    if (!table || !slot_pair || !pair_slot || !tiles || !n_tiles || T < 0 || top <= 0 || E <= 0 || E > MOE_MAX_EXPERTS || real < 0 ||
        real > E || tile_rows <= 0 || (long long)T * top > 0x3fffffffLL)
        return TM_ERR_ARG;
    return launch_moe_route(ids, table, T, top, E, real, tile_rows, slot_pair, pair_slot, tiles, n_tiles, stream);
}

extern "C" int tm_moe_route(const int* ids, const int* table, int T, int top, int E, int tile_rows, int* slot_pair, int* pair_slot,
                            int* tiles, int* n_tiles, hipStream_t stream) {
    if (!ids || !table || !slot_pair || !pair_slot || !tiles || !n_tiles || T < 0 || top <= 0 || E <= 0 || E > MOE_MAX_EXPERTS ||
        tile_rows <= 0 || (long long)T * top > 0x3fffffffLL)
        return TM_ERR_ARG;
    return launch_moe_route(ids, table, T, top, E, E, tile_rows, slot_pair, pair_slot, tiles, n_tiles, stream);
}

// ------------------------------------------------------------------------------------------------ grouped products

#define MG_TM 32            // rows of a tile (tile_rows of the route)
#define MG_TN 64
#define MG_TK 16

// MODE 1 (gated): C[slot, n] = silu(a . W[e][n]) * (a . W[e][F + n]), a = A[slot_pair[slot] / top]; C of type T.
// MODE 2         : C[slot, n] = relu(a . W[e][n])^2, the same a; C of type T.
// MODE 3 (gated): the clamped gate of tm_moe_clamped, the same a; C of type T.
// MODE 0         : C[slot, n] = A[slot] . W[e][n]; C float32.
template <typename T, int MODE>
__global__ __launch_bounds__(256) void moe_product_kernel(const T* __restrict__ A, int lda, const int* __restrict__ slot_pair, int top,
                                                          const T* __restrict__ W, void* __restrict__ Cv, int ldc,
                                                          const int* __restrict__ tiles, const int* __restrict__ n_tiles, int K,
                                                          int N, const float* __restrict__ pair_weight, float limit, float alpha) {
    constexpr bool GATED = MODE == 1 || MODE == 3, GATHER = MODE != 0;
    if ((int)blockIdx.x >= n_tiles[0]) return;
    __shared__ float As[MG_TM][MG_TK + 1];
    __shared__ float Bs[GATED ? 2 : 1][MG_TK][MG_TN + 1];
    __shared__ int src[MG_TM];
    const int e = tiles[3 * blockIdx.x], slot0 = tiles[3 * blockIdx.x + 1], rows = tiles[3 * blockIdx.x + 2];
    const int n0 = blockIdx.y * MG_TN;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const T* We = W + (size_t)e * (GATED ? 2 : 1) * N * K;
    if (threadIdx.x < MG_TM)
        src[threadIdx.x] = threadIdx.x < rows ? (GATHER ? slot_pair[slot0 + threadIdx.x] / top : slot0 + (int)threadIdx.x) : -1;
    __syncthreads();
    float acc[2][4] = {}, acu[2][4] = {};
    for (int k0 = 0; k0 < K; k0 += MG_TK) {
        for (int i = threadIdx.x; i < MG_TM * MG_TK; i += 256) {
            const int r = i / MG_TK, k = i % MG_TK;
            As[r][k] = (src[r] >= 0 && k0 + k < K) ? Elem<T>::load(A + (size_t)src[r] * lda + k0 + k) : 0.f;
        }
        for (int i = threadIdx.x; i < MG_TK * MG_TN; i += 256) {
            const int n = i / MG_TK, k = i % MG_TK;
            const bool in = n0 + n < N && k0 + k < K;
            Bs[0][k][n] = in ? Elem<T>::load(We + (size_t)(n0 + n) * K + k0 + k) : 0.f;
            if (GATED) Bs[1][k][n] = in ? Elem<T>::load(We + (size_t)(N + n0 + n) * K + k0 + k) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MG_TK; ++k) {
            const float a0 = As[ty * 2][k], a1 = As[ty * 2 + 1][k];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float b = Bs[0][k][tx * 4 + j];
                acc[0][j] += a0 * b;
                acc[1][j] += a1 * b;
                if (GATED) {
                    const float u = Bs[1][k][tx * 4 + j];
                    acu[0][j] += a0 * u;
                    acu[1][j] += a1 * u;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = ty * 2 + i;
        if (r >= rows) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            if (MODE == 3) {
                const float z = pair_weight ? pair_weight[slot_pair[slot0 + r]] : 1.f;
                Elem<T>::store((T*)Cv + (size_t)(slot0 + r) * ldc + n, clamped_glu_f32(z * acc[i][j], z * acu[i][j], alpha, limit));
            } else if (GATED) {
                const float g = acc[i][j], u = acu[i][j];
                Elem<T>::store((T*)Cv + (size_t)(slot0 + r) * ldc + n, g / (1.0f + __expf(-g)) * u);
            } else if (MODE == 2) {
                const float a = fmaxf(acc[i][j], 0.f);
                Elem<T>::store((T*)Cv + (size_t)(slot0 + r) * ldc + n, a * a);
            } else {
                ((float*)Cv)[(size_t)(slot0 + r) * ldc + n] = acc[i][j];
            }
        }
    }
}

extern "C" int tm_moe_gate_up(const void* x, int ldx, const int* slot_pair, int top, const void* W, void* act, const int* tiles,
                              const int* n_tiles, int max_tiles, int K, int F, int dtype, hipStream_t stream) {
    if (!x || !slot_pair || !W || !act || !tiles || !n_tiles || top <= 0 || K <= 0 || F <= 0 || ldx < K || max_tiles < 0) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (max_tiles == 0) return TM_OK;
    dim3 grid(max_tiles, (F + MG_TN - 1) / MG_TN);
    if (grid.y > 65535) return TM_ERR_ARG;
    if (dtype == TM_F32)
        moe_product_kernel<float, 1><<<grid, 256, 0, stream>>>((const float*)x, ldx, slot_pair, top, (const float*)W, act, F, tiles,
                                                                  n_tiles, K, F, nullptr, 0.f, 0.f);
    else
        moe_product_kernel<bf16_t, 1><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldx, slot_pair, top, (const bf16_t*)W, act, F, tiles,
                                                                   n_tiles, K, F, nullptr, 0.f, 0.f);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_moe_up_act(const void* x, int ldx, const int* slot_pair, int top, const void* W, void* act, const int* tiles,
                             const int* n_tiles, int max_tiles, int K, int F, int dtype, hipStream_t stream) {
    if (!x || !slot_pair || !W || !act || !tiles || !n_tiles || top <= 0 || K <= 0 || F <= 0 || ldx < K || max_tiles < 0) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (max_tiles == 0) return TM_OK;
    dim3 grid(max_tiles, (F + MG_TN - 1) / MG_TN);
    if (grid.y > 65535) return TM_ERR_ARG;
    if (dtype == TM_F32)
        moe_product_kernel<float, 2><<<grid, 256, 0, stream>>>((const float*)x, ldx, slot_pair, top, (const float*)W, act, F, tiles,
                                                               n_tiles, K, F, nullptr, 0.f, 0.f);
    else
        moe_product_kernel<bf16_t, 2><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldx, slot_pair, top, (const bf16_t*)W, act, F, tiles,
                                                                n_tiles, K, F, nullptr, 0.f, 0.f);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_moe_clamped(const void* x, int ldx, const int* slot_pair, int top, const float* pair_weight, const void* W, void* act,
                              const int* tiles, const int* n_tiles, int max_tiles, int K, int F, float limit, float alpha, int dtype,
                              hipStream_t stream) {
    if (!x || !slot_pair || !W || !act || !tiles || !n_tiles || top <= 0 || K <= 0 || F <= 0 || ldx < K || max_tiles < 0 || !(limit > 0.f))
        return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (max_tiles == 0) return TM_OK;
    dim3 grid(max_tiles, (F + MG_TN - 1) / MG_TN);
    if (grid.y > 65535) return TM_ERR_ARG;
    if (dtype == TM_F32)
        moe_product_kernel<float, 3><<<grid, 256, 0, stream>>>((const float*)x, ldx, slot_pair, top, (const float*)W, act, F, tiles,
                                                               n_tiles, K, F, pair_weight, limit, alpha);
    else
        moe_product_kernel<bf16_t, 3><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldx, slot_pair, top, (const bf16_t*)W, act, F, tiles,
                                                                n_tiles, K, F, pair_weight, limit, alpha);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

extern "C" int tm_moe_down(const void* act, const void* W, float* part, const int* tiles, const int* n_tiles, int max_tiles, int F,
                           int N, int dtype, hipStream_t stream) {
    if (!act || !W || !part || !tiles || !n_tiles || F <= 0 || N <= 0 || max_tiles < 0) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (max_tiles == 0) return TM_OK;
    dim3 grid(max_tiles, (N + MG_TN - 1) / MG_TN);
    if (grid.y > 65535) return TM_ERR_ARG;
    if (dtype == TM_F32)
        moe_product_kernel<float, 0><<<grid, 256, 0, stream>>>((const float*)act, F, nullptr, 1, (const float*)W, part, N, tiles,
                                                                   n_tiles, F, N, nullptr, 0.f, 0.f);
    else
        moe_product_kernel<bf16_t, 0><<<grid, 256, 0, stream>>>((const bf16_t*)act, F, nullptr, 1, (const bf16_t*)W, part, N, tiles,
                                                                    n_tiles, F, N, nullptr, 0.f, 0.f);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ part, const int* __restrict__ pair_slot,
                                                          T* __restrict__ y, int top, float weight, int N) {
    const int t = blockIdx.x;
    for (int c = threadIdx.x; c < N; c += 256) {
        float s = 0.f;
        for (int k = 0; k < top; ++k) s += weight * part[(size_t)pair_slot[t * top + k] * N + c];
        Elem<T>::store(y + (size_t)t * N + c, s);
    }
}

extern "C" int tm_moe_combine(const float* part, const int* pair_slot, void* y, int T, int top, float weight, int N, int dtype,
                              hipStream_t stream) {
    if (!part || !pair_slot || !y || T < 0 || top <= 0 || N <= 0) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (T == 0) return TM_OK;
    if (dtype == TM_F32)
        moe_combine_kernel<float><<<T, 256, 0, stream>>>(part, pair_slot, (float*)y, top, weight, N);
    else
        moe_combine_kernel<bf16_t><<<T, 256, 0, stream>>>(part, pair_slot, (bf16_t*)y, top, weight, N);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// ------------------------------------------------------------------------------------------------ a router

// A wavefront a token; lane l holds experts l, l + 64, ... (RT_MAX_PER_LANE of them: 1, 4 or 16 by the number of experts).
// Everything is 32-bit.
template <int RT_MAX_PER_LANE>
__global__ __launch_bounds__(TM_WAVE) void moe_router_kernel(const float* __restrict__ z, int ldz, const float* __restrict__ correction,
                                                             int E, int top, int* __restrict__ chosen, float* __restrict__ weight,
                                                             int over_chosen, int sigmoid) {
    const int t = blockIdx.x, lane = threadIdx.x;
    const float* zr = z + (size_t)t * ldz;
    float s[RT_MAX_PER_LANE], c[RT_MAX_PER_LANE];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < RT_MAX_PER_LANE; ++i) {
        const int e = lane + i * TM_WAVE;
        s[i] = e < E ? zr[e] : -INFINITY;
        m = fmaxf(m, s[i]);
    }
    m = sigmoid ? 0.f : wave_max(m);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < RT_MAX_PER_LANE; ++i) {
        const int e = lane + i * TM_WAVE;
        c[i] = s[i];                             // the output itself: what `over_chosen` ranks
        s[i] = e >= E ? 0.f : sigmoid ? 1.f / (1.f + expf(-s[i])) : expf(s[i] - m);     // m is the largest output, which is chosen first: these are the chosen ones' terms too
        sum += s[i];
    }
    sum = wave_sum(sum);
    if (!over_chosen) {
#pragma unroll
        for (int i = 0; i < RT_MAX_PER_LANE; ++i) {
            const int e = lane + i * TM_WAVE;
            if (!sigmoid) s[i] = s[i] / sum;
            c[i] = e < E ? s[i] + (correction ? correction[e] : 0.f) : -INFINITY;
        }
    }
    float total = 0.f;
    for (int k = 0; k < top; ++k) {
        float best = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < RT_MAX_PER_LANE; ++i)
            if (c[i] > best) best = c[i], at = lane + i * TM_WAVE;      // within a lane e ascends: the first of equals stays
        const float top_v = wave_max(best);
        int cand = (best == top_v) ? at : 0x7fffffff;
#pragma unroll
        for (int o = TM_WAVE / 2; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, TM_WAVE));
        float sc = 0.f;
#pragma unroll
        for (int i = 0; i < RT_MAX_PER_LANE; ++i)
            if (lane + i * TM_WAVE == cand) sc = s[i], c[i] = -INFINITY;
        sc = wave_sum(sc);                   // one lane holds it, the others 0
        total += sc;
        if (lane == 0) {
            chosen[(size_t)t * top + k] = cand;
            weight[(size_t)t * top + k] = sc;
        }
    }
    if (sigmoid) return;
    __syncthreads();                         // lane 0's scores, seen by the lanes that scale them
    const float inv = over_chosen ? 1.f / total : 1.f / (total + 1e-20f);
    for (int k = lane; k < top; k += TM_WAVE) weight[(size_t)t * top + k] *= inv;
}

extern "C" int tm_moe_router(const float* z, int ldz, const float* correction, int T, int E, int top, int* chosen, float* weight,
                             int over_chosen, int sigmoid, hipStream_t stream) {
    if (!z || !chosen || !weight || T < 0 || E <= 0 || E > MOE_MAX_EXPERTS || top <= 0 || top > E || ldz < E) return TM_ERR_ARG;
    if (T == 0) return TM_OK;
    if (over_chosen && (correction || sigmoid)) return TM_ERR_ARG;
    if (E <= TM_WAVE) moe_router_kernel<1><<<T, TM_WAVE, 0, stream>>>(z, ldz, correction, E, top, chosen, weight, over_chosen, sigmoid);
    else if (E <= 4 * TM_WAVE) moe_router_kernel<4><<<T, TM_WAVE, 0, stream>>>(z, ldz, correction, E, top, chosen, weight, over_chosen, sigmoid);
    else moe_router_kernel<MOE_MAX_EXPERTS / TM_WAVE><<<T, TM_WAVE, 0, stream>>>(z, ldz, correction, E, top, chosen, weight, over_chosen, sigmoid);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// A block is a token and 256 columns: few tokens still make many blocks, and a thread's loads (the pair's slot, then its row)
// wait once, not once a column.
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_weighted_kernel(const float* __restrict__ part, const int* __restrict__ pair_slot,
                                                                   const float* __restrict__ weight, const T* __restrict__ x, int ldx,
                                                                   const float* __restrict__ shared, const float* __restrict__ shared_gate,
                                                                   int ldg, T* __restrict__ y, int top, int N) {
    const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= N) return;
    const float sg = (shared && shared_gate) ? 1.f / (1.f + expf(-shared_gate[(size_t)t * ldg])) : 1.f;
    float s = 0.f;
    for (int k = 0; k < top; ++k) {
        const int slot = pair_slot[t * top + k];
        const float v = slot >= 0 ? part[(size_t)slot * N + c] : Elem<T>::load(x + (size_t)t * ldx + c);
        s += weight ? weight[(size_t)t * top + k] * v : v;
    }
    if (shared) s += sg * shared[(size_t)t * N + c];
    Elem<T>::store(y + (size_t)t * N + c, s);
}

// shared (float32 [T, N]) and shared_gate (float32, one number a token, rows ldg apart) may be null.
extern "C" int tm_moe_combine_weighted(const float* part, const int* pair_slot, const float* weight, const void* x, int ldx,
                                       const float* shared, const float* shared_gate, int ldg, void* y, int T, int top, int N, int dtype,
                                       hipStream_t stream) {
    if (!part || !pair_slot || !x || !y || T < 0 || top <= 0 || N <= 0 || ldx < N || (shared_gate && ldg < 1)) return TM_ERR_ARG;
    if (dtype != TM_F32 && dtype != TM_BF16) return TM_ERR_ARG;
    if (T == 0) return TM_OK;
    const dim3 grid(T, (N + 255) / 256);
    if (grid.y > 65535) return TM_ERR_ARG;
    if (dtype == TM_F32)
        moe_combine_weighted_kernel<float><<<grid, 256, 0, stream>>>(part, pair_slot, weight, (const float*)x, ldx, shared, shared_gate, ldg,
                                                                  (float*)y, top, N);
    else
        moe_combine_weighted_kernel<bf16_t><<<grid, 256, 0, stream>>>(part, pair_slot, weight, (const bf16_t*)x, ldx, shared, shared_gate, ldg,
                                                                   (bf16_t*)y, top, N);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
