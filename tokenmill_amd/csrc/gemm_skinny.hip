// C[M, N] = A[M, K] * W[N, K]^T (+ bias) for few rows (M <= 64) on MFMA, bfloat16 in, 32-bit sums.
//
// With so few rows the product is bound by reading W once. Each wavefront streams a strip of 16
// rows of W (16-byte loads straight into the MFMA A operand: 16 rows x 32 k per instruction) and
// multiplies it with all M activations rows (B operand, 16 tokens per tile). The result tile holds,
// per lane, four consecutive output features of one token.
//
//   split mode : the WAVES wavefronts of a block share one strip and split K between them; their
//                partial sums are added through LDS in wavefront order (for matrices with few rows,
//                so that enough wavefronts are in flight).
//   row mode   : each of the 4 wavefronts of a block has a strip of its own (matrices with many
//                rows, such as the output head).
//
// The K range of each wavefront and the order of all additions depend only on K and the mode,
// never on M: a token's result does not depend on how many other tokens the call holds.
// Fused epilogues: bias; silu(gate) * up for a stacked [gate; up] matrix (reference
// src/infer/model/layers.py:163-164), with gate and up rounded to bfloat16 first as if stored.
//
// The matrix is read row-major [N, K], or (decode steps, at most 16 tokens) in strip order: the
// 16-byte piece of lane (r, g) for k-step ks of strip s lies at ((s * ksteps + ks) * 4 + g) * ROWS + r
// pieces, so that a wavefront's load is one run of ROWS * 64 bytes instead of ROWS pieces a row
// apart (measured on an MI355X: 15% more bytes a second from HBM). Both give the same bits.
#include "common.h"
#include "api.h"
#include "fused_common.h"

typedef FFrag Frag;

__device__ __forceinline__ Frag load_frag(const bf16_t* row, int k, int K, bool row_ok) {
    Frag f;
    if (row_ok && k < K)
        f.u = *(const u32x4_t*)(row + k);
    else
        f.u = u32x4_t{0, 0, 0, 0};
    return f;
}

template <typename TC>
__device__ __forceinline__ void store4(TC* dst, const float v[4], int n_left);

template <>
__device__ __forceinline__ void store4<float>(float* dst, const float v[4], int n_left) {
    if (n_left >= 4 && ((uintptr_t)dst % 16) == 0) {
        *(f32x4_t*)dst = f32x4_t{v[0], v[1], v[2], v[3]};
    } else {
        for (int i = 0; i < 4 && i < n_left; ++i) dst[i] = v[i];
    }
}

template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* dst, const float v[4], int n_left) {
    if (n_left >= 4 && ((uintptr_t)dst % 8) == 0) {
        uint2 pk;
        pk.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
        pk.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
        *(uint2*)dst = pk;
    } else {
        for (int i = 0; i < 4 && i < n_left; ++i) dst[i] = f32_to_bf16(v[i]);
    }
}

// flags of a launch: the bias is 32-bit; the result is relu(.)^2 (after the bias, before the one rounding)
enum { SK_BIAS_F32 = 1, SK_RELU2 = 2 };

__device__ __forceinline__ float bias_at(const void* bias, int flags, int n) {
    return (flags & SK_BIAS_F32) ? ((const float*)bias)[n] : bf16_to_f32(((const bf16_t*)bias)[n]);
}

// --- at most 16 tokens, a strip's K split over wavefronts -------------------------------------------------------------------
// The output and down projections of decode steps. Such a launch waits for memory once and then for the loads of a CU to pass its
// address unit, 16 cycles an instruction whatever its lanes bring: with a strip of four rows a lane in four brought a part of
// the matrix and with one token a lane in sixteen a part of the activations, and every load stood under a test of its own (a down
// projection of 4,864 -> 896: 16 wavefronts of ten and ten loads, 2.1 us of the address unit for 39 KB a block).
//
// So an MFMA tile holds several ranges of K at once. The 16 rows of the A operand are the ROWS rows of the strip for each of
// SA = 16 / ROWS ranges, the 16 columns of the B operand are TOKS tokens for each of SB = 16 / TOKS ranges; what is computed where a
// range meets itself counts, the rest is dropped. VW is the number of ranges, a wavefront has SA of them and multiplies one
// load of the matrix by NB = SA / SB loads of activations, each into accumulators of its own. Which k a range has (as many k-steps as
// every other, in order) and the order in which the VW sums are added are those of gemm_skinny_kernel with VW wavefronts, so the
// bits are the same for any number of tokens. Loads are unconditional: what lies beyond the strip, a token or a range
// reads as zero by the bounds of its buffer descriptor.
//
// TURN: neighbouring lanes of the B operand are different tokens, one address a clock for the CU, and the loads of activations were most of a launch
// whose matrix lies in the caches. Four lanes beside each other load 64 bytes of a token (lane (4 q + p, g) column 4 q + g, piece p) and the
// pieces change lanes by ds_bpermute. us without / with, matrices in the caches (brought ahead, as in a step) and cold: 4,864 -> 896 4 tokens 3.87 / 3.41
// and 4.75 / 4.63, 8 5.05 / 4.44 and 6.15 / 5.88, 16 7.18 / 6.25 and 8.75 / 8.32; 8,960 -> 1,536 8 7.63 / 5.74 and 10.4 / 9.9; 18,944 -> 3,584 8 21.4 / 21.1
// and 28.2 / 27.4; 896 -> 9,728 16 5.25 / 3.88 and 7.1 / 6.9. The rule is few_turns below. The same bits.
template <int ROWS, int TOKS, int VW, int CH, typename TC, bool PACKED, bool TURN>
__global__ __launch_bounds__(64 * VW * ROWS / 16) void gemm_few_kernel(const bf16_t* __restrict__ A, int lda,
                                                                       const bf16_t* __restrict__ W,
                                                                       const void* __restrict__ bias, int flags,
                                                                       TC* __restrict__ C, int ldc, int M, int N, int K,
                                                                       float* __restrict__ accum, int ldacc) {
    constexpr int SA = 16 / ROWS, SB = 16 / TOKS, NB = SA / SB;
    static_assert(SA >= SB && VW % SA == 0, "whole wavefronts, and no range of the activations without one of the matrix");
    constexpr int BEYOND = 0x7ffffff0;
    __shared__ f32x4_t red[VW][ROWS / 4][16];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * ROWS;
    const int ksteps = (K + 31) / 32, per = (ksteps + VW - 1) / VW;
    const int range0 = wave * SA;                       // this wavefront's first range

    // what the epilogue (wavefront 0: lane = token lane % 16, rows n0 + 4 (lane / 16) + i) reads from memory is asked for first
    const int tok = r, nf = n0 + 4 * g;
    const bool epi = wave == 0 && 4 * g < ROWS && tok < M && nf < N;
    const bool fast = accum && N % 4 == 0 && ldacc % 4 == 0 && ((uintptr_t)accum % 16) == 0;      // the same in every lane
    f32x4_t current = {0.f, 0.f, 0.f, 0.f}, offset = {0.f, 0.f, 0.f, 0.f};
    if (wave == 0) {
        if (fast) current = *(const f32x4_t*)(accum + (epi ? (size_t)tok * ldacc + nf : 0));
        if (bias) {
#pragma unroll
            for (int i = 0; i < 4; ++i) offset[i] = bias_at(bias, flags, nf + i < N ? nf + i : 0);
        }
    }

    // the matrix: lane (r, g) has row r % ROWS, eight k at 8 g of a k-step of range r / ROWS
    constexpr int FRAG = 32 * ROWS;                     // packed: bfloat16 values of a (strip, k-step)
    const __amdgpu_buffer_rsrc_t wbuf = PACKED ? fd_buffer(W + (size_t)blockIdx.x * ksteps * FRAG, ksteps * FRAG * 2)
                                               : fd_buffer(W + (size_t)n0 * K, (N - n0 < ROWS ? N - n0 : ROWS) * K * 2);
    const int w_ks = (range0 + r / ROWS) * per;         // its first k-step ...
    const int w_end = w_ks + per < ksteps ? w_ks + per : ksteps;
    const int w_k = PACKED ? w_end : (w_end * 32 < K ? w_end * 32 : K) - 8 * g;     // ... and the first that is not its own (in k-steps or k)
    auto w_at = [&](int j) {
        const int ks = w_ks + j;
        if (PACKED) return ks < w_k ? ((ks * 4 + g) * ROWS + r % ROWS) * 16 : BEYOND;
        return ks * 32 < w_k ? ((r % ROWS) * K + ks * 32 + 8 * g) * 2 : BEYOND;
    };
    // the activations: lane (r, g) has token r % TOKS, eight k at 8 g of a k-step of range b SB + r / TOKS
    const __amdgpu_buffer_rsrc_t abuf = fd_buffer(A, ((M - 1) * lda + K) * 2);
    const int column = TURN ? 4 * (r / 4) + g : r, piece = TURN ? r % 4 : g;      // what it loads
    const int from = 4 * (16 * (r % 4) + 4 * (r / 4) + g);                        // the lane, in bytes, that has column r's piece g
    int a_k[NB], a_end[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int ks = (range0 + b * SB + column / TOKS) * per, end = ks + per < ksteps ? ks + per : ksteps;
        a_k[b] = ks * 32 + 8 * piece;
        a_end[b] = column % TOKS < M ? (end * 32 < K ? end * 32 : K) : 0;
    }
    const int a_row = (column % TOKS) * lda;

    f32x4_t acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // CH k-steps of every range at a time, every load issued before the first product
    for (int base = 0; base < per; base += CH) {
        Frag wf[CH], af[NB][CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int k = a_k[b] + (base + j) * 32;
                af[b][j].u = __builtin_amdgcn_raw_buffer_load_b128(abuf, base + j < per && k < a_end[b] ? (a_row + k) * 2 : BEYOND, 0, 0);
            }
            if constexpr (PACKED) wf[j].u = __builtin_amdgcn_raw_buffer_load_b128(wbuf, base + j < per ? w_at(base + j) : BEYOND, 0, 0);
        }
        if constexpr (!PACKED) {                                     // (both halves of a line of the matrix one after the other)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < CH; ++j) wf[j].u = __builtin_amdgcn_raw_buffer_load_b128(wbuf, base + j < per ? w_at(base + j) : BEYOND, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (TURN) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) af[b][j].u[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)af[b][j].u[e]);
                }
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].b, af[b][j].b, acc[b], 0, 0, 0);
            }
    }
    // lane: rows 4 g + i of the tile, so range 4 g / ROWS of the matrix; columns of range r / TOKS in each of the NB groups
    const int range = 4 * g / ROWS;
    f32x4_t own = acc[0];
#pragma unroll
    for (int b = 1; b < NB; ++b)
        if (range / SB == b) own = acc[b];
    if (range % SB == r / TOKS) red[range0 + range][g % (ROWS / 4)][r % TOKS] = own;
    __syncthreads();
    if (!epi) return;
    f32x4_t v = red[0][g][tok];
#pragma unroll
    for (int w = 1; w < VW; ++w) v += red[w][g][tok];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (bias) v[i] += offset[i];
        if (flags & SK_RELU2) {
            v[i] = fmaxf(v[i], 0.f);
            v[i] *= v[i];
        }
    }
    if (accum) {                // the rounded result goes into the 32-bit residual stream (each element has one owner)
        float* dst = accum + (size_t)tok * ldacc + nf;
        if (fast) {
#pragma unroll
            for (int i = 0; i < 4; ++i) current[i] += bf16_to_f32(f32_to_bf16(v[i]));
            *(f32x4_t*)dst = current;
        } else {
            for (int i = 0; i < 4 && nf + i < N; ++i) dst[i] += bf16_to_f32(f32_to_bf16(v[i]));
        }
    } else {
        const float out[4] = {v[0], v[1], v[2], v[3]};
        store4<TC>(C + (size_t)tok * ldc + nf, out, N - nf);
    }
}

// K-steps a round, for ranges of `per` of them: of the four depths a shape has kernels for, ascending, the last sets the rounds and the first
// that does with as many is taken. What a round asks for beyond a range reads as zero, but passes the address unit all the same: with
// one depth a shape (7, 8, 10 or 16) 896 -> 9,728 took 6.7 / 7.0 / 7.8 us at 1 / 8 / 16 tokens where it takes 5.1 / 5.5 / 6.7, 1,024 -> 1,024 and
// 2,048 -> 2,048 at 16 tokens 4.4 and 5.8 where they take 3.7 and 4.9.
static int few_depth(int per, int a, int b, int c, int d) {
    const int rounds = (per + d - 1) / d;
    return a * rounds >= per ? a : b * rounds >= per ? b : c * rounds >= per ? c : d;
}

// Do the activations' pieces change lanes behind their loads? Where the loads are many (a long K; else strips of 16 rows and K of 512 and more) and the
// tokens fill their places: with 9 of 16 and 5 of 8 tokens 4,864 -> 896 takes 6.0 for 5.7 and 4.4 for 4.3 us, with 4 of 16 4,096 -> 4,096 6.0 for 5.7
// (18,944 -> 3,584 level up to 5); over a short K and strips of 4 or 8 rows the exchange is longer than the wait (896 -> 896 8 tokens 3.0 / 3.4,
// 1,536 -> 1,536 3.2 / 3.3), and over 256 -> 4,096 too (2.55 / 2.67 at 10 tokens). And where rows lie in whole pieces of 64 bytes: four lanes' loads that straddle two
// lines are no fewer than before, and 2,056 -> 896 takes 3.9 for 4.4 us at 12 tokens, 1,032 -> 3,584 2.7 for 2.9. Where they do, over 70 matrices, the launch takes
// 0.68 to 1.04 of the time of the other order, the matrix in the caches, and 0.86 to 1.07 cold (above 1.04 at 12 to 14 tokens of strips of 4 rows).
static bool few_turns(int rows, int M, int K, bool long_k, const void* A, int lda) {
    if (lda % 32 || (uintptr_t)A % 64) return false;
    if (!long_k) return rows == 16 && M >= 10 && K >= 512;
    return rows == 4 ? 4 * M >= 3 * (M <= 4 ? 4 : M <= 8 ? 8 : 16) : M >= (rows == 8 ? 4 : 6);
}
static bool few_long_k(int rows, int N, int K) { return K >= 2048 && !(rows == 16 && (N + 15) / 16 >= 256); }

// ... of a packed matrix and activations at a whole line (for tests)
extern "C" int tm_skinny_turns(int M, int N, int K, int lda) {
    const int rows = tm_skinny_strip_rows(N, K);
    return few_turns(rows, M, K, few_long_k(rows, N, K), nullptr, lda);
}

// Ranges of K: 4, or 16 for a long K over few strips. `rows`: of a strip (16, 8 or 4).
template <typename TC, bool PACKED>
static int launch_few(const void* A, int lda, const void* W, int rows, const void* bias, int flags, void* C, int ldc, int M, int N,
                      int K, float* accum, int ldacc, hipStream_t stream) {
    if ((size_t)M * lda * 2 >= 0x7ffffff0u && M > 1) {          // rows so far apart that an offset does not hold it: one by one (the same bits)
        for (int m = 0; m < M; ++m) {
            const int rc = launch_few<TC, PACKED>((const bf16_t*)A + (size_t)m * lda, lda, W, rows, bias, flags, C ? (TC*)C + (size_t)m * ldc : nullptr,
                                                  ldc, 1, N, K, accum ? accum + (size_t)m * ldacc : nullptr, ldacc, stream);
            if (rc) return rc;
        }
        return TM_OK;
    }
    const int strips = (N + rows - 1) / rows;
    const bool long_k = few_long_k(rows, N, K);
    const int ksteps = (K + 31) / 32, per = long_k ? (ksteps + 15) / 16 : (ksteps + 3) / 4;
    const bool turn = PACKED && few_turns(rows, M, K, long_k, A, lda);
#define TM_FEW(ROWS_, TOKS_, VW_, CH_, TURN_)                                                                         \
    gemm_few_kernel<ROWS_, TOKS_, VW_, CH_, TC, PACKED, TURN_><<<strips, 4 * VW_ * ROWS_, 0, stream>>>(               \
        (const bf16_t*)A, lda, (const bf16_t*)W, bias, flags, (TC*)C, ldc, M, N, K, accum, ldacc)
#define TM_FEW_DEPTHS(ROWS_, TOKS_, VW_, A_, B_, C_, D_, TURN_)                                                       \
    switch (few_depth(per, A_, B_, C_, D_)) {                                                                         \
        case A_: TM_FEW(ROWS_, TOKS_, VW_, A_, TURN_); break;                                                         \
        case B_: TM_FEW(ROWS_, TOKS_, VW_, B_, TURN_); break;                                                         \
        case C_: TM_FEW(ROWS_, TOKS_, VW_, C_, TURN_); break;                                                         \
        default: TM_FEW(ROWS_, TOKS_, VW_, D_, TURN_);                                                                \
    }
#define TM_FEW_DEEP(ROWS_, TOKS_, VW_, A_, B_, C_, D_)                                                                \
    if (turn) { TM_FEW_DEPTHS(ROWS_, TOKS_, VW_, A_, B_, C_, D_, (PACKED && (VW_ == 16 || ROWS_ == 16))) }            \
    else { TM_FEW_DEPTHS(ROWS_, TOKS_, VW_, A_, B_, C_, D_, false) }
    if (rows == 4 && long_k) {
        if (M <= 4) { TM_FEW_DEEP(4, 4, 16, 4, 6, 8, 10) }
        else if (M <= 8) { TM_FEW_DEEP(4, 8, 16, 4, 6, 8, 10) }
        else { TM_FEW_DEEP(4, 16, 16, 4, 5, 6, 8) }
    } else if (rows == 4) {
        if (M <= 4) { TM_FEW_DEEP(4, 4, 4, 4, 6, 7, 8) }
        else if (M <= 8) { TM_FEW_DEEP(4, 8, 4, 4, 6, 7, 8) }
        else { TM_FEW_DEEP(4, 16, 4, 4, 6, 7, 8) }
    } else if (rows == 8 && long_k) {
        if (M <= 8) { TM_FEW_DEEP(8, 8, 16, 4, 6, 9, 11) }
        else { TM_FEW_DEEP(8, 16, 16, 4, 6, 9, 11) }
    } else if (rows == 8) {
        if (M <= 8) { TM_FEW_DEEP(8, 8, 4, 4, 6, 7, 8) }
        else { TM_FEW_DEEP(8, 16, 4, 4, 6, 7, 8) }
    } else if (long_k) {
        TM_FEW_DEEP(16, 16, 16, 5, 6, 8, 10)
    } else {
        TM_FEW_DEEP(16, 16, 4, 7, 8, 10, 14)
    }
#undef TM_FEW_DEPTHS
#undef TM_FEW_DEEP
#undef TM_FEW
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// NT: tiles of 16 tokens. WAVES: wavefronts per block. SPLIT: they share a strip and split K.
// SILU: W is [2 * N, K] = [gate; up] and the output is silu(gate) * up, N wide.
// PACKED: W is in strip order, strips of 16 rows, rows and k beyond the matrix zero-filled; with SILU
// the up rows' strips start at strip `up_strip0` (each half packed by itself).
template <int NT, int WAVES, bool SPLIT, bool SILU, typename TC, bool PACKED = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(const bf16_t* __restrict__ A, int lda,
                                                                 const bf16_t* __restrict__ W,
                                                                 const void* __restrict__ bias, int flags,
                                                                 TC* __restrict__ C, int ldc, int M, int N, int K,
                                                                 float* __restrict__ accum, int ldacc,
                                                                 int up_strip0 = 0) {
    constexpr int NACC = SILU ? 2 : 1, ROWS = 16;
    // k-steps in flight per wavefront (fewer where 16 wavefronts share the register file)
    constexpr int KCH = (WAVES > 4 && SILU && NT > 2) ? 4 : ((WAVES > 4 || NT > 2 || SILU) ? 8 : 16);
    __shared__ float red[SPLIT ? WAVES : 1][64][4 + 1];        // one accumulator tile at a time
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int strip = SPLIT ? blockIdx.x : blockIdx.x * WAVES + wave;
    const int n0 = strip * ROWS;
    // K range of this wavefront, in steps of 32
    const int ksteps = (K + 31) / 32;
    int ks0 = 0, ks1 = ksteps;
    if (SPLIT) {
        const int per = (ksteps + WAVES - 1) / WAVES;
        ks0 = wave * per;
        ks1 = ks0 + per < ksteps ? ks0 + per : ksteps;
    }
    constexpr int FRAG = 32 * ROWS;             // packed: bfloat16 values of a (strip, k-step)
    const bool w_ok = PACKED || n0 + r < N;
    const bf16_t* wrow;
    const bf16_t* urow = nullptr;
    if constexpr (PACKED) {
        const int lane_off = (g * ROWS + r) * 8;
        wrow = W + (size_t)strip * ksteps * FRAG + lane_off;
        if (SILU) urow = W + (size_t)(up_strip0 + strip) * ksteps * FRAG + lane_off;
    } else {
        wrow = W + (size_t)(n0 + r) * K + 8 * g;
        if (SILU) urow = W + (size_t)(N + n0 + r) * K + 8 * g;
    }
    // offset of k-step ks from wrow / urow, and how far a lane's eight values may reach
    auto w_at = [&](int ks) { return PACKED ? ks * FRAG : ks * 32; };
    const int w_end = PACKED ? ksteps * FRAG : K - 8 * g;
    const bf16_t* arow[NT];
    bool a_ok[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        a_ok[t] = 16 * t + r < M;
        arow[t] = A + (size_t)(16 * t + r) * lda + 8 * g;
    }
    f32x4_t acc[NACC][NT];
#pragma unroll
    for (int a = 0; a < NACC; ++a)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[a][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // What the accumulate epilogue will read is asked for now: it arrives while the matrix streams.
    const int nf = n0 + 4 * g;                  // this lane's output features nf + i (i = 0..3) of token 16t + r
    const bool acc_fast = accum && nf + 4 <= N && (ldacc % 4) == 0 && ((uintptr_t)accum % 16) == 0;
    f32x4_t resid_cur[NT];
    if (acc_fast && (!SPLIT || wave == 0)) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
            resid_cur[t] = 16 * t + r < M ? *(const f32x4_t*)(accum + (size_t)(16 * t + r) * ldacc + nf) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    if (n0 < N) {
        // KCH k-steps at a time with every load issued before the first product: a wavefront's whole
        // K range is at most one or two such groups, so it waits for memory once or twice, not per step.
        for (int base = ks0; base < ks1; base += KCH) {
            // With one tile of tokens (decode steps) the activations are asked for first: loads come back
            // in the order they were issued, and these few rows come from the cache long before the
            // matrix arrives from HBM. With more tiles there are no registers for that.
            Frag af[NT == 1 ? KCH : 1], wf[KCH], uf[SILU ? KCH : 1];
            if constexpr (NT == 1) {
#pragma unroll
                for (int j = 0; j < KCH; ++j)
                    af[j] = load_frag(arow[0], (base + j) * 32, K - 8 * g, a_ok[0] && base + j < ks1);
            }
#pragma unroll
            for (int j = 0; j < KCH; ++j) {
                const bool in = base + j < ks1;
                wf[j] = load_frag(wrow, w_at(base + j), w_end, w_ok && in);
                if (SILU) uf[j] = load_frag(urow, w_at(base + j), w_end, w_ok && in);
            }
#pragma unroll
            for (int j = 0; j < KCH; ++j) {
                const bool in = base + j < ks1;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    Frag a1;
                    if constexpr (NT == 1) a1 = af[j];
                    else a1 = load_frag(arow[t], (base + j) * 32, K - 8 * g, a_ok[t] && in);
                    acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].b, a1.b, acc[0][t], 0, 0, 0);
                    if (SILU) acc[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uf[j].b, a1.b, acc[1][t], 0, 0, 0);
                }
            }
        }
    }
    if (SPLIT) {
#pragma unroll
        for (int a = 0; a < NACC; ++a)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) red[wave][lane][i] = acc[a][t][i];
                __syncthreads();
                if (wave == 0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float v = red[0][lane][i];
                        for (int w = 1; w < WAVES; ++w) v += red[w][lane][i];
                        acc[a][t][i] = v;
                    }
                }
                __syncthreads();
            }
        if (wave != 0) return;
    }
    if (n0 >= N) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int tok = 16 * t + r;
        if (tok >= M || nf >= N) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x = acc[0][t][i];
            if (bias && nf + i < N) x += bias_at(bias, flags, nf + i);
            if (!SILU && (flags & SK_RELU2)) {
                x = fmaxf(x, 0.f);
                x *= x;
            }
            if (SILU) {
                const float gt = bf16_to_f32(f32_to_bf16(x));
                const float up = bf16_to_f32(f32_to_bf16(acc[1][t][i]));
                x = gt / (1.f + expf(-gt)) * up;
            }
            v[i] = x;
        }
        if (accum) {            // the rounded result goes into the 32-bit residual stream (each element has one owner)
            float* dst = accum + (size_t)tok * ldacc + nf;
            if (acc_fast) {
                f32x4_t cur = resid_cur[t];
#pragma unroll
                for (int i = 0; i < 4; ++i) cur[i] += bf16_to_f32(f32_to_bf16(v[i]));
                *(f32x4_t*)dst = cur;
            } else {
                for (int i = 0; i < 4 && nf + i < N; ++i) dst[i] += bf16_to_f32(f32_to_bf16(v[i]));
            }
        } else {
            store4<TC>(C + (size_t)tok * ldc + nf, v, N - nf);
        }
    }
}

template <int NT, bool SILU, typename TC>
static int launch_skinny(const void* A, int lda, const void* W, const void* bias, int flags, void* C, int ldc,
                         int M, int N, int K, float* accum, int ldacc, hipStream_t stream) {
    const int strips = (N + 15) / 16;
    if constexpr (NT == 1 && !SILU) {
        if (strips < 2048) return launch_few<TC, false>(A, lda, W, tm_skinny_strip_rows(N, K), bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    }
    if (strips >= 2048) {                      // many rows: a strip per wavefront
        gemm_skinny_kernel<NT, 4, false, SILU, TC><<<(strips + 3) / 4, 256, 0, stream>>>(
            (const bf16_t*)A, lda, (const bf16_t*)W, bias, flags, (TC*)C, ldc, M, N, K, accum, ldacc);
    } else if constexpr (NT > 1 || SILU) {
        if (strips >= 256 || K < 2048)         // a block of 4 wavefronts per strip
            gemm_skinny_kernel<NT, 4, true, SILU, TC><<<strips, 256, 0, stream>>>(
                (const bf16_t*)A, lda, (const bf16_t*)W, bias, flags, (TC*)C, ldc, M, N, K, accum, ldacc);
        else                                   // few rows, long K: 16 wavefronts per strip
            gemm_skinny_kernel<NT, 16, true, SILU, TC><<<strips, 1024, 0, stream>>>(
                (const bf16_t*)A, lda, (const bf16_t*)W, bias, flags, (TC*)C, ldc, M, N, K, accum, ldacc);
    }
    TM_CHECK_LAUNCH();
    return TM_OK;
}

template <bool SILU, typename TC>
static int launch_skinny_nt(const void* A, int lda, const void* W, const void* bias, int flags, void* C, int ldc,
                            int M, int N, int K, float* accum, int ldacc, hipStream_t stream) {
    switch ((M + 15) / 16) {
        case 1: return launch_skinny<1, SILU, TC>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
        case 2: return launch_skinny<2, SILU, TC>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
        case 3: return launch_skinny<3, SILU, TC>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
        case 4: return launch_skinny<4, SILU, TC>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
        default: return TM_ERR_ARG;
    }
}

// silu == 0: C[M, N] = A W^T + bias, W [N, K].   silu == 1: C[M, N] = silu(A Wg^T) * (A Wu^T), W = [Wg; Wu] [2N, K].
// silu == 2: C[M, N] = relu(A W^T + bias)^2.
// A, W bfloat16; C bfloat16 (out_dtype 1) or float32 (0); bias bfloat16 or float32 or null.
// accum != null: nothing is stored to C; the bfloat16-rounded result is added to accum[M, N] (float32, row
// stride ldacc) instead: the residual add of the layer, done by the product that feeds it.
// Needs M <= 64, K % 8 == 0, lda % 8 == 0 and 16-byte aligned A and W.
extern "C" int tm_gemm_skinny(const void* A, int lda, const void* W, const void* bias, int bias_dtype, void* C,
                              int ldc, int M, int N, int K, int out_dtype, int silu, float* accum, int ldacc,
                              hipStream_t stream) {
    if (M <= 0 || N <= 0) return TM_OK;
    const int relu2 = silu == 2;            // silu == 2: no second matrix, the result is relu(A W^T + bias)^2
    if (relu2) silu = 0;
    if (accum && (silu || ldacc < N)) return TM_ERR_ARG;
    if (!accum && !C) return TM_ERR_ARG;
    if (M > 64 || K <= 0 || (K % 8) || (lda % 8) || lda < K || ldc < N || ((uintptr_t)A % 16) || ((uintptr_t)W % 16))
        return TM_ERR_ARG;
    if (silu && bias) return TM_ERR_ARG;
    const int flags = (bias_dtype == TM_F32 ? SK_BIAS_F32 : 0) | (relu2 ? SK_RELU2 : 0);    // the kernel's flags
    if (out_dtype == TM_BF16)
        return silu ? launch_skinny_nt<true, bf16_t>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream)
                    : launch_skinny_nt<false, bf16_t>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    if (out_dtype == TM_F32 && !silu)
        return launch_skinny_nt<false, float>(A, lda, W, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    return TM_ERR_ARG;
}

// Rows of a strip that tm_gemm_skinny_packed wants a plain [N, K] matrix (no SiLU) packed in: 16, or
// 8 or 4 for a matrix with so few rows that 16-row strips would leave CUs without a block.
extern "C" int tm_skinny_strip_rows(int N, int K) {
    (void)K;
    if ((N + 15) / 16 >= 192) return 16;
    return (N + 7) / 8 >= 192 ? 8 : 4;
}

template <bool SILU, typename TC>
static int launch_skinny_packed(const void* A, int lda, const void* W, int rows, const void* bias, int flags, void* C, int ldc,
                                int M, int N, int K, float* accum, int ldacc, hipStream_t stream) {
    const int strips = (N + 15) / 16;
#define TM_PACKED(WV, SPL, BLOCKS)                                                                               \
    gemm_skinny_kernel<1, WV, SPL, SILU, TC, true><<<BLOCKS, 64 * WV, 0, stream>>>(                              \
        (const bf16_t*)A, lda, (const bf16_t*)W, bias, flags, (TC*)C, ldc, M, N, K, accum, ldacc, strips)
    if (rows == 16 && strips >= 2048) TM_PACKED(4, false, (strips + 3) / 4);      // many rows: a strip per wavefront
    else if constexpr (!SILU) return launch_few<TC, true>(A, lda, W, rows, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    else if (K < 2048 || strips >= 256) TM_PACKED(4, true, strips);
    else TM_PACKED(16, true, strips);
#undef TM_PACKED
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// tm_gemm_skinny for at most 16 rows with the matrix in strip order (tm_pack_layout in api.h): strips of
// `rows` rows (16, 8 or 4; 16 with silu, where Wg and Wu are each packed by themselves, Wu behind Wg).
extern "C" int tm_gemm_skinny_packed(const void* A, int lda, const void* W, int rows, const void* bias, int bias_dtype,
                                     void* C, int ldc, int M, int N, int K, int out_dtype, int silu, float* accum,
                                     int ldacc, hipStream_t stream) {
    if (M <= 0 || N <= 0) return TM_OK;
    const int relu2 = silu == 2;            // as in tm_gemm_skinny
    if (relu2) silu = 0;
    if (accum && (silu || ldacc < N)) return TM_ERR_ARG;
    if (!accum && !C) return TM_ERR_ARG;
    if (M > 16 || K <= 0 || (K % 8) || (lda % 8) || lda < K || ldc < N || ((uintptr_t)A % 16) || ((uintptr_t)W % 16) ||
        (rows != 16 && rows != 8 && rows != 4) || (silu && (rows != 16 || bias)))
        return TM_ERR_ARG;
    const int flags = (bias_dtype == TM_F32 ? SK_BIAS_F32 : 0) | (relu2 ? SK_RELU2 : 0);    // the kernel's flags
    if (out_dtype == TM_BF16)
        return silu ? launch_skinny_packed<true, bf16_t>(A, lda, W, rows, bias, flags, C, ldc, M, N, K, accum, ldacc, stream)
                    : launch_skinny_packed<false, bf16_t>(A, lda, W, rows, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    if (out_dtype == TM_F32 && !silu) return launch_skinny_packed<false, float>(A, lda, W, rows, bias, flags, C, ldc, M, N, K, accum, ldacc, stream);
    return TM_ERR_ARG;
}
