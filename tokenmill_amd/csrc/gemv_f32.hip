// The true 32-bit path's products of at most 16 rows (decode steps), on the 32-bit matrix unit: a plain product (with bias, or as
// 32-bit partial sums of a K split over blocks, which the next norm adds), gate|up with SiLU*up, q|k|v with bias, rotation and
// cache write.
//
// Such a product is bound by reading its matrix once (35 MB for gate|up of the 0.5B shape) and, where that is small, by the trips to
// memory. A block takes RT tiles of 16 matrix rows (SiLU and q|k|v: one, of 8 rows and the 8 that meet them, twice the blocks);
// its wavefronts split K into runs of steps of 16 k and ask for several steps of matrix and activations at once, so nothing goes through
// LDS but the wavefronts' sums at the end, added in wavefront order. The activations come from the second-level cache. Which k goes where
// depends on the matrix alone: a row's result does not depend on the other rows.
//
// The matrix instruction wants 16 bytes of row r at 4 g in lane (r, g): neighbouring lanes in different rows. A CU takes the addresses of a load
// in four lanes at a time where these lie beside each other, and one at a time where they do not, which was most of what small products took
// (64 clocks a load of 1 KB for 16). So four neighbouring lanes load 64 consecutive bytes, and the exchange that puts the pieces where the
// instruction wants them (lane (4 q + p, g) holds row 4 q + g at piece p, and wants row 4 q + p at piece g) is four ds_bpermute a load, which
// pass no memory; where that costs more than it gains (gm_turns) the lanes load in the instruction's order. Matrices of 6.5 MB and more (GM_LINES) are
// loaded two steps at a time, 128 bytes of eight rows an instruction, whole lines that pass the caches by (non-temporal), halves of lines would come from HBM
// twice as slowly; the step's parity lies in lane bit 4, where one instruction a register changes it for the row's lowest bit (in the instruction's
// order in bit 3: line_pair_half). The activations go the same way; one row of them is asked for as the
// instruction wants it, all sixteen lanes of a piece at one place. us with the loads in the instruction's order / now, cold matrices:
// q|k|v of the 0.5B shape at 1 / 8 / 16 rows 5.66 / 4.97, 6.40 / 5.65, 7.31 / 6.47, o 4.85 / 4.38, 5.58 / 5.07, 6.51 / 5.74, down 6.34 / 6.25, 7.25 / 6.56, 8.62 / 7.53, gate|up
// at 8 / 16 10.4 / 10.3, 12.3 / 11.2; 3,584 -> 2 x 18,944 at 8 / 16 106 / 91, 127 / 104, back at 2 / 8 46.2 / 44.5, 53.9 / 46.2; 2,048 -> 1,536 at 1 / 8 / 16
// 7.0 / 6.6, 8.2 / 7.7, 9.7 / 8.4. The same bits.
// Before that, a wavefront had 256 k of four rows, a lane 4 k each, and summed over the lanes by shuffles, 6 x 32 of them a wavefront:
// 19.0 us a product of the 0.5B shape on average, with SiLU*up and rotation in kernels behind it.
#include "common.h"
#include "api.h"

#include <type_traits>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

enum { GM_PLAIN = 0, GM_SILU = 1, GM_QKV = 2 };

struct GemvArgs {
    const float* A;             // [M, K], rows lda apart
    const float* W;             // [rows, K]
    const float* bias;          // [rows] or null
    float* C;                   // [M, N] rows ldc apart; SiLU: [M, I]; q|k|v: q [M, H D]
    float* parts;               // [gridDim.y][M][N] instead of C, or null
    int lda, ldc, M, N, K;
    int I;
    int H, KVH, D, page_shift;
    const float* cos_t;         // [positions, D / 2]
    const float* sin_t;
    const int* positions;
    const int* slots;           // or null
    float* k_pool;              // [pages, page, KVH, D]
    float* v_pool;              // [pages, KVH, D, page]
};

// GROUP: steps of 16 k whose products meet in sums of their own before they join the running one. AHEAD: groups a wavefront asks for
// at once: with one, a wavefront of the 0.5B shape waited for memory two times in a launch of 6 to 7 us (o 6.2 to 5.8, q|k|v 7.2 to 6.8).
// LINES: two steps as a pair of lines, else a load a step. ROWS: rows of activations that there are places for, 1, 8 (of a pair of lines: one
// load) or 16.
template <int EPI, int RT, int WAVES, int GROUP, int AHEAD, bool LINES, int ROWS, bool TURN>
__global__ __launch_bounds__(64 * WAVES) void gemv_mfma_f32_kernel(const GemvArgs a) {
    static_assert(EPI == GM_PLAIN || RT == 1, "");
    __shared__ __align__(16) f32x4_t red[WAVES][RT][TM_WAVE];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int u = blockIdx.x;
    // the first rows of the tiles
    int n0[RT], head = 0, j0 = 0;
    int far = 0;                                                // SiLU, q|k|v: how far on the rows of the tile's second half are
    if constexpr (EPI == GM_SILU) {                             // 8 gate rows and the 8 up rows that meet them
        n0[0] = 8 * u;
        far = a.I;
    } else if constexpr (EPI == GM_QKV) {                       // 8 channels of a head and the 8 they are rotated with
        const int per_head = a.D / 16;
        head = u / per_head;
        j0 = 8 * (u - head * per_head);
        n0[0] = head * a.D + j0;
        far = a.D / 2;
    } else {
#pragma unroll
        for (int t = 0; t < RT; ++t) n0[t] = (u * RT + t) * 16;
    }
    const int steps = a.K / 16;
    const int per_block = (steps + gridDim.y - 1) / gridDim.y;
    const int b0 = blockIdx.y * per_block, b1 = b0 + per_block < steps ? b0 + per_block : steps;
    const int per = (per_block + WAVES - 1) / WAVES;
    const int s0 = b0 + wave * per, s1 = s0 + per < b1 ? s0 + per : b1;
    // What a lane loads: 16 bytes at 4 * piece of a step of row 4 q + g, q = r / 4; of a pair of lines of the step whose parity is g's lower
    // bit, of rows 4 q + 2 (g / 2) + h. (Rows beyond the matrix, the half or the input: its last one, never stored.)
    static_assert(LINES || ROWS != 8, "");
    constexpr int HALVES = LINES ? 2 : 1;
    constexpr bool WHOLE = GROUP == 4 && (LINES || AHEAD == 1); // a full group's operands are all turned before its first product: 4,096 -> 4,096 at 8 rows 16.1 to 15.4
    const int q = r / 4, piece = TURN ? r % 4 : g, parity = !LINES ? 0 : TURN ? g % 2 : r / 8;
    // where a lane gets row r at piece g from, in bytes of lanes (eight rows of a pair of lines: the other step 16 lanes on)
    const int turn = 4 * (16 * (r % 4) + 4 * q + g);
    const int turn_x = LINES && ROWS == 8 ? 4 * (32 * (r % 2) + 4 * (r % 8 / 2) + g) : turn;
    const float* pa[HALVES];
    const float* pw[RT][HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
        const int row = !TURN ? (LINES ? r % 8 + 8 * h : r) : LINES ? 4 * q + 2 * (g / 2) + h : 4 * q + g, of = TURN && LINES && ROWS == 8 ? 2 * q + g / 2 : row;
        pa[h] = ROWS == 1 ? a.A + 4 * g : a.A + (size_t)(of < a.M ? of : a.M - 1) * a.lda + 4 * piece;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int end = EPI == GM_SILU ? a.I : a.N, at = n0[t] + (EPI == GM_PLAIN ? row : row % 8);
            const int n = (at < end ? at : end - 1) + (EPI != GM_PLAIN ? row / 8 * far : 0);
            pw[t][h] = a.W + (size_t)n * a.K + 4 * piece;
        }
    }
    auto turned = [&](int from, f32x4_t v) {
        f32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(v[e])));
        return o;
    };
    auto pair_half = [&](int half, f32x4_t lo, f32x4_t hi) {    // lane bit 4, the step's parity, changes places with h
        f32x4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(lo[e]), __float_as_uint(hi[e]), false, false)[half]);
        return o;
    };
    // What the epilogue waits for otherwise: the positions are asked for before the matrix (loads come back in their order), the
    // rotary rows, whose place hangs on them, behind its first round.
    int pos = 0, slot = -1;
    f32x4_t bias0 = {0.f, 0.f, 0.f, 0.f}, bias1 = bias0, cosv = bias0, sinv = bias0;
    const int ge = EPI == GM_PLAIN ? g : g % 2;                 // (SiLU, q|k|v: lanes beyond the tile's eight rows have no epilogue)
    if constexpr (EPI == GM_QKV) {
        const int row = r < a.M ? r : a.M - 1;
        pos = a.positions[row];
        slot = (a.slots ? a.slots : a.positions)[row];
        if (a.bias) {
            bias0 = *(const f32x4_t*)(a.bias + n0[0] + 4 * ge);
            bias1 = *(const f32x4_t*)(a.bias + n0[0] + far + 4 * ge);
        }
    }
    f32x4_t sum[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) sum[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto groups = [&](auto AT_ONCE, int s) {
        constexpr int GROUPS = decltype(AT_ONCE)::value, LOADS = LINES ? (GROUP * GROUPS + 1) / 2 : GROUP * GROUPS;
        f32x4_t w[RT][LOADS][HALVES], x[LOADS][LINES && ROWS == 16 ? 2 : 1];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int step = LINES ? s + 2 * i + parity : s + i, at = 16 * (step < s1 ? step : s1 - 1);  // (no load under a test: beyond the end the last step again)
            const int one = s + 2 * i + r / 8, at_one = 16 * (one < s1 ? one : s1 - 1);      // (one row: lanes r < 8 the first step, the others the second)
#pragma unroll
            for (int h = 0; h < HALVES; ++h) {
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    const f32x4_t* at_w = (const f32x4_t*)(pw[t][h] + at);
                    w[t][i][h] = LINES ? __builtin_nontemporal_load(at_w) : *at_w;
                }
                if (h == 0 || ROWS == 16) x[i][h] = *(const f32x4_t*)(pa[h] + (ROWS == 1 && LINES ? at_one : at));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (EPI == GM_QKV) {
            if (s == s0) {
                const size_t at = (size_t)pos * (a.D / 2) + j0 + 4 * ge;
                cosv = *(const f32x4_t*)(a.cos_t + at);
                sinv = *(const f32x4_t*)(a.sin_t + at);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        auto operands = [&](int i, f32x4_t& xf, f32x4_t (&wf)[RT]) {
            if constexpr (LINES) {
                if constexpr (ROWS == 1) xf = i % 2 ? line_pair_turned(x[i / 2][0]) : x[i / 2][0];
                else if constexpr (ROWS == 8) xf = TURN ? turned(turn_x + 64 * (i % 2), x[i / 2][0]) : i % 2 ? line_pair_turned(x[i / 2][0]) : x[i / 2][0];
                else xf = TURN ? turned(turn, pair_half(i % 2, x[i / 2][0], x[i / 2][1])) : line_pair_half(i % 2, x[i / 2][0], x[i / 2][1]);
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    wf[t] = TURN ? turned(turn, pair_half(i % 2, w[t][i / 2][0], w[t][i / 2][1])) : line_pair_half(i % 2, w[t][i / 2][0], w[t][i / 2][1]);
            } else {
                xf = ROWS == 1 || !TURN ? x[i][0] : turned(turn, x[i][0]);
#pragma unroll
                for (int t = 0; t < RT; ++t) wf[t] = TURN ? turned(turn, w[t][i][0]) : w[t][i][0];
            }
        };
#pragma unroll
        for (int j = 0; j < GROUPS; ++j) {
            if (s + j * GROUP >= s1) break;                     // the same for the whole wavefront
            // four sums a tile, of every fourth k, that join the running one here: short chains of roundings
            f32x4_t acc[RT][4];
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[t][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (WHOLE && s + (j + 1) * GROUP <= s1) {
                f32x4_t xf[GROUP], wf[GROUP][RT];
#pragma unroll
                for (int k = 0; k < GROUP; ++k) operands(j * GROUP + k, xf[k], wf[k]);
#pragma unroll
                for (int k = 0; k < GROUP; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int t = 0; t < RT; ++t)
                            acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k][t][e], xf[k][e], acc[t][e], 0, 0, 0);
            } else
#pragma unroll
            for (int i = j * GROUP; i < (j + 1) * GROUP; ++i) {
                if (s + i >= s1) break;
                f32x4_t xf, wf[RT];
                operands(i, xf, wf);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        acc[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[t][e], xf[e], acc[t][e], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < RT; ++t) sum[t] += (acc[t][0] + acc[t][1]) + (acc[t][2] + acc[t][3]);
        }
    };
    // what is left when no AHEAD groups are is one group less (two tiles have no registers for the second loop: it takes the head from 98 to
    // 151 us at 16 rows, and what they ask for beyond the end is the last step again)
    int s = s0;
    constexpr int LEAST = LINES && RT == 1 ? GROUP * (AHEAD - 1) : 0;
    for (; s + LEAST < s1; s += GROUP * AHEAD) groups(std::integral_constant<int, AHEAD>{}, s);
    if constexpr (LEAST > 0) {
        if (s < s1) groups(std::integral_constant<int, AHEAD - 1>{}, s);
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) red[wave][t][lane] = sum[t];
    __syncthreads();
    // lane (r, g): row r of A, rows 4 g .. + 3 of the tile
    if (EPI == GM_PLAIN ? wave >= RT : wave > 0 || g >= 2) return;
    auto total = [&](int t, int of) {
        f32x4_t v = red[0][t][of];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += red[w][t][of];
        return v;
    };
    if constexpr (EPI == GM_PLAIN) {
        const int n = n0[0] + 16 * wave + 4 * g;
        if (r >= a.M || n >= a.N) return;                       // N is a multiple of 4: a piece is whole or absent
        f32x4_t v = total(wave, lane);
        if (a.parts) {
            *(f32x4_t*)(a.parts + ((size_t)blockIdx.y * a.M + r) * a.N + n) = v;
            return;
        }
        if (a.bias) v += *(const f32x4_t*)(a.bias + n);
        *(f32x4_t*)(a.C + (size_t)r * a.ldc + n) = v;
    } else if constexpr (EPI == GM_SILU) {
        const int c = n0[0] + 4 * g;
        if (r >= a.M || c >= a.I) return;
        const f32x4_t gt = total(0, lane), up = total(0, lane + 32);
        f32x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gt[e] / (1.f + expf(-gt[e])) * up[e];
        *(f32x4_t*)(a.C + (size_t)r * a.ldc + c) = v;
    } else {
        if (r >= a.M) return;
        f32x4_t x = total(0, lane), y = total(0, lane + 32);
        if (a.bias) {
            x += bias0;
            y += bias1;
        }
        if (!a.slots) slot = -1;
        const int d = j0 + 4 * g;
        if (head < a.H + a.KVH) {
            f32x4_t y1, y2;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float p, q;
                rotate_pair(x[e], y[e], cosv[e], sinv[e], p, q);
                y1[e] = p;
                y2[e] = q;
            }
            float* dst = nullptr;
            if (head < a.H) dst = a.C + (size_t)r * a.ldc + head * a.D + d;
            else if (slot >= 0) dst = a.k_pool + ((size_t)slot * a.KVH + (head - a.H)) * a.D + d;
            if (dst) {
                *(f32x4_t*)dst = y1;
                *(f32x4_t*)(dst + a.D / 2) = y2;
            }
        } else if (slot >= 0) {
            const int vh = head - a.H - a.KVH;
            const int pg = slot >> a.page_shift, in_page = slot & ((1 << a.page_shift) - 1);
            float* dst = a.v_pool + ((((size_t)pg * a.KVH + vh) * a.D + d) << a.page_shift) + in_page;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dst[(size_t)e << a.page_shift] = x[e];
                dst[(size_t)(a.D / 2 + e) << a.page_shift] = y[e];
            }
        }
    }
}

static bool gm_aligned16(const void* p) { return p && ((uintptr_t)p % 16) == 0; }

// Whole 16-byte pieces, k in whole steps of 16.
extern "C" int tm_gemv_f32_mfma_takes(const void* A, int lda, const void* W, const void* bias, int M, int N, int K) {
    return M > 0 && M <= 16 && N > 0 && N % 4 == 0 && K >= 16 && K % 16 == 0 && lda >= K && lda % 4 == 0 && gm_aligned16(A) && gm_aligned16(W) &&
           (!bias || gm_aligned16(bias));
}

// Up to a block a CU, eight wavefronts split K into groups of four steps; more blocks than that have four wavefronts with groups of seven, whose
// blocks a CU hide each other's waits. A wavefront of the eight that has up to three groups asks for all of them at once; with more, of
// up to four rows, or where nearly every CU has a block, two groups at a time, else one (one group / two, us: 18,944 -> 3,584, 8 / 16 rows, 224 blocks
// 58.7 / 51.4, 65.7 / 61.4; 4,096 -> 4,096, 256 blocks 15.4 / 14.8, 17.3 / 16.5; 8,960 -> 1,536, 192 blocks 18.7 / 19.3, 22.1 / 22.9; 2,048 -> q|k|v of 2,560, 160
// blocks 8.8 / 9.0, 9.7 / 10.3). One of the four
// asks for two groups where it has them: a group at a time leaves half a pair's line, and gate|up of the 0.5B shape takes 12.2 us so for 10.2.
// Of the products with a load a step (GM_LINES), more than three groups a wavefront are asked for one at a time whatever the rows are (2,048 -> 2,048 cut
// into 16 steps a wavefront, 1 / 8 / 16 rows: two rounds of three groups 9.4 / 11.5 / 13.5 us, four of one 7.7 / 8.6 / 10.0).
constexpr size_t GM_LINES = 6656 * 1024;
constexpr int GM_LINES_K = 384;

template <int EPI, int RT, bool LINES, int ROWS, bool TURN>
static void gm_launch_rows(const GemvArgs& a, int units, int split, hipStream_t stream) {
    const int steps = (a.K / 16 + split - 1) / split, per = (steps + 7) / 8;
    const bool long_runs = LINES && per > 12 && (a.M <= 4 || (TURN && units * split >= 224));
    const dim3 grid(units, split);
    if (units * split > 256) {
        if constexpr (LINES) {
            if (steps > 4 * 7) {
                gemv_mfma_f32_kernel<EPI, RT, 4, 7, 2, LINES, ROWS, TURN><<<grid, 256, 0, stream>>>(a);
                return;
            }
        }
        gemv_mfma_f32_kernel<EPI, RT, 4, 7, 1, LINES, ROWS, TURN><<<grid, 256, 0, stream>>>(a);
        return;
    }
    if constexpr (LINES || RT == 1) {                           // (two tiles without lines: K of less than 384)
        if (per > 4 && (per <= 8 || long_runs)) {
            gemv_mfma_f32_kernel<EPI, RT, 8, 4, 2, LINES, ROWS, TURN><<<grid, 512, 0, stream>>>(a);
            return;
        }
        if (per > 8 && per <= 12) {
            gemv_mfma_f32_kernel<EPI, RT, 8, 4, 3, LINES, ROWS, TURN><<<grid, 512, 0, stream>>>(a);
            return;
        }
    }
    gemv_mfma_f32_kernel<EPI, RT, 8, 4, 1, LINES, ROWS, TURN><<<grid, 512, 0, stream>>>(a);
}

template <int EPI, int RT, bool LINES, bool TURN>
static void gm_launch_lines(const GemvArgs& a, int units, int split, hipStream_t stream) {
    if (a.M == 1) {
        gm_launch_rows<EPI, RT, LINES, 1, TURN>(a, units, split, stream);
        return;
    }
    if constexpr (LINES) {
        if (a.M <= 8) {
            gm_launch_rows<EPI, RT, LINES, 8, TURN>(a, units, split, stream);
            return;
        }
    }
    gm_launch_rows<EPI, RT, LINES, 16, TURN>(a, units, split, stream);
}

// Four neighbouring lanes side by side (TURN), or the instruction's order? Lines: matrices loaded as pairs of lines; per: steps a wavefront has.
// The exchange behind the loads costs a wavefront some hundreds of cycles a group, which it has to gain at the loads. It does not
//  - where rows are no whole lines (K % 32 = 16), so that the four lanes' 64 bytes lie in two: pairs of lines at 2 and 8 rows, K 720, 1,296 and 1,552, 3,584 to
//    32,000 columns, 1.03 to 1.08 of the time of the other order (M 16, 1.02 to 1.1), a load a step with K of 176 to 464 1.01 to 1.08, below and above 0.85 to 0.99;
//  - where more blocks than CUs have wavefronts of two groups of seven at once (K 768 to 896): of the 0.5B shape's head 1.04, 1.05, 1.05, 1.02 and 1.05 at 1 / 2 / 4 / 8 / 9
//    rows (0.99 at 16), 896 -> 16,384 1.07 to 1.11 (1.04), 896 -> 6,144 1.04, 1.06, 1.03, 0.97, 1.01, gate|up 1.02, 1.05, 1.04, 0.99 (12 rows: 0.94); K 640 0.94 to 1.03, K 960 0.8 to 0.92;
//  - at one row where a block is alone on its CU and not short (896 -> 4,096 1.03, 1,536 -> 3,584 1.07, 8,960 -> 4,096 1.05; K 512 0.96), and up to four if a
//    wavefront's groups are all asked for at once (1,536 -> 4,096 at 2 / 4 / 8 rows 1.06 / 1.03 / 0.99; 2,048 -> 4,096 0.97 / 0.96 / 0.92).
// Elsewhere, over 1,000 sizes, it is 0.92 on the mean, 0.58 to 1.04.
static bool gm_turns(int RT, bool lines, int K, int M, int blocks, int per) {
    if (K % 32) return !lines && (RT == 2 || K < 160 || K >= 512);
    if (!lines) return true;
    if (blocks > 256) return per < 12 || per > 14 || (RT == 2 ? M == 16 && blocks > 1024 : M > 4);
    return blocks < 224 || per < 7 || (M > 1 && (M > 4 || per > 12));
}

static bool gm_lines(int N, int K) { return (size_t)N * K * 4 >= GM_LINES && K >= GM_LINES_K; }
static bool gm_launch_turns(int RT, int M, int N, int K, int units, int split) {
    const int steps = (K / 16 + split - 1) / split, waves = units * split > 256 ? 4 : 8;
    return gm_turns(RT, gm_lines(N, K), K, M, units * split, (steps + waves - 1) / waves);
}

template <int EPI, int RT>
static void gm_launch(const GemvArgs& a, int units, int split, hipStream_t stream) {
    const bool lines = gm_lines(a.N, a.K), turn = gm_launch_turns(RT, a.M, a.N, a.K, units, split);
    if (lines && turn) gm_launch_lines<EPI, RT, true, true>(a, units, split, stream);
    else if (lines) gm_launch_lines<EPI, RT, true, false>(a, units, split, stream);
    else if (RT == 2 || turn) gm_launch_lines<EPI, RT, false, true>(a, units, split, stream);
    else if constexpr (RT == 1) gm_launch_lines<EPI, RT, false, false>(a, units, split, stream);
}

// two tiles a block read the activations once for both, where that still gives every CU a block
static bool gm_two_tiles(int N) { return (N + 31) / 32 >= 256; }

// Do neighbouring lanes of the plain product load what lies side by side? (for tests)
extern "C" int tm_gemv_f32_turns(int M, int N, int K) {
    return gm_two_tiles(N) ? gm_launch_turns(2, M, N, K, (N + 31) / 32, 1) : gm_launch_turns(1, M, N, K, (N + 15) / 16, 1);
}

extern "C" int tm_gemv_f32_mfma(const float* A, int lda, const float* W, const float* bias, float* C, int ldc, int M, int N, int K,
                                hipStream_t stream) {
    if (!tm_gemv_f32_mfma_takes(A, lda, W, bias, M, N, K) || !gm_aligned16(C) || ldc < N || ldc % 4) return TM_ERR_ARG;
    GemvArgs a{};
    a.A = A; a.W = W; a.bias = bias; a.C = C; a.lda = lda; a.ldc = ldc; a.M = M; a.N = N; a.K = K;
    if (gm_two_tiles(N)) gm_launch<GM_PLAIN, 2>(a, (N + 31) / 32, 1, stream);
    else gm_launch<GM_PLAIN, 1>(a, (N + 15) / 16, 1, stream);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// Parts that K is split into where 16-row tiles are too few for the chip (a part keeps at least 32 steps of 16 k, two a wavefront).
extern "C" int tm_gemv_f32_parts(int N, int K) {
    const int units = (N + 15) / 16;
    int parts = 1;
    while (parts < 8 && units * parts * 2 <= 256 && K / 16 / (parts * 2) >= 32) parts *= 2;
    return parts;
}

// parts[p][m][n], p < tm_gemv_f32_parts(N, K)
extern "C" int tm_gemv_f32_mfma_split(const float* A, int lda, const float* W, float* parts, int M, int N, int K, hipStream_t stream) {
    if (!tm_gemv_f32_mfma_takes(A, lda, W, nullptr, M, N, K) || !gm_aligned16(parts)) return TM_ERR_ARG;
    GemvArgs a{};
    a.A = A; a.W = W; a.parts = parts; a.lda = lda; a.M = M; a.N = N; a.K = K;
    const int units = (N + 15) / 16;
    gm_launch<GM_PLAIN, 1>(a, units, tm_gemv_f32_parts(N, K), stream);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// act[m, i] = silu(gate) * up, W [2 I, K]
extern "C" int tm_gemv_f32_gate_up_silu(const float* A, int lda, const float* W, float* act, int M, int I, int K, hipStream_t stream) {
    if (I <= 0 || I % 4 || !gm_aligned16(act) || !tm_gemv_f32_mfma_takes(A, lda, W, nullptr, M, 2 * I, K)) return TM_ERR_ARG;
    GemvArgs a{};
    a.A = A; a.W = W; a.C = act; a.lda = lda; a.ldc = I; a.M = M; a.N = 2 * I; a.K = K; a.I = I;
    gm_launch<GM_SILU, 1>(a, (I + 7) / 8, 1, stream);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

// as tm_tile_qkv_rope, in 32-bit; head sizes that are multiples of 32
extern "C" int tm_gemv_f32_qkv_rope(const float* A, int lda, const float* W, const float* bias, float* q, int M, int K, int H, int KVH, int D,
                                    const float* cos_t, const float* sin_t, const int* positions, const int* slots, float* k_pool,
                                    float* v_pool, int page, hipStream_t stream) {
    const int N = (H + 2 * KVH) * D;
    if (H <= 0 || KVH <= 0 || D <= 0 || D % 32 || !gm_aligned16(q) || !gm_aligned16(cos_t) || !gm_aligned16(sin_t) || !positions || page <= 0 ||
        (page & (page - 1)) || (slots && (!gm_aligned16(k_pool) || !v_pool)) || !tm_gemv_f32_mfma_takes(A, lda, W, bias, M, N, K))
        return TM_ERR_ARG;
    GemvArgs a{};
    a.A = A; a.W = W; a.bias = bias; a.C = q; a.lda = lda; a.ldc = H * D; a.M = M; a.N = N; a.K = K;
    a.H = H; a.KVH = KVH; a.D = D; a.cos_t = cos_t; a.sin_t = sin_t; a.positions = positions; a.slots = slots; a.k_pool = k_pool; a.v_pool = v_pool;
    while ((1 << a.page_shift) < page) ++a.page_shift;
    gm_launch<GM_QKV, 1>(a, N / 16, 1, stream);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
