// A wide product of at most 16 bfloat16 rows into 32-bit results (the output head: logits of the rows that are sampled), over the
// row-major matrix.
//
// It is bound by reading the matrix once, 272 MB at the 0.5B shape, so the loads are whole lines: two steps of 32 k of eight rows an instruction, 128 bytes of
// each, passing the caches by; lanes exchange what belongs to rows of the other eight (line_pair_half). A block takes RT tiles of
// 16 matrix rows, which share the activations, its wavefronts split K and their sums meet in LDS, in halves. Which k goes where depends on the matrix alone.
// choose.h says which heads it takes (tm_head_few). Against the library's product, cold matrices, us: 151,936 x 896 at 1 / 8 rows 51 / 52 to 40 / 44, 152,064 x 3,584 226 / 239 to 164 / 170 (6.6 and 6.4 TB/s).
#include "common.h"
#include "api.h"

#include <type_traits>

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

union GvFrag {
    u32x4_t u;
    bf16x8_t b;
};

constexpr int GV_WAVES = 4;

// STEPS: k-steps a wavefront asks for at once. OVER8: more than eight rows of activations.
template <int RT, int STEPS, bool OVER8>
__global__ __launch_bounds__(64 * GV_WAVES) void gemv_bf16_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, float* __restrict__ C,
                                                                  int ldc, int M, int N, int K) {
    static_assert(STEPS % 4 == 0 && RT <= GV_WAVES, "");
    __shared__ __align__(16) f32x4_t red[GV_WAVES][RT][TM_WAVE];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16, r8 = r % 8, second = r / 8;
    const int n0 = blockIdx.x * RT * 16;
    const int steps = K / 32, per = (steps + 2 * GV_WAVES - 1) / (2 * GV_WAVES) * 2;    // whole pairs
    const int s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;
    // rows r % 8 and 8 + r % 8 (rows beyond the matrix or the input: its last one, never stored)
    const bf16_t *pa[2], *pw[RT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = r8 + 8 * h;
        pa[h] = A + (size_t)(row < M ? row : M - 1) * lda + 8 * g;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int n = n0 + 16 * t + row;
            pw[t][h] = W + (size_t)(n < N ? n : N - 1) * K + 8 * g;
        }
    }
    f32x4_t acc[RT][2];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t][0] = acc[t][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto round = [&](auto AT_ONCE, int s) {
        constexpr int COUNT = decltype(AT_ONCE)::value;
        u32x4_t w[COUNT / 2][RT][2], x[COUNT / 2][OVER8 ? 2 : 1];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < COUNT / 2; ++i) {
            const int step = s + 2 * i + second, at = 32 * (COUNT > 2 || step < s1 ? step : s1 - 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (h == 0 || OVER8) x[i][h] = *(const u32x4_t*)(pa[h] + at);
#pragma unroll
                for (int t = 0; t < RT; ++t) w[i][t][h] = __builtin_nontemporal_load((const u32x4_t*)(pw[t][h] + at));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < COUNT; ++i) {
            if (COUNT == 2 && s + i >= s1) break;                   // (half a pair at the end of K; the same for the whole wavefront)
            GvFrag xf, wf;
            xf.u = OVER8 ? line_pair_half(i % 2, x[i / 2][0], x[i / 2][OVER8 ? 1 : 0]) : i % 2 ? line_pair_turned(x[i / 2][0]) : x[i / 2][0];
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                wf.u = line_pair_half(i % 2, w[i / 2][t][0], w[i / 2][t][1]);
                acc[t][i % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.b, xf.b, acc[t][i % 2], 0, 0, 0);
            }
        }
    };
    // whole rounds, then a half one and pairs (a load under a test would be put behind it)
    int s = s0;
    for (; s + STEPS <= s1; s += STEPS) round(std::integral_constant<int, STEPS>{}, s);
    for (; s + STEPS / 2 <= s1; s += STEPS / 2) round(std::integral_constant<int, STEPS / 2>{}, s);
    for (; s < s1; s += 2) round(std::integral_constant<int, 2>{}, s);
#pragma unroll
    for (int t = 0; t < RT; ++t) red[wave][t][lane] = acc[t][0] + acc[t][1];
    __syncthreads();
    // lane (r, g) of wavefront t: row r of A, rows 4 g .. + 3 of tile t
    const int n = n0 + 16 * wave + 4 * g;
    if (wave >= RT || r >= M || n >= N) return;                     // N is a multiple of 4: a piece is whole or absent
    f32x4_t v[GV_WAVES];
#pragma unroll
    for (int k = 0; k < GV_WAVES; ++k) v[k] = red[k][wave][lane];
    *(f32x4_t*)(C + (size_t)r * ldc + n) = (v[0] + v[2]) + (v[1] + v[3]);
}

static bool gv_aligned(const void* p) { return p && ((uintptr_t)p % 16) == 0; }

// Whole 16-byte pieces, k in whole steps of 32, and a block a CU at the least.
extern "C" int tm_gemv_bf16_takes(const void* A, int lda, const void* W, const void* C, int ldc, int M, int N, int K) {
    return M > 0 && M <= 16 && N >= 16384 && N % 4 == 0 && K >= 32 && K % 32 == 0 && lda >= K && lda % 8 == 0 && ldc >= N && ldc % 4 == 0 && gv_aligned(A) &&
           gv_aligned(W) && gv_aligned(C);
}

extern "C" int tm_gemv_bf16(const void* A, int lda, const void* W, float* C, int ldc, int M, int N, int K, hipStream_t stream) {
    if (!tm_gemv_bf16_takes(A, lda, W, C, ldc, M, N, K)) return TM_ERR_ARG;
    // two tiles a block, or, where the activations are two loads a pair, four (151,936 x 896 and 152,064 x 3,584 at 8 rows 43.9 and 170.1 us with two,
    // 45.0 and 176.4 with four; at 16 rows 52.3 and 195.9, 49.6 and 189.0; twice the steps at once are 49 us at one row for 40)
    const int tiles = M > 8 ? 4 : 2, blocks = (N + 16 * tiles - 1) / (16 * tiles);
    if (M > 8) gemv_bf16_kernel<4, 8, true><<<blocks, 64 * GV_WAVES, 0, stream>>>((const bf16_t*)A, lda, (const bf16_t*)W, C, ldc, M, N, K);
    else gemv_bf16_kernel<2, 8, false><<<blocks, 64 * GV_WAVES, 0, stream>>>((const bf16_t*)A, lda, (const bf16_t*)W, C, ldc, M, N, K);
    TM_CHECK_LAUNCH();
    return TM_OK;
}
