// Matrix products of prompt-sized steps on the bfloat16 matrix unit, each with its layer's own epilogue: gate|up with SiLU*up;
// q|k|v with bias, rotation and cache write; a plain store; 32-bit partial sums of a product A W^T whose K is split over groups of blocks (or is
// not, one part); the products of experts. The same kernel on the 32-bit matrix unit is the true 32-bit path's.
//
// A block of four wavefronts computes a tile of BM rows by BN matrix rows, BM x BN / 4 a wavefront, k in steps of 64. Both
// operands come straight into LDS (16 bytes a lane, no registers in between) into a ring of ST buffers, ST - 1 to ST steps
// ahead of the products; a wavefront waits for its own loads of a step by count and meets the others at one barrier a step.
// The operand fragments of half a step (32 k) are read from LDS while the half before is multiplied. The blocks stay: each
// walks tiles b, b + gridDim.x, ... as ONE stream of steps, so the loads of the next tile are on their way while a tile's
// epilogue stores, and the ring never runs empty inside a launch.
//
// LDS. A load instruction of a wavefront fills 1,024 bytes in lane order: eight rows of 128 bytes. Lane l brings row l / 8 and,
// of its eight 16-byte pieces, the one whose place in the row is l % 8 after the XOR below, so an operand load (lane (r, g):
// piece g of row r) meets no bank twice and the global side still reads whole 128-byte lines.
//
// Which matrix row an LDS row holds is the epilogue's choice: 64 LDS rows are a "unit", for SiLU 32 gate rows and the 32 up
// rows that meet them, for q|k|v 32 channels of a head and the 32 they are rotated with, else 64 consecutive rows. A pair of
// 16-row matrix tiles takes its rows in the order 8 (r / 4) + r % 4 (+ 4), so that a lane ends with eight consecutive
// columns of a row of C: 16-byte stores.
#include "common.h"
#include "api.h"
#include "fused_common.h"
#include "ahead.h"

#include <type_traits>

enum { GT_SILU = 0, GT_QKV = 1, GT_PARTS = 2, GT_STORE = 3, GT_EXPERT_SILU = 4, GT_EXPERT_CLAMPED = 5, GT_EXPERT_RELU2 = 6, GT_EXPERT_DOWN = 7 };

struct TileArgs {
    const void* A;              // [M, K], rows lda apart
    const void* W;              // [rows, K]
    const void* bias;           // [rows] or null
    void* C;                    // [M, N] rows ldc apart; PARTS: float [split][M][N]
    int M, N, K, lda, ldc;      // N: matrix rows (SiLU: twice I)
    int bias_f32;
    int tiles_m, tiles_n, splits, band;
    int I;                      // SiLU: columns of the result
    // q|k|v
    int H, KVH, D, page_shift;
    uint32_t head_inverse;      // unit_inverse(D / 64)
    const float* cos_t;         // [positions, D / 2]
    const float* sin_t;
    const int* positions;       // [M]
    const int* slots;           // [M]; < 0: not stored; or null
    void* k_pool;               // [pages, page, KVH, D]
    void* v_pool;               // [pages, KVH, D, page]
    // experts: a matrix a group (W [groups, rows, K]); row tiles (group, first slot, slots) from the route, n_tiles[0] of them with up
    // to tile_rows slots, which blocks take BM at a time; slot i reads row row_src[i] / src_div of A (row_src null: row i)
    const int* tiles;
    const int* n_tiles;
    const int* row_src;
    int src_div, tile_rows;
    const float* pair_weight;   // clamped gate: [pairs], multiplies the products of slot i by pair_weight[row_src[i]]; or null
    float limit, alpha;
    int grid;                   // blocks that walk tiles
};

// Where a tile lies.
struct GtPlace {
    int tn, sp;                 // column tile, part of K
    int m0, end;                // its rows: m0 .. end - 1 at most
    int group;
};

// An operand fragment: 16 bytes of a row, 8 bfloat16 or 4 float32 values
union GtFrag {
    u32x4_t u;
    bf16x8_t b;
    f32x4_t f;
};

// eight results of a row in the tensors' type, 16-byte stores
template <typename T>
__device__ __forceinline__ void gt_store8(T* dst, const float (&v)[8]) {
    if constexpr (sizeof(T) == 4) {
        *(f32x4_t*)dst = f32x4_t{v[0], v[1], v[2], v[3]};
        *(f32x4_t*)(dst + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
    } else {
        *(u32x4_t*)dst = u32x4_t{fd_pack(v[0], v[1]), fd_pack(v[2], v[3]), fd_pack(v[4], v[5]), fd_pack(v[6], v[7])};
    }
}

// two values rounded to the tensors' type and back, by one conversion
template <typename T>
__device__ __forceinline__ void gt_round2(float& a, float& b) {
    if constexpr (sizeof(T) == 4) return;
    const uint32_t u = fd_pack(a, b);
    a = __uint_as_float(u << 16);
    b = __uint_as_float(u & 0xffff0000u);
}

// x / (1 + exp(-x)). Of a bfloat16 x the division is a reciprocal, one correction of the quotient by its remainder and the unit's
// own last step for infinities; a quarter of both sides keeps the reciprocal of the largest divisors normal. The same bits as
// the division for every bfloat16 x, in seven instructions for eleven: at one wavefront a SIMD an epilogue's instructions are
// its time (2,048 rows of 896 -> 2 x 4,864, in a step: 4.3 us more than the one-instruction exponential and reciprocal, whose
// error is 3e-6 of the value at the far end where this one's is 1.3e-7; with the division itself 6.1 us more).
//
// exp(-x) after Cody and Waite: -x log2(e) from the constant's two parts, its whole number to the exponent, 2 to the rest by the hardware. x is
// held to +-128, where that ends in infinity and zero, in place of the two comparisons and choices that expf has behind it; the same
// bits for every bfloat16 x (gate|up with SiLU*up, launches in a row, 896 -> 2 x 4,864 at 300 / 541 / 1,024 / 2,048 rows 11.0 / 14.9 /
// 25.3 / 39.7 to 10.7 / 14.7 / 24.6 / 38.8 us).
__device__ __forceinline__ float gt_exp_minus(float x) {
#pragma clang fp contract(off)
    const float c = __builtin_amdgcn_fmed3f(x, -128.f, 128.f), t = c * -1.44269502f, n = __builtin_rintf(t);
    const float rest = fmaf(c, -1.92596299e-8f, fmaf(c, -1.44269502f, -t));
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((t - n) + rest), (int)n);
}
template <typename T>
__device__ __forceinline__ float gt_silu(float x) {
    if constexpr (sizeof(T) == 4) return x / (1.f + expf(-x));
    const float e = gt_exp_minus(x);
    const float n = 0.25f * x, d = fmaf(e, 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(d), q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}

template <int N>
__device__ __forceinline__ void gt_wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// ... until those of at most `left` steps (and MOST), NL a step, are on their way
template <int MOST, int NL>
__device__ __forceinline__ void gt_wait_steps(int left) {
    if constexpr (MOST > 0) {
        if (left < MOST) return gt_wait_steps<MOST - 1, NL>(left);
    }
    gt_wait_loads<MOST * NL>();
}

// Tile p of the launch. The blocks of one XCD (b % 8) walk a run of neighbouring tiles, `band` row tiles of a column tile first,
// so that what an XCD's blocks read at a time overlaps in its L2. False: no further tile.
template <bool GROUPED>
__device__ __forceinline__ bool gt_place(const TileArgs& a, int BM, int p, GtPlace& at) {
    const int per_entry = GROUPED ? a.tile_rows / BM : 1;
    const int tiles_m = GROUPED ? __builtin_amdgcn_readfirstlane(a.n_tiles[0]) * per_entry : a.tiles_m;
    const int total = tiles_m * a.tiles_n * a.splits;
    const int chunk = (total + 7) / 8;
    const int t = (p % 8) * chunk + p / 8;
    if (p / 8 >= chunk || t >= total) return false;
    at.sp = t / (tiles_m * a.tiles_n);
    const int in = t - at.sp * tiles_m * a.tiles_n;
    const int band = in / (a.band * a.tiles_n);
    const int rows = tiles_m - a.band * band < a.band ? tiles_m - a.band * band : a.band;
    const int q = in - band * a.band * a.tiles_n;
    at.tn = q / rows;
    const int tm = a.band * band + q - at.tn * rows;
    if (GROUPED) {
        const int* e = a.tiles + 3 * (tm / per_entry);
        const int first = __builtin_amdgcn_readfirstlane(e[1]);
        at.group = __builtin_amdgcn_readfirstlane(e[0]);
        at.m0 = first + tm % per_entry * BM;
        at.end = first + __builtin_amdgcn_readfirstlane(e[2]);
    } else {
        at.group = 0;
        at.m0 = tm * BM;
        at.end = a.M;
    }
    return true;
}

// ... or the next one behind it (the block's tiles are `stride` apart) that has a row
template <bool GROUPED>
__device__ __forceinline__ bool gt_next(const TileArgs& a, int BM, int stride, int& p, GtPlace& at) {
    while (gt_place<GROUPED>(a, BM, p, at)) {
        if (!GROUPED || at.m0 < at.end) return true;
        p += stride;
    }
    return false;
}

// the matrix row that row q of unit u holds
template <int EPI>
__device__ __forceinline__ int gt_matrix_row(const TileArgs& a, int u, int q) {
    int n;
    if (EPI == GT_SILU || EPI == GT_EXPERT_SILU || EPI == GT_EXPERT_CLAMPED) {
        n = 32 * u + (q & 31);
        n = n < a.I ? n : a.I - 1;
        if (q >= 32) n += a.I;
        return n;
    }
    if (EPI == GT_QKV) {
        const int per_head = a.D / 64, head = unit_head(u, a.head_inverse);
        n = head * a.D + 32 * (u - head * per_head) + (q & 31) + (q >= 32 ? a.D / 2 : 0);
    } else {
        n = 64 * u + q;
    }
    return n < a.N ? n : a.N - 1;
}

// MT, NT: 16-row tiles of A and of the matrix a wavefront multiplies; WM x WN = 4 wavefronts; ST: buffers of the ring
template <typename T, int EPI, int MT, int NT, int WM, int WN, int ST, int OCC, bool BRINGS = false>
__global__ __launch_bounds__(256, OCC) void gemm_tile_kernel(const TileArgs a, const TmAheadArg<BRINGS> ahead) {
    extern __shared__ __align__(16) unsigned char gt_smem[];
    if constexpr (BRINGS) {
        ahead_with(a.A, a.W, a.M, a.N, a.K, a.lda, a.tiles_m, a.tiles_n, a.splits, a.band, a.D, a.head_inverse, a.positions, a.slots, a.bias, a.bias_f32);
        if ((int)blockIdx.x >= a.grid) return tm_bring_ahead(ahead, blockIdx.x, 4);
    }
    const int stride = BRINGS ? a.grid : gridDim.x;
    constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN, ROWS = BM + BN;
    constexpr bool GROUPED = EPI >= GT_EXPERT_SILU, GATED = EPI == GT_SILU || EPI == GT_EXPERT_SILU || EPI == GT_EXPERT_CLAMPED;
    // Behind a block's last tile there is nothing to load. Tiles of a middle size load nothing then; the others load the same bytes
    // again, which keeps one loop and its waits: the smallest are bound by the length of a step and by their code's way into the CU (with
    // a second loop 896 -> 896 at 77 rows 4.1 to 4.3 us), the largest have no register left for it. What it gives the middle ones, 896 wide,
    // 2,048 rows: gate|up 40.6 to 40.2 us, down 27.8 to 27.5, o level.
    constexpr bool QUIET = sizeof(T) == 2 && MT >= 2 && MT <= 5;
    constexpr int STAGE = ROWS * 128, NL = ROWS / 32;               // bytes of a buffer; loads a wavefront makes for it
    static_assert(BM % 32 == 0 && BN % 64 == 0 && NT % 4 == 0, "");
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)gt_smem;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int r = lane % 16, g = lane / 16;
    const int wm = wave / WN, wn = wave % WN;
    constexpr int ES = sizeof(T), KSTEP = 128 / ES;                 // a step is 128 bytes of every row
    const int ksteps = a.K / KSTEP;
    const int per = (ksteps + a.splits - 1) / a.splits;             // k-steps of a part

    // --- the loading side: runs ahead of the products over the block's tiles ---
    uint32_t voff[NL];
    const unsigned char *lA = (const unsigned char*)a.A, *lW = (const unsigned char*)a.W;
    int l_p = blockIdx.x;
    bool l_more = true;
    auto next_load_tile = [&]() {
        GtPlace at_;
        if (!l_more || !gt_next<GROUPED>(a, BM, stride, l_p, at_)) {             // no further tile: nothing, or the same bytes again, never multiplied
            l_more = false;
            if constexpr (!QUIET) {
                lA = (const unsigned char*)a.A;
                lW = (const unsigned char*)a.W;
            }
            return;
        }
        l_p += stride;
        const int k0 = at_.sp * per;
        lA = (const unsigned char*)a.A + (size_t)k0 * 128;
        lW = (const unsigned char*)a.W + (size_t)k0 * 128 + (GROUPED ? (size_t)at_.group * a.N * a.K * ES : 0);
        const int in8 = lane / 8, at = lane % 8;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int R = (wave + 4 * i) * 8 + in8;                 // row of the buffer
            if (i < BM / 32) {
                int m = at_.m0 + R;
                m = m < at_.end ? m : at_.end - 1;
                if (GROUPED && a.row_src) m = a.row_src[m] / a.src_div;
                voff[i] = (uint32_t)m * (uint32_t)a.lda * ES + (uint32_t)((at ^ ((R >> 1) & 7)) * 16);
            } else {
                const int Rb = R - BM;
                const int n = gt_matrix_row<EPI>(a, at_.tn * (BN / 64) + Rb / 64, Rb % 64);
                voff[i] = (uint32_t)n * (uint32_t)a.K * ES + (uint32_t)((at ^ (((Rb >> 1) & 1) | (((Rb >> 3) & 3) << 1))) * 16);
            }
        }
    };
    auto issue_one = [&](uint32_t dst, int i) { fd_load_lds(dst + i * 4096, voff[i], i < BM / 32 ? (const void*)lA : (const void*)lW); };
    auto issued = [&]() {
        lA += QUIET || l_more ? 128 : 0;
        lW += QUIET || l_more ? 128 : 0;
    };

    // --- the multiplying side ---
    GtPlace at_;
    int p = blockIdx.x;
    if (!gt_next<GROUPED>(a, BM, stride, p, at_)) return;
    next_load_tile();
#pragma unroll
    for (int s = 0; s < ST; ++s) {                                  // (every part of K has at least ST steps)
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + s * STAGE + wave * 1024);
#pragma unroll
        for (int i = 0; i < NL; ++i) issue_one(dst, i);
        issued();
    }

    // 32-bit operands: the accumulators hold the sum of a block of k, which joins the running total at the block's end (one chain
    // of roundings over all of K loses several times what a blocked sum does). The block's chain and the chain of the blocks
    // both round: 64 k up to 7,680 k a part, 128 beyond (rms error of the result, one part, blocks of 32 / 64 / 128 k: K 896
    // 1.4 / 1.6 / 2.1e-7, 4,864 2.5 / 2.1 / 2.3e-7, 18,944 4.5 / 3.4 / 3.0e-7; within 1% of each other in time).
    const int joins = per > 240 ? 4 : 2;
    constexpr int TM_ = ES == 4 ? MT : 1, TN_ = ES == 4 ? NT : 1;
    f32x4_t acc[MT][NT], total[TM_][TN_];
    auto join = [&]() {
        if constexpr (ES == 4) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    total[i][j] += acc[i][j];
                    acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if constexpr (ES == 4) total[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
    };
    clear();
    GtFrag fa[2][MT], fb[2][NT];
    const int rb = 8 * (r / 4) + r % 4;
    const int offA = (wm * MT * 16 + r) * 128 + ((g ^ ((r >> 1) & 7)) << 4);
    const int offB = (BM + wn * NT * 16 + rb) * 128 + ((g ^ (((rb >> 1) & 1) | (((rb >> 3) & 3) << 1))) << 4);
    // One half of a step: the products of half `half`, and spread between them the reads of the other half's operands (from
    // buffer `from`) and, with dst, the loads of the step ST ahead. The order is the program's: the barriers between the groups
    // keep the compiler from gathering the reads.
    // 32-bit fragments are multiplied a quarter at a time, each quarter over all accumulators before the next, so that no instruction waits
    // for the one before it (against all four quarters of a pair in a row: gate|up of 100 / 1,000 / 1,500 rows of 896 35.9 / 146 / 220 to
    // 34.1 / 143 / 213 us, q|k|v of 300 20.6 to 19.5; the order of an accumulator's sums is the same).
    constexpr int READS = MT + NT, QUARTERS = ES == 4 ? 4 : 1, PRODUCTS = MT * NT * QUARTERS;
    auto multiply = [&](int half, int i) {
        const int n = i % (MT * NT), e = i / (MT * NT);
        const GtFrag &w = fb[half][n % NT], &x = fa[half][n / NT];
        f32x4_t& c = acc[n / NT][n % NT];
        if constexpr (ES == 4) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w.f[e], x.f[e], c, 0, 0, 0);
        else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.b, x.b, c, 0, 0, 0);
    };
    auto half_step = [&](auto HALF, int from, auto LOADS, uint32_t dst) {
        constexpr int half = decltype(HALF)::value, other = 1 - half;
        const unsigned char* pa = gt_smem + from * STAGE + (offA ^ (other * 64));
        const unsigned char* pb = gt_smem + from * STAGE + (offB ^ (other * 64));
#pragma unroll
        for (int q = 0; q < READS; ++q) {
            if (q == 0) fa[other][0].u = *(const u32x4_t*)pa;
            else if (q <= NT) fb[other][q - 1].u = *(const u32x4_t*)(pb + ((q - 1) / 2) * 4096 + ((q - 1) & 1) * 512);
            else fa[other][q - NT].u = *(const u32x4_t*)(pa + (q - NT) * 2048);
            if constexpr (decltype(LOADS)::value) {
#pragma unroll
                for (int i = q * NL / READS; i < (q + 1) * NL / READS; ++i) issue_one(dst, i);
            }
#pragma unroll
            for (int i = q * PRODUCTS / READS; i < (q + 1) * PRODUCTS / READS; ++i) multiply(half, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    gt_wait_loads<(ST - 1) * NL>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");                                  // (the barrier alone holds no read back from before it)
    int buf = 0;
    while (true) {
        // the first half's operands of a tile: read here, not behind the tile before, whose epilogue needs the registers
        fa[0][0].u = *(const u32x4_t*)(gt_smem + buf * STAGE + offA);
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[0][j].u = *(const u32x4_t*)(gt_smem + buf * STAGE + offB + (j / 2) * 4096 + (j & 1) * 512);
#pragma unroll
        for (int i = 1; i < MT; ++i) fa[0][i].u = *(const u32x4_t*)(gt_smem + buf * STAGE + offA + i * 2048);
        const int k0 = at_.sp * per;
        const int steps = ksteps - k0 < per ? ksteps - k0 : per;
        // what the epilogue's addresses hang on: asked for now where there are registers for it, so that the end of the tile waits
        // for one trip and not for two
        int pos[EPI == GT_QKV ? MT : 1], slot[EPI == GT_QKV ? MT : 1];
        auto read_places = [&]() {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int m = at_.m0 + (wm * MT + i) * 16 + r;
                pos[i] = a.positions[m < a.M ? m : a.M - 1];
                slot[i] = a.slots ? a.slots[m < a.M ? m : a.M - 1] : -1;
            }
        };
        constexpr int UNITS = NT / 4;
        constexpr bool BIAS_EARLY = EPI == GT_QKV && MT <= 5 && UNITS == 1;
        u32x4_t bias0[UNITS], bias1[UNITS], bias2[UNITS], bias3[UNITS];     // eight and eight values: 32-bit, or bfloat16 in bias0 and bias2
        auto read_bias = [&](int un) {
            const int u = at_.tn * (BN / 64) + wn * UNITS + un, head = unit_head(u, a.head_inverse);
            const int c = head * a.D + 32 * (u - head * (a.D / 64)) + 8 * g, at = c + a.D / 2 < a.N ? c : 0;
            const size_t size = a.bias_f32 ? 4 : 2;
            const unsigned char *lo = (const unsigned char*)a.bias + at * size, *hi = lo + a.D / 2 * size;
            bias0[un] = bias1[un] = bias2[un] = bias3[un] = u32x4_t{0, 0, 0, 0};
            if (a.bias) {
                bias0[un] = *(const u32x4_t*)lo;
                bias2[un] = *(const u32x4_t*)hi;
                if (a.bias_f32) {
                    bias1[un] = *(const u32x4_t*)(lo + 16);
                    bias3[un] = *(const u32x4_t*)(hi + 16);
                }
            }
        };
        if constexpr (EPI == GT_QKV && MT <= 5) read_places();
        // (marks of the clock inside the kernel: the bias, asked for at the end and cold, took 1,800 to 2,800 of a tile's 15,000 to 33,000 cycles in
        // front of the rotary rows' trip. With it here and a unit's head found without a division, 896 -> 1,152 at 77 / 544 / 2,048
        // rows 8.3 / 8.8 / 16.5 to 7.8 / 8.2 / 14.6 us)
        if constexpr (BIAS_EARLY) read_bias(0);
        int block = 0;
        // the loads are ST steps ahead: those of the last ST steps are the next tile's
        auto step = [&](auto LOADS, int left) {                     // left (without loads): this tile's steps from here on
            half_step(std::integral_constant<int, 0>{}, buf, std::false_type{}, 0u);
            // the next step's rows have arrived (this wavefront's, then everybody's), and this step's have been read
            if constexpr (decltype(LOADS)::value) gt_wait_loads<(ST - 2) * NL>();
            else gt_wait_steps<ST - 2, NL>(left - 2);
            __builtin_amdgcn_s_barrier();
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + wave * 1024);
            buf = buf + 1 == ST ? 0 : buf + 1;
            asm volatile("" ::: "memory");
            half_step(std::integral_constant<int, 1>{}, buf, LOADS, dst);
            if constexpr (decltype(LOADS)::value) issued();
            if constexpr (ES == 4) {
                if (++block == joins) {
                    block = 0;
                    join();
                }
            }
        };
#pragma unroll 1
        for (int part = 0; part < 2; ++part) {
            if (part) {
                next_load_tile();
                if (QUIET && !l_more) break;
            }
#pragma unroll 1
            for (int s = part ? ST : steps - ST; s > 0; --s) step(std::true_type{}, 0);
        }
        if constexpr (QUIET) {
            if (!l_more) {
#pragma unroll 1
                for (int s = ST; s > 0; --s) step(std::false_type{}, s);
            }
        }
        // --- the tile's results ---
        join();
        if constexpr (EPI == GT_QKV && MT > 5) read_places();
#pragma unroll
        for (int un = 0; un < NT / 4; ++un) {
            const int u = at_.tn * (BN / 64) + wn * (NT / 4) + un;      // the unit
            // a lane's columns: eight from c0 on and eight from c1 on (indices into the matrix's rows)
            int c0, c1, head = 0, d0 = 0;
            bool ok0, ok1;
            if (GATED) {
                c0 = 32 * u + 8 * g;
                c1 = a.I + c0;
                ok0 = ok1 = c0 < a.I;
            } else if (EPI == GT_QKV) {
                const int per_head = a.D / 64;
                head = unit_head(u, a.head_inverse);
                d0 = 32 * (u - head * per_head) + 8 * g;
                c0 = head * a.D + d0;
                c1 = c0 + a.D / 2;
                ok0 = ok1 = c1 < a.N;
            } else {
                c0 = 64 * u + 8 * g;
                c1 = c0 + 32;
                ok0 = c0 < a.N;
                ok1 = c1 < a.N;
            }
            // q|k|v: the bias and (a few rows at a time) the rows' cosines and sines, all asked for before the first is used
            constexpr int AHEAD = EPI != GT_QKV ? 1 : MT <= 5 ? MT : 4;
            f32x4_t bias[4], cs[AHEAD][2], sn[AHEAD][2];
            if constexpr (EPI == GT_QKV) {
                if constexpr (!BIAS_EARLY) read_bias(un);
                auto widen = [](uint32_t lo, uint32_t hi) {
                    return f32x4_t{__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u), __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)};
                };
                const u32x4_t lo = bias0[un], hi = bias2[un];
                bias[0] = a.bias_f32 ? as_f32x4(lo) : widen(lo[0], lo[1]);
                bias[1] = a.bias_f32 ? as_f32x4(bias1[un]) : widen(lo[2], lo[3]);
                bias[2] = a.bias_f32 ? as_f32x4(hi) : widen(hi[0], hi[1]);
                bias[3] = a.bias_f32 ? as_f32x4(bias3[un]) : widen(hi[2], hi[3]);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (EPI == GT_QKV) {
                    if (i % AHEAD == 0 && head < a.H + a.KVH) {
#pragma unroll
                        for (int k = 0; k < AHEAD && i + k < MT; ++k) {
                            const size_t at = (size_t)pos[i + k] * (a.D / 2) + d0;
#pragma unroll
                            for (int e = 0; e < 2; ++e) {
                                cs[k][e] = *(const f32x4_t*)(a.cos_t + at + 4 * e);
                                sn[k][e] = *(const f32x4_t*)(a.sin_t + at + 4 * e);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                const int m = at_.m0 + (wm * MT + i) * 16 + r;
                float x[8], y[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int at = 4 * un;
                    x[e] = ES == 4 ? total[ES == 4 ? i : 0][ES == 4 ? at : 0][e] : acc[i][at][e];
                    x[4 + e] = ES == 4 ? total[ES == 4 ? i : 0][ES == 4 ? at + 1 : 0][e] : acc[i][at + 1][e];
                    y[e] = ES == 4 ? total[ES == 4 ? i : 0][ES == 4 ? at + 2 : 0][e] : acc[i][at + 2][e];
                    y[4 + e] = ES == 4 ? total[ES == 4 ? i : 0][ES == 4 ? at + 3 : 0][e] : acc[i][at + 3][e];
                }
                if (m >= at_.end) continue;
                if (EPI == GT_PARTS || EPI == GT_EXPERT_DOWN) {
                    float* dst = (float*)a.C + ((size_t)(GROUPED ? 0 : at_.sp) * a.M + m) * a.N;
                    if (ok0) {
                        *(f32x4_t*)(dst + c0) = f32x4_t{x[0], x[1], x[2], x[3]};
                        *(f32x4_t*)(dst + c0 + 4) = f32x4_t{x[4], x[5], x[6], x[7]};
                    }
                    if (ok1) {
                        *(f32x4_t*)(dst + c1) = f32x4_t{y[0], y[1], y[2], y[3]};
                        *(f32x4_t*)(dst + c1 + 4) = f32x4_t{y[4], y[5], y[6], y[7]};
                    }
                } else if (EPI == GT_STORE) {
                    T* dst = (T*)a.C + (size_t)m * a.ldc;
                    if (ok0) gt_store8(dst + c0, x);
                    if (ok1) gt_store8(dst + c1, y);
                } else if (EPI == GT_EXPERT_RELU2) {
                    T* dst = (T*)a.C + (size_t)m * a.ldc;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        x[e] = fmaxf(x[e], 0.f) * fmaxf(x[e], 0.f);
                        y[e] = fmaxf(y[e], 0.f) * fmaxf(y[e], 0.f);
                    }
                    if (ok0) gt_store8(dst + c0, x);
                    if (ok1) gt_store8(dst + c1, y);
                } else if (EPI == GT_EXPERT_SILU || EPI == GT_EXPERT_CLAMPED) {
                    if (!ok0) continue;
                    float v[8];
                    const float w = EPI == GT_EXPERT_CLAMPED && a.pair_weight ? a.pair_weight[a.row_src[m]] : 1.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[e] = EPI == GT_EXPERT_CLAMPED ? clamped_glu_f32(w * x[e], w * y[e], a.alpha, a.limit)
                                                        : x[e] / (1.0f + __expf(-x[e])) * y[e];
                    gt_store8((T*)a.C + (size_t)m * a.ldc + c0, v);
                } else if (EPI == GT_SILU) {
                    if (!ok0) continue;
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        gt_round2<T>(x[e], x[e + 1]);
                        gt_round2<T>(y[e], y[e + 1]);
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = gt_silu<T>(x[e]) * y[e];
                    gt_store8((T*)a.C + (size_t)m * a.ldc + c0, v);
                } else {
                    if (!ok0) continue;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        x[e] += bias[e / 4][e % 4];
                        y[e] += bias[2 + e / 4][e % 4];
                    }
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        gt_round2<T>(x[e], x[e + 1]);
                        gt_round2<T>(y[e], y[e + 1]);
                    }
                    const int row_slot = slot[EPI == GT_QKV ? i : 0];
                    if (head < a.H + a.KVH) {
                        float y1[8], y2[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) rotate_pair(x[e], y[e], cs[i % AHEAD][e / 4][e % 4], sn[i % AHEAD][e / 4][e % 4], y1[e], y2[e]);
                        T* dst = nullptr;
                        if (head < a.H) dst = (T*)a.C + (size_t)m * a.ldc + head * a.D + d0;
                        else if (row_slot >= 0) dst = (T*)a.k_pool + ((size_t)row_slot * a.KVH + (head - a.H)) * a.D + d0;
                        if (dst) {
                            gt_store8(dst, y1);
                            gt_store8(dst + a.D / 2, y2);
                        }
                    } else if (row_slot >= 0) {
                        const int vh = head - a.H - a.KVH;
                        const int pg = row_slot >> a.page_shift, in_page = row_slot & ((1 << a.page_shift) - 1);
                        T* dst = (T*)a.v_pool + ((((size_t)pg * a.KVH + vh) * a.D + d0) << a.page_shift) + in_page;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            Elem<T>::store(dst + ((size_t)e << a.page_shift), x[e]);
                            Elem<T>::store(dst + ((size_t)(a.D / 2 + e) << a.page_shift), y[e]);
                        }
                    }
                }
            }
        }
        p += stride;
        if (!gt_next<GROUPED>(a, BM, stride, p, at_)) break;
        clear();
    }
    gt_wait_loads<0>();                                             // nothing of the ring is in flight when the block ends
}

// --- which tile, how many parts of K ---------------------------------------------------------------------------------------

// The tiles there are: 16-row tiles a wavefront (of A, of the matrix), wavefronts (down, across), buffers, blocks a CU; then the
// microseconds a 64-wide step and an epilogue of one block take when a CU has one, and of two when it has two. A large tile
// moves the fewest bytes per product, small ones are for launches that would leave CUs idle, the one with eight buffers for
// matrices that come from HBM under few rows (q|k|v of the 0.5B shape at 77 rows, in a step: 12.6 us with four, 8.9 with
// eight). Fitted to 1,900 timings on an MI355X with cold matrices (the 0.5B and 7B shapes' four matrices, 70 to 6,500 rows, K in
// one to eight parts): the shape these figures choose takes 3% longer than the best one on average. Large tiles stand at this
// card's limit (products of 16,384^3 reach 1.55 PFLOP/s; 224 x 256 tiles 1.6 once the ring runs), small ones at the latency
// of a step.
#define GT_SHAPES(X)                                       \
    X(0, 8, 8, 2, 2, 2, 1, 1.206, 10.0, 0, 0)              \
    X(1, 7, 8, 2, 2, 2, 1, 1.133, 8.79, 0, 0)              \
    X(2, 6, 8, 2, 2, 2, 1, 1.096, 7.59, 0, 0)              \
    X(3, 5, 8, 2, 2, 3, 1, 0.784, 7.50, 0, 0)              \
    X(4, 4, 8, 2, 2, 3, 1, 0.755, 6.15, 0, 0)              \
    X(5, 3, 8, 2, 2, 3, 1, 0.685, 4.61, 0, 0)              \
    X(6, 4, 4, 2, 2, 4, 1, 0.483, 3.58, 0, 0)              \
    X(7, 2, 4, 2, 2, 3, 2, 0.400, 1.48, 0.581, 3.28)       \
    X(8, 1, 4, 4, 1, 4, 2, 0.232, 1.01, 0.342, 1.94)       \
    X(9, 1, 4, 4, 1, 8, 1, 0.213, 1.16, 0, 0)              \
    X(10, 1, 4, 2, 2, 4, 2, 0.318, 1.02, 0.273, 0.61)
// Tiles between those, 128 columns wide, for rows whose tiles of the table above are one round of the chip only with a larger one (gt_pick).
// Fitted to 149 timings of eleven matrices at 100 to 4,000 rows, one round each, against what the table's choice took there.
#define GT_BETWEEN(X)                                      \
    X(11, 3, 4, 2, 2, 5, 1, 0.422, 2.68, 0, 0)             \
    X(12, 5, 4, 2, 2, 4, 1, 0.488, 4.51, 0, 0)             \
    X(13, 6, 4, 2, 2, 3, 1, 0.533, 5.60, 0, 0)             \
    X(14, 7, 4, 2, 2, 3, 1, 0.622, 4.90, 0, 0)
struct GtShape { int BM, BN, ST, OCC; double step, epi, step2, epi2; };
#define GT_SHAPE(id, MT, NT, WM, WN, ST, OCC, s1, e1, s2, e2) {16 * MT * WM, 16 * NT * WN, ST, OCC, s1, e1, s2, e2},
static const GtShape gt_shapes[] = {GT_SHAPES(GT_SHAPE) GT_BETWEEN(GT_SHAPE)};
#define GT_COUNT(...) +1
constexpr int GT_N_SHAPES = GT_SHAPES(GT_COUNT), GT_N_ALL = sizeof(gt_shapes) / sizeof(gt_shapes[0]);
constexpr int GT_CUS = 256;
constexpr double GT_BYTES_US = 14e6;        // what the CUs take out of the second-level caches together

static long long gt_tiles(const GtShape& t, int M, int N, int splits) { return (long long)((M + t.BM - 1) / t.BM) * ((N + t.BN - 1) / t.BN) * splits; }

// Microseconds a launch takes beyond its start: rounds of blocks, or the operands' way into the CUs.
static double gt_cost(const GtShape& t, int M, int N, int K, int splits) {
    const int per = (K / 64 + splits - 1) / splits;
    const long long tiles = gt_tiles(t, M, N, splits);
    const bool pairs = t.OCC > 1 && tiles > GT_CUS;
    const long long slots = pairs ? 2 * GT_CUS : GT_CUS;
    const double compute = (double)((tiles + slots - 1) / slots) * (pairs ? per * t.step2 + t.epi2 : per * t.step + t.epi);
    const double bytes = (double)tiles * (t.BM + t.BN) * per * 128 / GT_BYTES_US;
    return compute > bytes ? compute : bytes;
}

// Every part of K has to fill the ring.
static bool gt_splits_ok(const GtShape& t, int K, int splits) {
    const int steps = K / 64, per = (steps + splits - 1) / splits;
    return steps - (splits - 1) * per >= t.ST;
}

static int gt_choose(int M, int N, int K, int splits, double* cost = nullptr) {
    int best = -1;
    double least = 0;
    for (int i = 0; i < GT_N_SHAPES; ++i) {
        if (!gt_splits_ok(gt_shapes[i], K, splits)) continue;
        const double c = gt_cost(gt_shapes[i], M, N, K, splits);
        if (best < 0 || c < least) best = i, least = c;
    }
    if (cost) *cost = least;
    return best;
}

// What part of the table's choice's time by these figures a tile between may take at most to be taken, 0: never. Each is what timings say: 2,200 sizes for which
// seven hundredths less were enough, at 65 to 4,096 rows, took 0.94 of their former time, but 183 of them 1.02 to 1.36. Those were
//  - 96 rows for as many rows of tiles of 128 x 128: nothing fewer is multiplied, and the shorter step is not what the operands' way allows (278 sizes, 1.01 on the mean, to
//    1.19); with more of those 0.92, but where the operands' way is most of the time 1.12 at the worst (0.58 of it at 128 x 128, or 16% cheaper, is where that ends);
//  - tiles larger than those they stand in for, which had only seemed bound by the operands' way (160 rows for 128 x 128, 10 sizes, 1.31; 96 for 64 x 64, 8 sizes, 1.05;
//    32 x 64 are, 0.85);
//  - 224 rows by less than 12% (155 sizes, 0.99, to 1.14).
// Of 2,200 drawn anew that take one now, 22 take more than 1.02 of their former time, 1.08 at the worst, 0.915 on the mean.
static double gt_between_line(int i, int table, int M, int N, int K, int splits) {
    const GtShape &t = gt_shapes[i], &of = gt_shapes[table];
    const bool wide = of.BN == 128 && of.BM == 128;
    if (i == 11) {
        if (table == 8 || (wide && (M + t.BM - 1) / t.BM == (M + of.BM - 1) / of.BM)) return 0;
        const int per = (K / 64 + splits - 1) / splits;
        const bool way = (double)gt_tiles(of, M, N, splits) * (of.BM + of.BN) * per * 128 / GT_BYTES_US >= 0.58 * (per * of.step + of.epi);
        return wide && way ? 0.84 : 0.93;
    }
    if (i == 12 && wide) return 0;
    return i == 14 ? 0.88 : 0.93;
}

// The tile a launch takes: the table's choice, which also says into how many parts K is cut, or a tile between where that is one round of the chip,
// cheaper by these figures (gt_between_line), and not bound by the operands' way into the CUs. us: gate|up of the 0.5B shape at 250 rows 128 x 128 13.4, 96 x 128 11.9,
// at 544 96 x 256 17.1, 192 x 128 15.9, at 640 128 x 256 19.3, 224 x 128 17.6; q|k|v at 2,048 13.2 / 11.3; 1,792 -> q|k|v of 4,608 at 1,024 96 x 256 30.1, 160 x 128 24.2.
// Every tile adds a row's products in one order.
static int gt_pick(int M, int N, int K, int splits) {
    double table_cost, least = 0;
    const int table = gt_choose(M, N, K, splits, &table_cost);
    if (table < 0) return table;
    int best = table;
    const int per = (K / 64 + splits - 1) / splits;
    for (int i = GT_N_SHAPES; i < GT_N_ALL; ++i) {
        const GtShape& t = gt_shapes[i];
        const long long tiles = gt_tiles(t, M, N, splits);
        const double cost = per * t.step + t.epi;
        if (tiles > GT_CUS || !gt_splits_ok(t, K, splits) || (double)tiles * (t.BM + t.BN) * per * 128 / GT_BYTES_US >= 0.92 * cost) continue;
        if (cost < gt_between_line(i, table, M, N, K, splits) * table_cost && (best == table || cost < least)) best = i, least = cost;
    }
    return best;
}

template <typename T, int EPI, int MT, int NT, int WM, int WN, int ST, int OCC>
static int gt_launch(TileArgs& a, hipStream_t stream, TmAhead* ahead = nullptr) {
    constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN, LDS = (BM + BN) * 128 * ST;
    static_assert(LDS * OCC <= 160 * 1024, "");
    static const hipError_t allowed = hipFuncSetAttribute((const void*)gemm_tile_kernel<T, EPI, MT, NT, WM, WN, ST, OCC>,
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (allowed != hipSuccess) return TM_ERR_LAUNCH;
    // (experts: M is the most row tiles the route can give, tiles of a.tile_rows rows)
    constexpr bool GROUPED = EPI >= GT_EXPERT_SILU, GATED = EPI == GT_SILU || EPI == GT_EXPERT_SILU || EPI == GT_EXPERT_CLAMPED;
    a.tiles_m = GROUPED ? a.M * (a.tile_rows / BM) : (a.M + BM - 1) / BM;
    a.tiles_n = GATED ? (2 * ((a.I + 31) / 32 * 32) + BN - 1) / BN : (a.N + BN - 1) / BN;
    // row tiles an XCD's blocks take beside each other: all of them where K is short enough for their rows to stay in its L2
    const int most = a.K > 2048 ? 6 : 16, bands = (a.tiles_m + most - 1) / most;
    // experts: two row tiles, mostly of one expert, beside all its columns (against four: 80 to 106 us where BM is 128)
    a.band = GROUPED ? 2 : (a.tiles_m + bands - 1) / bands;
    const int chunk = (a.tiles_m * a.tiles_n * a.splits + 7) / 8;
    const int grid = 8 * chunk < GT_CUS * OCC ? 8 * chunk : GT_CUS * OCC;
    a.grid = grid;
    // (only q|k|v's small tiles leave CUs idle)
    if constexpr (EPI == GT_QKV && sizeof(T) == 2 && BM * BN <= 64 * 128) {
        if (const int more = ahead ? ahead_spare_layers(*ahead, 8, grid) : 0) {
            static const hipError_t raised = hipFuncSetAttribute((const void*)gemm_tile_kernel<T, EPI, MT, NT, WM, WN, ST, OCC, true>,
                                                                 hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
            if (raised != hipSuccess) return TM_ERR_LAUNCH;
            gemm_tile_kernel<T, EPI, MT, NT, WM, WN, ST, OCC, true><<<grid + 8 * more, 256, LDS, stream>>>(a, *ahead);
            TM_CHECK_LAUNCH();
            return TM_OK;
        }
    }
    if (ahead) ahead->n = 0;
    gemm_tile_kernel<T, EPI, MT, NT, WM, WN, ST, OCC><<<grid, 256, LDS, stream>>>(a, TmNoAhead{});
    TM_CHECK_LAUNCH();
    return TM_OK;
}

template <int EPI>
static int gt_go(TileArgs& a, int shape, hipStream_t stream, TmAhead* ahead = nullptr) {
    switch (shape) {
#define GT_CASE(id, MT, NT, WM, WN, ST, OCC, s1, e1, s2, e2) case id: return gt_launch<bf16_t, EPI, MT, NT, WM, WN, ST, OCC>(a, stream, ahead);
        GT_SHAPES(GT_CASE)
        GT_BETWEEN(GT_CASE)
    }
    return TM_ERR_ARG;
}

// Which of the tiles above a product runs with.
extern "C" int tm_gemm_tile_picked(int M, int N, int K, int splits) {
    return M > 0 && N > 0 && K >= 256 && splits > 0 ? gt_pick(M, N, K, splits) : -1;
}

// Which of the first table's: the one that says how K is cut.
extern "C" int tm_gemm_tile_shape(int M, int N, int K, int splits) {
    return M > 0 && N > 0 && K >= 256 && splits > 0 ? gt_choose(M, N, K, splits) : -1;
}

static bool gt_aligned(const void* p) { return p && ((uintptr_t)p % 16) == 0; }

// Whole 16-byte pieces everywhere, k in whole steps, rows that 32-bit offsets reach.
extern "C" int tm_gemm_tile_takes(const void* A, int lda, const void* W, int M, int N, int K) {
    return M > 0 && N > 0 && N % 8 == 0 && K >= 256 && K % 64 == 0 && lda >= K && lda % 8 == 0 && gt_aligned(A) && gt_aligned(W) &&
           (long long)M * lda * 2 < (1ll << 32) && (long long)N * K * 2 < (1ll << 32) && (long long)M * N < (1ll << 40);
}

// act[m, i] = silu(gate) * up with gate|up = A W^T, W [2 I, K] (gate rows, then up rows)
extern "C" int tm_tile_gate_up_silu(const void* A, int lda, int M, int K, const void* W, void* act, int I, hipStream_t stream) {
    if (I <= 0 || I % 8 || !gt_aligned(act) || !tm_gemm_tile_takes(A, lda, W, M, 2 * I, K)) return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = act;
    a.M = M; a.N = 2 * I; a.K = K; a.lda = lda; a.ldc = I; a.I = I; a.splits = 1;
    return gt_go<GT_SILU>(a, gt_pick(M, 2 * I, K, 1), stream);
}

// q (rotated, [M, H D]), and k and v to the cache, of q|k|v = A W^T + bias; head sizes of whole units (64), rotated over the
// whole head; slots (null: nothing is stored) as in tm_rope_kv_write
int tile_qkv_rope_ahead(const void* A, int lda, int M, int K, const void* W, const void* bias, int bias_dtype, void* q, int H,
                                int KVH, int D, const float* cos_t, const float* sin_t, const int* positions, const int* slots,
                                void* k_pool, void* v_pool, int page, TmAhead& ahead, hipStream_t stream) {
    const int N = (H + 2 * KVH) * D;
    if (H <= 0 || KVH <= 0 || D <= 0 || D % 64 || !gt_aligned(q) || !cos_t || !sin_t || !positions || page <= 0 || (page & (page - 1)) ||
        (bias && bias_dtype != TM_NONE && !gt_aligned(bias)) || !gt_aligned(cos_t) || !gt_aligned(sin_t) || (slots && (!gt_aligned(k_pool) || !v_pool)) || !tm_gemm_tile_takes(A, lda, W, M, N, K))
        return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = q;
    a.bias = bias_dtype == TM_NONE ? nullptr : bias; a.bias_f32 = bias_dtype == TM_F32;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = H * D; a.splits = 1;
    a.H = H; a.KVH = KVH; a.D = D; a.head_inverse = unit_inverse(D / 64); a.cos_t = cos_t; a.sin_t = sin_t; a.positions = positions; a.slots = slots;
    a.k_pool = k_pool; a.v_pool = v_pool;
    while ((1 << a.page_shift) < page) ++a.page_shift;
    return gt_go<GT_QKV>(a, gt_pick(M, N, K, 1), stream, &ahead);
}

extern "C" int tm_tile_qkv_rope(const void* A, int lda, int M, int K, const void* W, const void* bias, int bias_dtype, void* q, int H,
                                int KVH, int D, const float* cos_t, const float* sin_t, const int* positions, const int* slots,
                                void* k_pool, void* v_pool, int page, hipStream_t stream) {
    TmAhead none;
    return tile_qkv_rope_ahead(A, lda, M, K, W, bias, bias_dtype, q, H, KVH, D, cos_t, sin_t, positions, slots, k_pool, v_pool, page, none, stream);
}

// Parts that a plain product's K is split into, whose 32-bit sums the next norm adds; 0: the library's product is the better one.
// Few tiles leave CUs idle for the library and for one part alike; a part costs a write and a read of its sums.
// Up to 64 rows there is one row of tiles: 64 columns wide, with a ring of five buffers, two blocks a CU, and as many parts as
// give each CU a block, each at least as deep as the ring. Of the tiles above and 1 to 8 parts, 8 to 64 rows, this was the best
// or within 4% of it at ten matrices from 896 x 896 to 5,120 x 27,648, but for long K with columns enough for 128 wide tiles to
// give three CUs in four a block: those take 64 x 128 tiles, in as many parts (with the norm, 5 / 17 / 32 / 48 / 64 rows, us:
// 18,944 -> 3,584 64 wide in four parts 29.1 / 29.5 / 30.5 / 32.3 / 34.6, 128 wide in eight 29.4 / 29.8 / 30.3 / 31.2 / 32.1;
// 27,648 -> 5,120, which choose.h streams in such steps, in three and six 53.6 / 54.0 / 55.2 / 59.2 / 63.1 and 54.0 / 54.5 / 55.8 / 56.8 /
// 58.3; 13,952 -> 2,048, which
// 128 wide tiles would leave half the CUs without, stays at eight parts of 64, 15.8 to 18.3).
// How K is cut hangs on N and K alone: a row's result does not change with the number of rows.
constexpr int GT_FEW_ROWS = 64, GT_FEW_RING = 5, GT_FEW_WIDE_RING = 3;
static bool gt_few(int M, int K) { return M <= GT_FEW_ROWS && K >= 64 * GT_FEW_RING; }
static bool gt_few_wide(int N, int K) { return K / 64 > 200 && (N + 127) / 128 * 8 >= GT_CUS * 3 / 4; }
static int gt_few_parts(int N, int K) {
    const int columns = gt_few_wide(N, K) ? 128 : 64, ring = gt_few_wide(N, K) ? GT_FEW_WIDE_RING : GT_FEW_RING;
    int parts = GT_CUS / ((N + columns - 1) / columns);
    parts = parts < 1 ? 1 : parts > 8 ? 8 : parts;
    while (parts > 1 && K / 64 - (parts - 1) * ((K / 64 + parts - 1) / parts) < ring) --parts;
    return parts;
}

extern "C" int tm_tile_linear_parts(int M, int N, int K) {
    if (M <= 0 || N <= 0 || N % 8 || K < 256 || K % 64) return 0;
    if (gt_few(M, K)) return (N + 63) / 64 <= 2 * GT_CUS ? gt_few_parts(N, K) : 0;
    if ((long long)((M + 127) / 128) * ((N + 127) / 128) > GT_CUS) return 0;
    int best = 0;
    double least = 0;
    for (int splits = 1; splits <= 8; ++splits) {
        double c;
        if (gt_choose(M, N, K, splits, &c) < 0) continue;
        c += (double)splits * M * N * 4 / 5e6;                      // the norm reads them
        if (!best || c < least) best = splits, least = c;
    }
    return best;
}

// parts[p][m][n], p < tm_tile_linear_parts(M, N, K): the partial sums of A W^T
extern "C" int tm_tile_linear_split(const void* A, int lda, int M, int K, const void* W, int N, float* parts, hipStream_t stream) {
    const int splits = tm_tile_linear_parts(M, N, K);
    if (splits < 1 || !gt_aligned(parts) || !tm_gemm_tile_takes(A, lda, W, M, N, K)) return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = parts;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = N; a.splits = splits;
    if (gt_few(M, K))
        return gt_few_wide(N, K) ? gt_launch<bf16_t, GT_PARTS, 2, 4, 2, 2, GT_FEW_WIDE_RING, 2>(a, stream)
                                 : gt_launch<bf16_t, GT_PARTS, 1, 4, 4, 1, GT_FEW_RING, 2>(a, stream);
    return gt_go<GT_PARTS>(a, gt_pick(M, N, K, splits), stream);
}

TmTilePieces tile_pieces_gate_up(int M, int I, int K) {
    const int shape = gt_pick(M, 2 * I, K, 1);
    return shape < 0 ? TmTilePieces{} : TmTilePieces{gt_shapes[shape].BN / 2, 1, K / 64};
}
TmTilePieces tile_pieces_qkv(int M, int N, int K) {
    const int shape = gt_pick(M, N, K, 1);
    return shape < 0 ? TmTilePieces{} : TmTilePieces{gt_shapes[shape].BN, 1, K / 64};
}
TmTilePieces tile_pieces_split(int M, int N, int K) {
    const int parts = tm_tile_linear_parts(M, N, K);
    if (parts < 1) return {};
    const int shape = gt_few(M, K) ? 0 : gt_pick(M, N, K, parts);
    if (shape < 0) return {};
    const int columns = gt_few(M, K) ? (gt_few_wide(N, K) ? 128 : 64) : gt_shapes[shape].BN;
    return {columns, parts, (K / 64 + parts - 1) / parts};
}

// C[m, n] = A W^T, rows ldc apart, in bfloat16 (out_dtype 1) or, with ldc = N, float32 (0)
extern "C" int tm_tile_linear(const void* A, int lda, int M, int K, const void* W, int N, void* C, int ldc, int out_dtype, hipStream_t stream) {
    if (!gt_aligned(C) || ldc < N || ldc % 8 || (out_dtype != TM_BF16 && out_dtype != TM_F32) || (out_dtype == TM_F32 && ldc != N) ||
        !tm_gemm_tile_takes(A, lda, W, M, N, K))
        return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = C;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.splits = 1;
    return out_dtype == TM_F32 ? gt_go<GT_PARTS>(a, gt_pick(M, N, K, 1), stream) : gt_go<GT_STORE>(a, gt_pick(M, N, K, 1), stream);
}

// --- the same in 32-bit ---------------------------------------------------------------------------------------------------
//
// The 32-bit matrix unit takes sixteen times as long over a product, so a step of a tile of 64 x 64 (1,024 cycles of it) hides
// every load and read, and small tiles leave the fewest CUs idle in a last round: three blocks a CU, one shape (gate|up of 1,000 /
// 4,096 rows 154 / 537 us; two blocks a CU 159 / 566, 128 x 64 160 / 523, 64 x 128 160 / 524, 128 x 128 189 / 562; 111 / 455 at the
// unit's peak). Against the kernel of gemm_f32_mfma.hip (16 k at a time through registers), 0.5B shape, 1,000 rows, in us a layer:
// gate|up with SiLU*up 192 to 143, q|k|v with rotation 50 to 33, o and down 197 to 89.

#define GT_F32 float, EPI, 1, 4, 4, 1, 3, 3
constexpr int GT_F32_TILE = 64, GT_F32_STEP = 32, GT_F32_RING = 3;

template <int EPI>
static int gt_go_f32(TileArgs& a, hipStream_t stream) {
    return gt_launch<GT_F32>(a, stream);
}

extern "C" int tm_tile_f32_takes(const void* A, int lda, const void* W, int M, int N, int K) {
    return M > 0 && N > 0 && N % 8 == 0 && K >= GT_F32_STEP * GT_F32_RING && K % GT_F32_STEP == 0 && lda >= K && lda % 4 == 0 && gt_aligned(A) &&
           gt_aligned(W) && (long long)M * lda * 4 < (1ll << 32) && (long long)N * K * 4 < (1ll << 32);
}

extern "C" int tm_tile_f32_gate_up_silu(const void* A, int lda, int M, int K, const void* W, void* act, int I, hipStream_t stream) {
    if (I <= 0 || I % 8 || !gt_aligned(act) || !tm_tile_f32_takes(A, lda, W, M, 2 * I, K)) return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = act;
    a.M = M; a.N = 2 * I; a.K = K; a.lda = lda; a.ldc = I; a.I = I; a.splits = 1;
    return gt_go_f32<GT_SILU>(a, stream);
}

extern "C" int tm_tile_f32_qkv_rope(const void* A, int lda, int M, int K, const void* W, const void* bias, void* q, int H, int KVH, int D,
                                    const float* cos_t, const float* sin_t, const int* positions, const int* slots, void* k_pool,
                                    void* v_pool, int page, hipStream_t stream) {
    const int N = (H + 2 * KVH) * D;
    if (H <= 0 || KVH <= 0 || D <= 0 || D % 64 || !gt_aligned(q) || (bias && !gt_aligned(bias)) || !gt_aligned(cos_t) || !gt_aligned(sin_t) || !positions ||
        page <= 0 || (page & (page - 1)) || (slots && (!gt_aligned(k_pool) || !v_pool)) || !tm_tile_f32_takes(A, lda, W, M, N, K))
        return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = q; a.bias = bias; a.bias_f32 = 1;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = H * D; a.splits = 1;
    a.H = H; a.KVH = KVH; a.D = D; a.head_inverse = unit_inverse(D / 64); a.cos_t = cos_t; a.sin_t = sin_t; a.positions = positions; a.slots = slots; a.k_pool = k_pool; a.v_pool = v_pool;
    while ((1 << a.page_shift) < page) ++a.page_shift;
    return gt_go_f32<GT_QKV>(a, stream);
}

// Parts of K for a product whose sums the next norm adds: as many as give each CU a block of one row of tiles, eight at most, seven
// steps at least to a part; from N and K alone, so that a row's result does not change with the number of rows (the sums of a
// part and the norm's addition of the parts are in a fixed order). Few rows want many parts and many rows few, whose sums the
// norm reads; with the norm, 17 / 100 / 300 / 1,000 / 4,096 rows, us: 4,864 -> 896 in one part 85 / 86 / 87 / 89 / 298, in
// eight 16 / 19 / 39 / 76 / 290; 896 -> 896 in one 21 / 22 / 22 / 25 / 68, four 10 / 11 / 17 / 28 / 72, seven 9 / 10 / 15 / 31 /
// 84; 2,048 -> 2,048 in one 40 / 40 / 43 / 74 / 268, eight 11 / 18 / 34 / 87 / 353; 3,584 -> 3,584 in one 65 / 66 / 119 / 224 /
// 791, four 23 / 37 / 79 / 210 / 842. (The rows decide only whether there is a product.)
extern "C" int tm_tile_f32_parts(int M, int N, int K) {
    if (M <= 0 || N <= 0 || N % 8 || K < GT_F32_STEP * GT_F32_RING || K % GT_F32_STEP) return 0;
    const int steps = K / GT_F32_STEP;
    int parts = GT_CUS / ((N + GT_F32_TILE - 1) / GT_F32_TILE);
    parts = parts < steps / 7 ? parts : steps / 7;
    parts = parts < 1 ? 1 : parts > 8 ? 8 : parts;
    while (parts > 1 && steps - (parts - 1) * ((steps + parts - 1) / parts) < GT_F32_RING) --parts;
    return parts;
}

// parts[p][m][n], p < splits: the partial sums of A W^T (splits 1: the product itself)
extern "C" int tm_tile_f32_linear_split(const void* A, int lda, int M, int K, const void* W, int N, float* parts, int splits, hipStream_t stream) {
    if (splits < 1 || !gt_aligned(parts) || !tm_tile_f32_takes(A, lda, W, M, N, K)) return TM_ERR_ARG;
    const int steps = K / GT_F32_STEP, per = (steps + splits - 1) / splits;
    if (steps - (splits - 1) * per < GT_F32_RING) return TM_ERR_ARG;
    TileArgs a{};
    a.A = A; a.W = W; a.C = parts;
    a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = N; a.splits = splits;
    return gt_go_f32<GT_PARTS>(a, stream);
}

// --- the products of experts -----------------------------------------------------------------------------------------------
//
// A tile of the route (128 slots, or 64) by 256 matrix rows: these products stand at what the CUs take out of the second-level
// caches, so the larger tile wins although an expert's last one is seldom full (16 experts of 187 slots on average: 3 tiles of 64
// or 2 of 128 slots). Against grouped_mfma.hip (128 slots by 64 or 128 rows, 32 k a step through registers and padded LDS rows),
// 3,000 pairs of 16 experts of 2,048 x 2,048, gate|up with silu and down, in us: 144 + 84 to 80 + 45; 64 x 256 123 + 62, 64 x 128
// 117 + 67, 128 x 128 99 + 50. The matrices alone take 54 + 27 to read.

template <int EPI>
static int gt_expert(const void* A, int lda, const int* row_src, int src_div, const void* W, void* C, int ldc, const int* tiles, const int* n_tiles,
                     int max_tiles, int tile_rows, int K, int N, int I, const float* pair_weight, float limit, float alpha, hipStream_t stream) {
    TileArgs a{};
    a.A = A; a.W = W; a.C = C; a.M = max_tiles; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.splits = 1; a.I = I;
    a.tiles = tiles; a.n_tiles = n_tiles; a.row_src = row_src; a.src_div = src_div; a.tile_rows = tile_rows;
    a.pair_weight = pair_weight; a.limit = limit; a.alpha = alpha;
    return tile_rows % 128 == 0 ? gt_launch<bf16_t, EPI, 4, 8, 2, 2, 3, 1>(a, stream) : gt_launch<bf16_t, EPI, 2, 8, 2, 2, 3, 1>(a, stream);
}

// Whole 16-byte pieces, k in whole steps that fill the ring, tiles of whole 64 rows; `rows`: the most rows of A there are.
extern "C" int tm_tile_experts_takes(const void* A, int lda, long long rows, const void* W, const void* C, int tile_rows, int K, int N) {
    return tile_rows % 64 == 0 && tile_rows > 0 && K >= 192 && K % 64 == 0 && N % 16 == 0 && lda % 8 == 0 && gt_aligned(A) && gt_aligned(W) &&
           gt_aligned(C) && rows * lda * 2 < (1ll << 32) && (long long)N * K * 2 < (1ll << 32);
}

// The products of tm_moe_gate_up_mfma (kind 0), tm_moe_clamped_mfma (1), tm_moe_up_act_mfma (2: N rows an expert) and
// tm_moe_down_mfma (3); their operands, checked by them.
extern "C" int tm_tile_experts(int kind, const void* A, int lda, const int* row_src, int src_div, const void* W, void* C, const int* tiles,
                               const int* n_tiles, int max_tiles, int tile_rows, int K, int F, const float* pair_weight, float limit, float alpha,
                               hipStream_t stream) {
#define GT_EXPERT_GO(EPI, N, I) gt_expert<EPI>(A, lda, row_src, src_div, W, C, F, tiles, n_tiles, max_tiles, tile_rows, K, N, I, pair_weight, limit, alpha, stream)
    switch (kind) {
        case 0: return GT_EXPERT_GO(GT_EXPERT_SILU, 2 * F, F);
        case 1: return GT_EXPERT_GO(GT_EXPERT_CLAMPED, 2 * F, F);
        case 2: return GT_EXPERT_GO(GT_EXPERT_RELU2, F, 0);
        case 3: return GT_EXPERT_GO(GT_EXPERT_DOWN, F, 0);
    }
#undef GT_EXPERT_GO
    return TM_ERR_ARG;
}
