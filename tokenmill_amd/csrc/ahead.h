// The matrices of the products that follow, brought into the second-level caches by blocks beside those of a kernel that leaves most of the
// chip idle.
//
// In steps of few tokens a layer of a small model is five or six launches of a few microseconds, and a product's launch waits for its matrix
// from HBM before it does anything (0.5B shape, 1 and 8 tokens, the same matrix again, out of the caches, against a cold one: gate|up 6.1 / 6.3 to
// 4.0 / 4.4 us, down 4.2 / 6.2 to 3.0 / 5.0, q|k|v 4.4 to 3.9, o 2.7 / 3.2 to 2.5 / 2.9; out of the memory-side cache alone gate|up 5.3 / 5.7),
// while HBM idles during the attention and the norms. Their order is known, so blocks behind a kernel's own read a word of every line
// of what the next ones need. The eight compute dies have a second-level cache each, of 4 MB, and take a launch's blocks in turn, so a block
// brings what the blocks of the product with the same index modulo eight read. If they did not, the matrix would come from the
// memory-side cache: nothing depends on it but time.
//
// Which kernel brings what stands in step_program.hip (Run::ahead).
#pragma once
#include "common.h"

#include <type_traits>

constexpr int TM_AHEAD_MATRICES = 4, TM_AHEAD_LINE = 128;

// 2^31 / d rounded up, and x / d by it (for x (d - 1) + d below 2^31)
__host__ __device__ __forceinline__ uint32_t ahead_inverse(int d) { return (uint32_t)(((1ull << 31) + d - 1) / d); }
__host__ __device__ __forceinline__ int ahead_over(int x, uint32_t inverse) { return (int)(((uint64_t)(uint32_t)(2 * x + 1) * inverse) >> 32); }

// What the blocks of a product read, a piece at a time. A packed matrix: a piece is a strip, strips lie one after the other; block b has the units
// b, b + blocks, ... or, with `together`, the units b together, b together + 1, ...; a unit is one strip, or strip u and strip units + u (gate
// and up), or, of q|k|v, a strip of each half of a head (q and k) or two neighbours (v). A row-major matrix: a piece is the rows of a column tile of the
// product and their bytes of a part of K; pieces in the order of the tiled product's blocks, of which a die has a run.
struct alignas(64) TmAheadMatrix {
    const unsigned char* base;                  // (matrices of less than 2 GB)
    int end;                                    // runs (64 lines of a piece) of a die up to and with this matrix's
    int runs;                                   // in a piece
    uint32_t runs_inverse;
    short two, row_major;                       // pieces of a unit are two
    union {
        struct {
            int cols, first, strip_bytes, units, blocks, together;      // units of a round a die has at most, the first round
            int head_units, rot_heads;          // units of a head (0: not q|k|v), heads of q and k
            uint32_t cols_inverse, head_inverse;
        } packed;
        struct {
            int columns, tiles, rows, lines, all_lines, second, row_end;        // pieces, column tiles, rows and lines a row of a piece, lines of a row,
            uint32_t tiles_inverse, lines_inverse;                              // first row of the second half (up), rows of a half
        } rows;
    };
};
static_assert(sizeof(TmAheadMatrix) == 64, "one load of sixteen words");

struct TmAhead {
    TmAheadMatrix m[TM_AHEAD_MATRICES];
    int n = 0;                                  // 0: nothing is brought
    int first, blocks;                          // linear indices of the blocks that bring it, behind the launch's own
    int rows = 0;                               // a matrix is row-major

    // rounds [first_round, last_round) of a packed matrix's units
    void packed(const void* base, int strip_bytes, int units, bool two, int product_blocks, bool together = false, int first_round = 0,
                int last_round = 1 << 30, int head_units = 0, int rot_heads = 0) {
        const int rounds = (units + product_blocks - 1) / product_blocks;
        last_round = last_round < rounds ? last_round : rounds;
        if (first_round >= last_round) return;
        TmAheadMatrix x{};
        x.packed = {(product_blocks + 7) / 8, first_round, strip_bytes, units, product_blocks, together ? rounds : 0, head_units, rot_heads,
                    ahead_inverse((product_blocks + 7) / 8), head_units ? ahead_inverse(head_units) : 0};
        put(x, base, (strip_bytes + TM_AHEAD_LINE - 1) / TM_AHEAD_LINE, x.packed.cols * (last_round - first_round), two);
    }
    // a row-major matrix [halves x row_end, K], halves 2 if `two`: column tiles of `tile_rows` rows of a half, K (64 a line in bfloat16) in parts of `lines` lines
    void row_major(const void* base, int row_end, int K, int tile_rows, int parts, int lines, bool two) {
        TmAheadMatrix x{};
        const int tiles = (row_end + tile_rows - 1) / tile_rows;
        x.row_major = 1;
        rows = 1;
        x.rows = {tiles * parts, tiles, tile_rows, lines, K / 64, two ? row_end : 0, row_end, ahead_inverse(tiles), ahead_inverse(lines)};
        put(x, base, tile_rows * lines, (tiles * parts + 7) / 8, two);
    }
    int total() const { return n ? m[n - 1].end : 0; }

private:
    void put(TmAheadMatrix& x, const void* base, int piece_lines, int units, bool two) {
        x.base = (const unsigned char*)base;
        x.two = two;
        x.runs = (piece_lines + TM_WAVE - 1) / TM_WAVE, x.runs_inverse = ahead_inverse(x.runs);
        x.end = total() + units * (two ? 2 : 1) * x.runs;
        m[n++] = x;
    }
};

// Line `lane` of run e of a die's runs of matrix m: its place in the matrix, or -1 where there is none. All but the last lines hangs on the run alone.
// ROWS: the matrix may be row-major.
template <bool ROWS>
__host__ __device__ __forceinline__ int ahead_line(const TmAheadMatrix& m, int die, int e, int lane) {
    int q = ahead_over(e, m.runs_inverse);
    const int run = e - q * m.runs, part = m.two ? q & 1 : 0, line = run * TM_WAVE + lane;
    q >>= m.two;
    if (ROWS && m.row_major) {
        const auto& r = m.rows;
        const int c = die * r.columns / 8 + q;
        const int k = ahead_over(c, r.tiles_inverse), row0 = (c - k * r.tiles) * r.rows;
        const int row = ahead_over(line, r.lines_inverse), at = k * r.lines + line - row * r.lines;
        if (c >= (die + 1) * r.columns / 8 || row >= r.rows || row0 + row >= r.row_end || at >= r.all_lines) return -1;
        return ((part * r.second + row0 + row) * r.all_lines + at) * TM_AHEAD_LINE;
    }
    const auto& r = m.packed;
    const int round = ahead_over(q, r.cols_inverse), b = die + 8 * (q - round * r.cols);
    const int u = r.together ? b * r.together + r.first + round : b + (r.first + round) * r.blocks;
    int strip = part * r.units + u;
    if (r.head_units) {
        const int head = ahead_over(u, r.head_inverse), jt = u - head * r.head_units;
        strip = 2 * r.head_units * head + (head < r.rot_heads ? jt + part * r.head_units : 2 * jt + part);
    }
    if (b >= r.blocks || u >= r.units || line * TM_AHEAD_LINE >= r.strip_bytes) return -1;
    return strip * r.strip_bytes + line * TM_AHEAD_LINE;
}

// In front of the branch that tells such blocks from a kernel's own: the arguments named arrive with the one it compares, by one wait. Left to
// itself the compiler asks for them behind the branch, a trip to memory later (0.3 to 0.4 us a launch).
template <typename... T>
__device__ __forceinline__ void ahead_with(const T&... args) {
    (([&](const auto& x) { asm volatile("" ::"s"(x)); })(args), ...);
}

// What tm_bring_ahead does where the matrices are all packed, or may be row-major.
template <bool ROWS>
__device__ __forceinline__ void bring_runs(const TmAhead& a, int die, int e, int all) {
    constexpr int DEEP = ROWS ? 8 : 4;
    const int lane = threadIdx.x % TM_WAVE, total = a.m[a.n - 1].end;
    while (e < total) {
        uint32_t word[DEEP];
#pragma unroll
        for (int j = 0; j < DEEP; ++j) {
            word[j] = 0;
            if (e >= total) continue;
            int i = 0;
            while (e >= a.m[i].end) ++i;
            const TmAheadMatrix m = a.m[i];      // (one use of the kernel's argument: with hundreds the compiler keeps a copy of it in scratch memory)
            const int line = ahead_line<ROWS>(m, die, e - (i ? a.m[i - 1].end : 0), lane);
            if (line >= 0) word[j] = *(const uint32_t*)(m.base + (uint32_t)line);
            e += all;
        }
#pragma unroll
        for (int j = 0; j < DEEP; ++j) asm volatile("" ::"v"(word[j]));
    }
}

// block: the linear index of a block of `waves` wavefronts in its grid. A wavefront takes every n-th run, a line a lane, four (eight) on their way at once; a word
// of each is read and nothing is done with it. What runs in front of the loads is most of such a block's life, so everything but a lane's place in a
// run is the same in every lane, there is no division, and the code is short, since it comes into a CU cold, a line at a time. A step of one request,
// us: so 622, eight loads at once 622 (of row-major matrices, where a wavefront has more, 1,802 to 1,770 beside two portions of 241 tokens), with the code for row-major matrices in the way of packed ones 636, the words to LDS in place of registers
// (a loop of few instructions) 634, four of each matrix in a row of code 661.
__device__ __forceinline__ void tm_bring_ahead(const TmAhead& a, int block, int waves) {
    // (every line of the arguments that is read here arrives by one wait)
    ahead_with(a.first, a.blocks, a.n, a.m[0].end, a.m[1].end, a.m[2].end, a.m[3].end);
    static_assert(TM_AHEAD_MATRICES == 4, "the lines named above");
    const int at = block - a.first;
    if (at >= a.blocks) return;
    const int all = (a.blocks - at % 8 + 7) / 8 * waves;             // wavefronts of this die's blocks
    const int e = at / 8 * waves + __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE);
    if (a.rows) bring_runs<true>(a, block % 8, e, all);
    else bring_runs<false>(a, block % 8, e, all);
}

// What a kernel that may carry such blocks or not has as its last argument.
struct TmNoAhead {};
template <bool AHEAD>
using TmAheadArg = std::conditional_t<AHEAD, TmAhead, TmNoAhead>;
template <bool AHEAD>
inline TmAheadArg<AHEAD> ahead_arg(const TmAhead& a) {
    if constexpr (AHEAD) return a;
    else return TmNoAhead{};
}

// Layers of `layer` blocks behind the `own` blocks of a grid whose kernel fills a CU with one: as many as find a CU and are asked for, at least
// one (of which what finds no CU returns at once); none, and nothing is brought (ahead.n = 0), where CUs are scarce.
inline int ahead_spare_layers(TmAhead& ahead, int layer, int own) {
    const int idle = 256 - own, most = ahead.blocks < idle ? ahead.blocks : idle;
    const int layers = !ahead.n || idle < 64 ? 0 : most / layer > 0 ? most / layer : 1;
    if (layers == 0) ahead.n = 0;
    ahead.first = own;
    ahead.blocks = layers * layer < idle ? layers * layer : idle;
    return layers;
}

// The kernels that have room for such blocks, as the functions of api.h without `_ahead`. Of `ahead` the caller sets the matrices and how many blocks
// there should be.
int attn_decode_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool, const int* block_tables,
                      int table_width, const int* context_lens, float* part_o, float* part_ml, int max_chunks, int S, int H, int KVH, int D, int page,
                      float scale, int window, int keep, float softcap, const float* sink, const void* cgate, int ldcg, TmAhead ahead, hipStream_t stream);
int attn_decode_whole_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool, const int* block_tables,
                            int table_width, const int* context_lens, int max_chunks, int S, int H, int KVH, int D, int page, float scale, int window,
                            int keep, float softcap, const float* sink, const void* cgate, int ldcg, TmAhead ahead, hipStream_t stream);
int fused_norm_qkv_rope_ahead(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M, int K, const void* W, const void* bias,
                              int bias_dtype, void* q_out, int H, int KVH, int D, const float* cos_t, const float* sin_t, const int* positions,
                              const int* slots, void* k_pool, void* v_pool, int page, TmAhead ahead, hipStream_t stream);
int fused_norm_gate_up_silu_ahead(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M, int K, const void* W, void* act_out,
                                  int I, TmAhead ahead, hipStream_t stream);

// ... and these, which bring what they are asked to if they have room for the blocks, and else set ahead.n to 0
int tile_qkv_rope_ahead(const void* A, int lda, int M, int K, const void* W, const void* bias, int bias_dtype, void* q, int H, int KVH, int D,
                        const float* cos_t, const float* sin_t, const int* positions, const int* slots, void* k_pool, void* v_pool, int page,
                        TmAhead& ahead, hipStream_t stream);
int attn_prefill_ahead(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool, const int* block_tables,
                       int table_width, const int* tiles, int n_tiles, int H, int KVH, int D, int page, float scale, int window, int keep, float softcap,
                       const float* sink, const void* cgate, int ldcg, TmAhead& ahead, hipStream_t stream, struct TmDecodes* beside = nullptr);

// Single decoded tokens that a launch over prompt portions attends too (choose.h: tm_prefill_takes_decodes), of the same pools, strides and options; as
// attn_decode_whole_ahead's arguments.
struct TmDecodes {
    const void* q;
    void* out;
    const int* tables;
    const int* context_lens;
    const void* cgate;
    int n, chunks;
    float cap_out;              // (attn_prefill_ahead's own)
};
bool decode_args_ok(const void* q, int q_stride, const void* out, int out_stride, int table_width, int max_chunks, int H, int KVH, int D, int page,
                    float scale, int window, int keep, float softcap, const void* cgate, int ldcg);

// What the blocks of the tiled products read of their matrix at a time (gemm_tile.hip): rows of a column tile (gate|up: of either half), and K in
// so many parts of so many steps of 64.
struct TmTilePieces {
    int rows, parts, steps;
};
TmTilePieces tile_pieces_gate_up(int M, int I, int K);
TmTilePieces tile_pieces_qkv(int M, int N, int K);
TmTilePieces tile_pieces_split(int M, int N, int K);
int stream_gate_up_units(int I);                // units a block of the streamed gate|up has (gemm_stream.hip)
