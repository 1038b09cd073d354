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

constexpr int TM_AHEAD_MATRICES = 2, TM_AHEAD_LINE = 128, TM_AHEAD_RUN = TM_WAVE * TM_AHEAD_LINE;

// 2^31 / d rounded up, and x / d by it (for x (d - 1) + d below 2^31)
__host__ __device__ __forceinline__ uint32_t ahead_inverse(int d) { return (uint32_t)(((1ull << 31) + d - 1) / d); }
__host__ __device__ __forceinline__ int ahead_over(int x, uint32_t inverse) { return (int)(((uint64_t)(2 * x + 1) * inverse) >> 32); }

// A packed matrix (strips one after the other) of a product whose block b takes the units b, b + blocks, ... A unit is one strip; or strip u and
// strip units + u (gate and up); or, of q|k|v, a strip of each half of a head (q and k) or two neighbours (v).
struct TmAheadMatrix {
    const unsigned char* base;
    int strip_bytes, runs;                      // a run: 64 lines
    int units, blocks, cols, first;             // cols: blocks of a die at most; first: the round of units that is the first to be brought
    int two, head_units, rot_heads;             // strips of a unit are two; units of a head (0: not q|k|v), heads of q and k
    uint32_t runs_inverse, cols_inverse, head_inverse;
    int end;                                    // runs of a die up to and with this matrix's
};

struct TmAhead {
    TmAheadMatrix m[TM_AHEAD_MATRICES];
    int n = 0;                                  // 0: nothing is brought
    int first, blocks;                          // linear indices of the blocks that bring it, behind the launch's own

    // rounds [first, last) of the units
    void add(const void* base, int strip_bytes, int units, bool two, int product_blocks, int first_round = 0, int last_round = 1 << 30,
             int head_units = 0, int rot_heads = 0) {
        const int rounds = (units + product_blocks - 1) / product_blocks;
        last_round = last_round < rounds ? last_round : rounds;
        if (first_round >= last_round) return;
        TmAheadMatrix& x = m[n];
        x.base = (const unsigned char*)base;
        x.strip_bytes = strip_bytes;
        x.runs = (strip_bytes + TM_AHEAD_RUN - 1) / TM_AHEAD_RUN;
        x.units = units, x.blocks = product_blocks, x.cols = (product_blocks + 7) / 8, x.first = first_round;
        x.two = two, x.head_units = head_units, x.rot_heads = rot_heads;
        x.runs_inverse = ahead_inverse(x.runs), x.cols_inverse = ahead_inverse(x.cols), x.head_inverse = head_units ? ahead_inverse(head_units) : 0;
        x.end = (n ? m[n - 1].end : 0) + x.cols * (last_round - first_round) * (two ? 2 : 1) * x.runs;
        ++n;
    }
    int total() const { return n ? m[n - 1].end : 0; }
};

// Run e of a die: its matrix, its strip there and its place in the strip; false where the die has no such unit.
__host__ __device__ __forceinline__ bool ahead_run(const TmAhead& a, int die, int e, int& matrix, int& strip, int& run) {
    matrix = 0;
    while (matrix + 1 < a.n && e >= a.m[matrix].end) ++matrix;
    const TmAheadMatrix& m = a.m[matrix];
    if (matrix) e -= a.m[matrix - 1].end;
    int q = ahead_over(e, m.runs_inverse);
    run = e - q * m.runs;
    const int part = m.two ? q & 1 : 0;
    q >>= m.two;
    const int round = ahead_over(q, m.cols_inverse), b = die + 8 * (q - round * m.cols), u = b + (m.first + round) * m.blocks;
    strip = part * m.units + u;
    if (m.head_units) {
        const int head = ahead_over(u, m.head_inverse), jt = u - head * m.head_units;
        strip = 2 * m.head_units * head + (head < m.rot_heads ? jt + part * m.head_units : 2 * jt + part);
    }
    return b < m.blocks && u < m.units;
}

// block: the linear index of a block of `waves` wavefronts in its grid. Eight lines a lane are on their way at once; a word of each is read and
// nothing is done with it. Everything but a lane's place in a run is the same in every lane, and there is no division: with them this took
// longer than the kernels beside it.
__device__ __forceinline__ void tm_bring_ahead(const TmAhead& a, int block, int waves) {
    const int at = block - a.first;
    const int mine = (a.blocks - at % 8 + 7) / 8;                    // blocks of this die
    const int wave = at / 8 * waves + __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), all = mine * waves;
    const int lane_at = threadIdx.x % TM_WAVE * TM_AHEAD_LINE, total = a.m[a.n - 1].end;
    for (int e0 = wave; e0 < total; e0 += 8 * all) {
        uint32_t word[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            int matrix, strip, run;
            word[j] = 0;
            if (e0 + j * all >= total || !ahead_run(a, block % 8, e0 + j * all, matrix, strip, run)) continue;
            const TmAheadMatrix& m = a.m[matrix];
            const int off = run * TM_AHEAD_RUN + lane_at;
            word[j] = *(const uint32_t*)(m.base + (size_t)strip * m.strip_bytes + (off < m.strip_bytes ? off : 0));
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" ::"v"(word[j]));
    }
}

// In front of the branch that tells such blocks from a kernel's own: the arguments named arrive with the one it compares, by one wait. Left to
// itself the compiler asks for them behind the branch, a trip to memory later (0.3 to 0.4 us a launch).
template <typename... T>
__device__ __forceinline__ void ahead_with(const T&... args) {
    (([&](const auto& x) { asm volatile("" ::"s"(x)); })(args), ...);
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
