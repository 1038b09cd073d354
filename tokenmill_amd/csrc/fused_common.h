// What the decode-step products that end in a layer's own epilogue share: their arguments, the pair
// of matrix strips a block multiplies, small helpers.
#pragma once
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

union FFrag {
    u32x4_t u;
    bf16x8_t b;
};

__device__ __forceinline__ uint32_t fd_pack(float a, float b) {
    const bf16x2_t v = __builtin_convertvector(f32x2_t{a, b}, bf16x2_t);
    return *(const uint32_t*)&v;
}

__device__ __forceinline__ float fd_round(float a) { return bf16_to_f32(f32_to_bf16(a)); }

__device__ __forceinline__ f32x4_t as_f32x4(const u32x4_t u) { return __builtin_bit_cast(f32x4_t, u); }

// A buffer of `bytes` at `base` (the same in every lane): loads beyond it read as zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t fd_buffer(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// 16 bytes a lane from base + voff (bytes) to LDS at lds (bytes, wave-uniform) + 16 * lane
__device__ __forceinline__ void fd_load_lds(uint32_t lds, uint32_t voff, const void* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "m0", "memory");
}

#define FD_EPI_QKV 0
#define FD_EPI_SILU 1
#define FD_KCH 8            // k-steps of one register group of matrix loads, per wavefront (one group in all)
#define FD_KCH_PIPE 6       // the same where two groups take turns
#define FD_XPAD 16          // padding of an LDS row of x, in elements: with K a multiple of 32 the rows are 32 bytes more than a multiple of 64 apart, which the operand loads read free of bank conflicts (with 8 they take twice as long)
#define FD_RC 8             // 4-element vectors of a residual row a thread keeps in registers

// A unit's head without a division, which is some thirty instructions in a row in front of a kernel's first loads: the host's
// 2^31 / d rounded up (d: units a head has), the upper half of whose product with 2 u + 1 is u / d (for u (d - 1) + d below 2^31).
__host__ __device__ __forceinline__ uint32_t unit_inverse(int d) { return (uint32_t)(((1ull << 31) + d - 1) / d); }
__device__ __forceinline__ int unit_head(int u, uint32_t inverse) { return (int)__umulhi((uint32_t)(2 * u + 1), inverse); }

// rows of x a block keeps in LDS for M tokens
__host__ __device__ __forceinline__ int fused_rows(int M) { return M <= 4 ? 4 : (M <= 8 ? 8 : 16); }

// 4-element vectors a thread holds where one round of loads covers a row: rows of up to 1,024 in 4 or 8 rows of x
__host__ __device__ constexpr int fused_row_vectors(int threads) { return 2048 / threads; }

// Elements between the rows of x in LDS: whole k-steps (zeros beyond K) and the padding.
__host__ __device__ __forceinline__ int fused_x_stride(int K) { return (K + 31) / 32 * 32 + FD_XPAD; }

struct FusedArgs {
    // norm + product
    const float* resid;     // [M, K] (the kernel that starts at the norm)
    const bf16_t* X;        // [M, K], rows ldx apart: the normed input (the kernel that starts behind the norm)
    int ldx;
    const void* norm_w;     // [K]
    int norm_w_f32;
    float eps;
    int M, K;
    const bf16_t* W;        // the matrix in strip order (see tm_pack_layout in api.h), strips of the kernel's ROWS
    int up_strip0;          // SiLU epilogue: index of the first strip of the up rows
    const void* bias;       // [rows] or null
    int bias_f32;
    // QKV epilogue
    bf16_t* q_out;          // [M, H*D]
    int H, KVH, D;
    uint32_t head_inverse;  // unit_inverse of the units a head has
    const float* cos_t;     // [max_pos, D/2]
    const float* sin_t;
    const int* positions;   // [M]
    const int* slots;       // [M]; < 0: not stored
    bf16_t* k_pool;         // [pages, page, KVH, D]
    bf16_t* v_pool;         // [pages, KVH, D, page]
    int page_shift;
    // SiLU epilogue
    bf16_t* act_out;        // [M, I]
    int I;
};

// The two strips of ROWS matrix rows a block multiplies together ("unit" u).
struct FusedUnit {
    int nA, nB;             // first rows of the strips
    int sA, sB;             // their indices in the packed matrix
    int head, jt;           // QKV: the head and which slice of it
};

// Unit u of a product whose strips have ROWS rows.
template <int EPI, int ROWS>
__device__ __forceinline__ FusedUnit fused_unit_of(const FusedArgs& a, int u) {
    FusedUnit t;
    t.head = 0;
    t.jt = 0;
    if (EPI == FD_EPI_QKV) {
        t.head = unit_head(u, a.head_inverse);
        t.jt = u - t.head * (a.D / (2 * ROWS));
        if (t.head < a.H + a.KVH) {                                  // the two halves of ROWS rotary pairs
            t.nA = t.head * a.D + ROWS * t.jt;
            t.nB = t.nA + a.D / 2;
        } else {
            t.nA = t.head * a.D + 2 * ROWS * t.jt;
            t.nB = t.nA + ROWS;
        }
        t.sA = t.nA / ROWS;                                          // D % 32 == 0: every strip starts on a multiple of ROWS
        t.sB = t.nB / ROWS;
    } else {                                                         // gate rows and the up rows that meet them
        t.nA = ROWS * u;
        t.nB = a.I + ROWS * u;
        t.sA = u;
        t.sB = a.up_strip0 + u;                                      // (rows beyond I are zeros in the packed matrix)
    }
    return t;
}

// Blocks of the gate|up product that starts at the norm: one round, each with the same number of pairs of strips (tm_fused_norm_gate_up_silu).
inline int fused_gate_up_blocks(int I) {
    const int units = (I + 15) / 16, per_block = (units + 255) / 256;
    return (units + per_block - 1) / per_block;
}
