// Shared device helpers for the gfx950 kernels: storage types, wave/block reductions, checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define TM_WAVE 64

// dtype codes of the C interface
#define TM_F32 0
#define TM_BF16 1
#define TM_NONE (-1)

// error codes of the C interface (0 = ok)
#define TM_OK 0
#define TM_ERR_ARG 1        // an argument the kernel cannot run with
#define TM_ERR_LAUNCH 2     // the runtime refused the launch
#define TM_ERR_UNSUPPORTED 3 // a library has no routine for the request: use another path

typedef uint16_t bf16_t;    // bfloat16 bits

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
    return __uint_as_float(((uint32_t)v) << 16);
}

// round to nearest even; NaN stays NaN (the conversion instruction: one in place of the seven of integer arithmetic that gave the
// same bits, which the norms and epilogues of small steps waited for one after the other)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    return __builtin_bit_cast(bf16_t, (__bf16)f);
}

template <typename T> struct Elem;
template <> struct Elem<float> {
    static __device__ __forceinline__ float load(const float* p) { return *p; }
    static __device__ __forceinline__ void store(float* p, float v) { *p = v; }
    static __device__ __forceinline__ float round(float v) { return v; }
};
template <> struct Elem<bf16_t> {
    static __device__ __forceinline__ float load(const bf16_t* p) { return bf16_to_f32(*p); }
    static __device__ __forceinline__ void store(bf16_t* p, float v) { *p = f32_to_bf16(v); }
    static __device__ __forceinline__ float round(float v) { return bf16_to_f32(f32_to_bf16(v)); }
};

// Sixteen bytes of a row as 32-bit floats: 4 float32 values or 8 bfloat16 values.
template <typename T> struct Piece;
template <> struct Piece<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ void unpack(const uint4& u, float* f) {
        f[0] = __uint_as_float(u.x); f[1] = __uint_as_float(u.y); f[2] = __uint_as_float(u.z); f[3] = __uint_as_float(u.w);
    }
};
template <> struct Piece<bf16_t> {
    static constexpr int N = 8;
    static __device__ __forceinline__ void unpack(const uint4& u, float* f) {
        f[0] = __uint_as_float(u.x << 16); f[1] = __uint_as_float(u.x & 0xffff0000u);
        f[2] = __uint_as_float(u.y << 16); f[3] = __uint_as_float(u.y & 0xffff0000u);
        f[4] = __uint_as_float(u.z << 16); f[5] = __uint_as_float(u.z & 0xffff0000u);
        f[6] = __uint_as_float(u.w << 16); f[7] = __uint_as_float(u.w & 0xffff0000u);
    }
};

// The rotation of a pair (x1, x2) by the angle whose cosine and sine are c and s (reference
// src/infer/model/layers.py:60-64). Every product and each sum is rounded to 32-bit on its own, as a tensor
// library's x1 * cos - x2 * sin is: left to itself the compiler fuses a product into the sum, and which one it
// picks differs from one kernel (or one instantiation of a kernel) to the next, so that the same token would get
// other last bits from the kernel for 8 rows than from the kernel for 40.
__device__ __forceinline__ void rotate_pair(float x1, float x2, float c, float s, float& y1, float& y2) {
#pragma clang fp contract(off)
    const float a = x1 * c, b = x2 * s, d = x2 * c, e = x1 * s;
    y1 = a - b;
    y2 = d + e;
}

// sigmoid from the hardware's exponential
__device__ __forceinline__ float sigmoid_fast(float x) { return 1.0f / (1.0f + __expf(-x)); }

// the clamped gated activation g sigmoid(alpha g) (u + 1), g = min(gate, limit), u = up held to +-limit
__device__ __forceinline__ float clamped_glu_f32(float g, float u, float alpha, float limit) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
}

// tanh from the hardware's exp2 and reciprocal: 1 - 2 / (e^(2x) + 1), exact at both ends (e^(2x) = inf or 0); its absolute
// error of about 1e-7 is far below a bfloat16 score's own
__device__ __forceinline__ float tanh_fast(float x) {
    return 1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * 2.8853900817779268f) + 1.f);
}

// Exchanges between the lanes of a wavefront by instructions of the vector unit (row permutations, swaps of rows and of halves)
// in place of __shfl_xor, which goes through LDS: a butterfly of six steps takes some 60 cycles, by LDS some 700, and in
// kernels of a few microseconds nothing else runs meanwhile. Every lane of a group that exchanges has to be active.
//
// lane_sum<OFF>(v): v + (v of lane ^ OFF); lane_max likewise. The same values meet as by __shfl_xor, so the same bits.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// {lo, hi} = v of the lower numbered of lane and lane ^ OFF, and of the other one
template <int OFF>
__device__ __forceinline__ void lane_halves(float v, float& lo, float& hi) {
    static_assert(OFF == 16 || OFF == 32, "rows of 16 lanes, or halves of the wavefront");
    const uint32_t u = __float_as_uint(v);
    if constexpr (OFF == 32) {
        const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        lo = __uint_as_float(p[0]), hi = __uint_as_float(p[1]);
    } else {
        const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        lo = __uint_as_float(p[0]), hi = __uint_as_float(p[1]);
    }
}
template <int OFF>
__device__ __forceinline__ void lane_pair(float v, float& a, float& b) {       // {a, b} = {v, v of lane ^ OFF}, in either order
    static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16 || OFF == 32, "a power of two below 64");
    if constexpr (OFF >= 16) {
        lane_halves<OFF>(v, a, b);
    } else {
        a = v;
        if constexpr (OFF == 8) b = dpp_move<0x128>(v);                         // row_ror:8
        else if constexpr (OFF == 4) b = dpp_move<0x1b>(dpp_move<0x141>(v));    // row_half_mirror, then quad_perm [3,2,1,0]
        else if constexpr (OFF == 2) b = dpp_move<0x4e>(v);                     // quad_perm [2,3,0,1]
        else b = dpp_move<0xb1>(v);                                             // quad_perm [1,0,3,2]
    }
}
template <int OFF>
__device__ __forceinline__ float lane_sum(float v) {
    float a, b;
    lane_pair<OFF>(v, a, b);
    return a + b;
}
template <int OFF>
__device__ __forceinline__ float lane_max(float v) {
    float a, b;
    lane_pair<OFF>(v, a, b);
    return fmaxf(a, b);
}

// Rows as the 16-row matrix instructions want them: lane (r, g) = (lane % 16, lane / 16) holds 16 bytes of row r at place g, so a load of an
// operand takes 64 bytes of each of sixteen rows, and a CU takes a line in at the same cost whole or half. Two operands that are the two halves of 128
// bytes are loaded as a pair instead, lo: 16 bytes of row r % 8 at place g of its half r / 8, hi: the same of row 8 + r % 8; this is half 0 or 1 of
// them for row r. V: four 32-bit values. Every lane is active.
template <typename V>
__device__ __forceinline__ V line_pair_half(int half, V lo, V hi) {
    V o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const auto l = lo[e], h = hi[e];
        // (row_ror:8, written to the upper or the lower eight lanes of each sixteen)
        const int v = half ? __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, h), __builtin_bit_cast(int, l), 0x128, 0xf, 0x3, false)
                           : __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, l), __builtin_bit_cast(int, h), 0x128, 0xf, 0xc, false);
        o[e] = __builtin_bit_cast(std::remove_const_t<decltype(l)>, v);
    }
    return o;
}
// half 1 of rows r < 8, where nobody looks at the others
template <typename V>
__device__ __forceinline__ V line_pair_turned(V lo) {
    V o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const auto l = lo[e];
        o[e] = __builtin_bit_cast(std::remove_const_t<decltype(l)>, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, l), 0x128, 0xf, 0xf, false));
    }
    return o;
}

__device__ __forceinline__ float wave_sum(float v) {
    return lane_sum<1>(lane_sum<2>(lane_sum<4>(lane_sum<8>(lane_sum<16>(lane_sum<32>(v))))));
}

__device__ __forceinline__ float wave_max(float v) {
    return lane_max<1>(lane_max<2>(lane_max<4>(lane_max<8>(lane_max<16>(lane_max<32>(v))))));
}

// Sum over a block of NT threads (NT a multiple of 64, at most 1024). Every thread gets the result.
// The order of the additions is fixed by the thread layout, never by the data.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* smem /* NT/64 floats */) {
    v = wave_sum(v);
    const int wave = threadIdx.x / TM_WAVE, lane = threadIdx.x % TM_WAVE;
    __syncthreads();
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < NT / TM_WAVE; ++w) total += smem[w];
    return total;
}

#define TM_CHECK_LAUNCH()                                        \
    do {                                                         \
        hipError_t e_ = hipGetLastError();                       \
        if (e_ != hipSuccess) return TM_ERR_LAUNCH;              \
    } while (0)
