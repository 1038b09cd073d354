// Decode-step products with the RMSNorm in front and the layer's own epilogue behind, for at most 16
// tokens (bfloat16 weights and activations, 32-bit residual stream and sums).
//
//   x = weight * round(resid * rsqrt(mean(resid^2) + eps))     (reference src/infer/model/layers.py:41-44)
//   is computed by every block into LDS (a few KB of L2 reads against a matrix streamed from HBM), then
//
//   QKV epilogue  : y = x Wqkv^T + b; q and k rotated by their token's position; q to a dense
//                   [M, H*D] buffer, k and v straight to their cache slots
//                   (reference src/infer/model/layers.py:142-147,60-64; src/infer/kv/paged_cache.py:40-43)
//   SiLU epilogue : act = silu(x Wgate^T) * (x Wup^T)          (reference src/infer/model/layers.py:163-164)
//
// A unit is two strips of 16 or 8 matrix rows whose results meet in the epilogue (the two halves of a rotary pair; gate and up). Four or
// eight wavefronts split its K; partial sums are added through LDS in wavefront order. A block takes one unit or two at a
// time, and the next ones after them, behind one norm. Everything is rounded where the unfused path stores a bfloat16 tensor, so both
// paths agree up to the order of 32-bit sums.
#include "common.h"
#include "api.h"
#include "fused_common.h"
#include "ahead.h"

#include <type_traits>

// Elements between the rows of x in LDS: whole k-steps, one of zeros and the padding.
__host__ __device__ __forceinline__ int fused_norm_stride(int K) { return fused_x_stride(K) + 32; }

// ROWS: rows of a strip (16 or 8). Short strips leave rows of the MFMA tile empty (their lanes load what the others load)
// and double the number of units, for matrices that would otherwise give fewer blocks than the chip has CUs.
// WAVES: wavefronts that split the K of a unit (4, or 8 for a long K). UNITS: units a block multiplies at once, each by WAVES
// wavefronts of its own; with more units than that times the grid a block goes on to the next ones, after one norm for all.
// PIPE: a wavefront's K range is longer than one group of FD_KCH steps, and two register groups take
// turns so that loads are always in flight (more registers; not worth them when one group holds it all).
//
// These launches are bound by the trips to memory that wait for each other and by what runs between them, not by bytes: marks of
// the clock inside the kernel showed 0.5 us for the positions (by scalar loads) before the first vector load, the residual rows
// waited for BEHIND the matrix that was asked for first (loads come back in their order), and 1.2 us for the norm itself, of
// which the sum's exchange through LDS was half. So everything that hangs on nothing is asked for at once, in the order it is
// needed: positions and slots, residual rows, norm weights, the matrix, the bias; the rotary rows as soon as the positions are
// there; the norm runs while the matrix is on its way. Loads are unconditional: what lies beyond a row, a strip or a wavefront's
// range of k reads as zero by the bounds of its buffer descriptor.
//
// PLAIN: the norm's weights are bfloat16 and the threads that share a row hold all of it in one round of loads (launch_fused_shape):
// straight code from the loads to LDS. The other way takes any K and either type.
template <int EPI, int ROWS, bool PIPE, int WAVES, int UNITS, bool PLAIN, bool AHEAD>
__global__ __launch_bounds__(64 * WAVES * UNITS, WAVES * UNITS == 4 ? 2 : 1) void fused_norm_gemm_kernel(const FusedArgs a,
                                                                                                       const int n_units, const int blocks,
                                                                                                       const TmAhead ahead) {
    constexpr int KCH = PIPE ? FD_KCH_PIPE : FD_KCH;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if constexpr (AHEAD) {
        ahead_with(a.resid, a.norm_w, a.norm_w_f32, a.eps, a.M, a.K, a.W, n_units);
        if constexpr (EPI == FD_EPI_QKV) ahead_with(a.bias, a.bias_f32, a.H, a.KVH, a.D, a.head_inverse, a.cos_t, a.sin_t, a.positions, a.slots);
        else ahead_with(a.up_strip0, a.act_out, a.I);
        if ((int)blockIdx.x >= blocks) return tm_bring_ahead(ahead, blockIdx.x, WAVES * UNITS);
    }
    constexpr int THREADS = 64 * WAVES * UNITS, RC = PLAIN ? fused_row_vectors(THREADS) : FD_RC;
    bf16_t* xs = (bf16_t*)smem_raw;                                  // [4, 8 or 16 rows][fused_norm_stride]
    __shared__ f32x4_t red[UNITS][WAVES][2][64];
    const int K = a.K, M = a.M;
    const int ksteps = (K + 31) / 32;
    const int per = (ksteps + WAVES - 1) / WAVES;
    const int xstride = fused_norm_stride(K);
    const int block_wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TM_WAVE), lane = threadIdx.x % TM_WAVE;
    const int slot_of_block = block_wave / WAVES, wave = block_wave % WAVES;      // which of the block's units, which part of its K
    const int r = lane % 16, g = lane / 16;
    const int ks0 = wave * per;
    const int ks1 = ks0 + per < ksteps ? ks0 + per : ksteps;

    // The matrix comes in strip order: the 16-byte piece of lane (r, g) for k-step ks of strip s lies at
    // ((s * ksteps + ks) * 4 + g) * ROWS + r pieces, so a wavefront's load is one run of ROWS * 64 bytes
    // and a strip is one run of memory; rows and k beyond the matrix are zeros there.
    constexpr int FRAG = 32 * ROWS;                                  // bfloat16 values of a (strip, k-step)
    const int lane_off = (g * ROWS + (r < ROWS ? r : 0)) * 16;
    FusedUnit cu;
    __amdgpu_buffer_rsrc_t wA, wB;                                   // this wavefront's strips, up to the end of its k
    auto take_unit = [&](int u) {
        const bool live = u < n_units;                               // (the same in every lane)
        cu = fused_unit_of<EPI, ROWS>(a, live ? u : 0);
        const int bytes = live && ks1 > ks0 ? ks1 * FRAG * 2 : 0;
        wA = fd_buffer(a.W + (size_t)cu.sA * ksteps * FRAG, bytes);
        wB = fd_buffer(a.W + (size_t)cu.sB * ksteps * FRAG, bytes);
    };
    auto load_group = [&](auto& ga, auto& gb, int base) {
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            const int at = lane_off + (base + j) * (FRAG * 2);
            ga[j].u = __builtin_amdgcn_raw_buffer_load_b128(wA, at, 0, 0);
            gb[j].u = __builtin_amdgcn_raw_buffer_load_b128(wB, at, 0, 0);
        }
    };

    // --- everything that hangs on nothing, in the order it is needed ---
    const int tok = r;                                               // the epilogue's token of this lane
    const bool epi_lane = wave == 0 && tok < M && 4 * g < ROWS;
    int tok_pos = 0, tok_slot = 0;
    if constexpr (EPI == FD_EPI_QKV) {
        const int t = tok < M ? tok : 0;
        tok_pos = a.positions[t];
        tok_slot = (a.slots ? a.slots : a.positions)[t];
    }
    // A row of the residual stream is shared by tpr threads of one wavefront (256 threads: 16 rows x 16 threads, 8 x 32, or 4 x 64);
    // each keeps its first RC vectors in registers between the two passes. Rows beyond M are the last one again, for
    // tokens that do not exist.
    constexpr int LOG_THREADS = THREADS == 256 ? 8 : 9;
    static_assert(THREADS == 1 << LOG_THREADS, "4 or 8 wavefronts");
    const int mpad = fused_rows(M);
    const int tshift = LOG_THREADS - (mpad == 4 ? 2 : mpad == 8 ? 3 : 4) < 6 ? LOG_THREADS - (mpad == 4 ? 2 : mpad == 8 ? 3 : 4) : 6;
    const int tpr = 1 << tshift;
    const int row = threadIdx.x >> tshift, sub = threadIdx.x & (tpr - 1);
    const int step = 4 * tpr;
    const __amdgpu_buffer_rsrc_t rbuf = fd_buffer(a.resid, M * K * 4);
    const __amdgpu_buffer_rsrc_t nbuf = fd_buffer(a.norm_w, a.norm_w_f32 ? 0 : K * 2);
    const int row0 = (row < M ? row : M - 1) * K;
    auto resid_at = [&](int c) {                                     // (beyond the row: a place beyond the buffer)
        return as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(rbuf, c < K ? (row0 + c) * 4 : 0x7ffffff0, 0, 0));
    };
    f32x4_t cache[RC];
    u32x2_t wraw[RC];                                                // bfloat16 weights of the norm
#pragma unroll
    for (int j = 0; j < RC; ++j) cache[j] = resid_at(sub * 4 + j * step);
    if constexpr (PLAIN) {
#pragma unroll
        for (int j = 0; j < RC; ++j) wraw[j] = __builtin_amdgcn_raw_buffer_load_b64(nbuf, (sub * 4 + j * step) * 2, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    FFrag fa[KCH], fb[KCH], fa2[PIPE ? KCH : 1], fb2[PIPE ? KCH : 1];
    int u0 = blockIdx.x;
    take_unit(u0 + slot_of_block * blocks);
    load_group(fa, fb, ks0);
    if constexpr (PIPE) load_group(fa2, fb2, ks0 + KCH);
    __builtin_amdgcn_sched_barrier(0);

    struct EpilogueInputs {
        f32x4_t bias_f[2];          // four rows of a strip as loaded: a 32-bit bias, or
        u32x2_t bias_h[2];          // a bfloat16 one
        f32x4_t cos, sin;
    };
    const int bias_kind = !a.bias ? 0 : (a.bias_f32 ? 2 : 1);       // the same for every lane
    auto epilogue_inputs = [&]() {
        EpilogueInputs e{};
        if constexpr (EPI == FD_EPI_QKV) {
            // lanes beyond the strip's rows (4 g >= ROWS) have no epilogue: they read what group 0 reads
            const int ge = 4 * g < ROWS ? 4 * g : 0;
            const int ia = cu.nA + ge, ib = cu.nB + ge;             // (the bias is 16-byte aligned)
            const int width = (a.H + 2 * a.KVH) * a.D;
            const __amdgpu_buffer_rsrc_t bf = fd_buffer(a.bias, bias_kind == 2 ? width * 4 : 0), bh = fd_buffer(a.bias, bias_kind == 1 ? width * 2 : 0);
            e.bias_f[0] = as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(bf, ia * 4, 0, 0));
            e.bias_f[1] = as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(bf, ib * 4, 0, 0));
            e.bias_h[0] = __builtin_amdgcn_raw_buffer_load_b64(bh, ia * 2, 0, 0);
            e.bias_h[1] = __builtin_amdgcn_raw_buffer_load_b64(bh, ib * 2, 0, 0);
            // value heads have no rotary row: they read that of the first pair and do not use it
            const int jt = cu.head < a.H + a.KVH ? cu.jt : 0;
            const size_t at = (size_t)tok_pos * (a.D / 2) + ROWS * jt + ge;
            e.cos = *(const f32x4_t*)(a.cos_t + at);
            e.sin = *(const f32x4_t*)(a.sin_t + at);
        }
        return e;
    };

    // --- x = norm(resid) into LDS, while the matrix is on its way ---
    EpilogueInputs e_next;
    if (row < mpad) {                                                // (the same in every lane of a wavefront)
        bf16_t* xrow = xs + (size_t)row * xstride;
        auto squares = [](const f32x4_t v) { return v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]; };
        // With two units a block twice as many threads share a row of more than four: vector j of a thread of one unit's wavefronts lies
        // with the lower half of the row's lanes for an even j and with the upper half for an odd one. They exchange the squares and add
        // them in that thread's order, so that a row's factor has the same bits whatever the matrix's height.
        const int halves = UNITS == 1 || mpad == 4 ? 1 : 2;
        auto add_squares = [&](float ss, const f32x4_t (&v)[RC]) {
            if (halves == 1) {
#pragma unroll
                for (int j = 0; j < RC; ++j) ss += squares(v[j]);
            } else {
                float lo[RC], hi[RC];
                if (mpad == 8) {
#pragma unroll
                    for (int j = 0; j < RC; ++j) lane_halves<32>(squares(v[j]), lo[j], hi[j]);
                } else {
#pragma unroll
                    for (int j = 0; j < RC; ++j) lane_halves<16>(squares(v[j]), lo[j], hi[j]);
                }
#pragma unroll
                for (int j = 0; j < RC; ++j) ss = (ss + lo[j]) + hi[j];
            }
            return ss;
        };
        float ss = add_squares(0.f, cache);
        __builtin_amdgcn_sched_barrier(0);
        e_next = epilogue_inputs();                                  // (the positions came before the rows)
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!PLAIN) {
            // the rest of a long row in groups of RC loads that are in flight together
            for (int c0 = sub * 4 + RC * step; c0 - sub * 4 < K; c0 += RC * step) {
                f32x4_t v[RC];
#pragma unroll
                for (int j = 0; j < RC; ++j) v[j] = resid_at(c0 + j * step);
                ss = add_squares(ss, v);
            }
        }
        ss = lane_sum<8>(lane_sum<4>(lane_sum<2>(lane_sum<1>(ss))));
        if (tpr >= 32 * halves) ss = lane_sum<16>(ss);
        if (tpr >= 64 * halves) ss = lane_sum<32>(ss);
        const float rs = rsqrtf(ss / (float)K + a.eps);
        auto emit = [&](int c, const f32x4_t v, const f32x4_t w) {
            uint2 pk;
            pk.x = fd_pack(w[0] * fd_round(v[0] * rs), w[1] * fd_round(v[1] * rs));
            pk.y = fd_pack(w[2] * fd_round(v[2] * rs), w[3] * fd_round(v[3] * rs));
            *(uint2*)(xrow + (c < K ? c : xstride - 4)) = pk;         // (what lies beyond the row: into the padding, which nobody reads)
        };
        auto widen = [](const u32x2_t wv) {
            return f32x4_t{__uint_as_float(wv.x << 16), __uint_as_float(wv.x & 0xffff0000u),
                           __uint_as_float(wv.y << 16), __uint_as_float(wv.y & 0xffff0000u)};
        };
        if constexpr (PLAIN) {
#pragma unroll
            for (int j = 0; j < RC; ++j) emit(sub * 4 + j * step, cache[j], widen(wraw[j]));
        } else {
            // groups of values (the first from the registers, the others read again) and their weights
            const __amdgpu_buffer_rsrc_t wbuf = fd_buffer(a.norm_w, a.norm_w_f32 ? K * 4 : 0);
            for (int c0 = sub * 4; c0 - sub * 4 < K; c0 += RC * step) {
                f32x4_t w[RC];
                if (a.norm_w_f32) {
#pragma unroll
                    for (int j = 0; j < RC; ++j)
                        w[j] = as_f32x4(__builtin_amdgcn_raw_buffer_load_b128(wbuf, c0 + j * step < K ? (c0 + j * step) * 4 : 0x7ffffff0, 0, 0));
                } else {
#pragma unroll
                    for (int j = 0; j < RC; ++j) wraw[j] = __builtin_amdgcn_raw_buffer_load_b64(nbuf, (c0 + j * step) * 2, 0, 0);
#pragma unroll
                    for (int j = 0; j < RC; ++j) w[j] = widen(wraw[j]);
                }
                if (c0 != sub * 4) {
#pragma unroll
                    for (int j = 0; j < RC; ++j) cache[j] = resid_at(c0 + j * step);
                }
#pragma unroll
                for (int j = 0; j < RC; ++j) emit(c0 + j * step, cache[j], w[j]);
            }
        }
        for (int c = K + sub; c < xstride - FD_XPAD; c += tpr) xrow[c] = 0;      // whole k-steps, and one of zeros
    } else {
        e_next = epilogue_inputs();
    }
    __syncthreads();

    const bf16_t* xr = xs + (size_t)(r & (mpad - 1)) * xstride + 8 * g;
    f32x4_t accA, accB;
    auto multiply_group = [&](const auto& ga, const auto& gb, int base) {
#pragma unroll
        for (int j = 0; j < KCH; ++j) {                              // (steps beyond ks1: zeros by the zeros behind the row; an infinity of x would not do)
            FFrag xf;
            xf.u = *(const u32x4_t*)(xr + (base + j < ks1 ? base + j : ksteps) * 32);
            accA = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga[j].b, xf.b, accA, 0, 0, 0);
            accB = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gb[j].b, xf.b, accB, 0, 0, 0);
        }
    };
    for (;;) {
        const EpilogueInputs e = e_next;                                 // asked for before this unit's products began
        accA = f32x4_t{0.f, 0.f, 0.f, 0.f};
        accB = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if constexpr (PIPE) {
            // fa holds group `base` and fa2 the one after it, loaded or on their way: two groups are
            // always in flight while one is multiplied
            for (int base = ks0; base < ks1; base += 2 * KCH) {
                multiply_group(fa, fb, base);
                if (base + 2 * KCH < ks1) load_group(fa, fb, base + 2 * KCH);
                if (base + KCH >= ks1) break;
                multiply_group(fa2, fb2, base + KCH);
                if (base + 3 * KCH < ks1) load_group(fa2, fb2, base + 3 * KCH);
            }
        } else {
            for (int base = ks0; base < ks1; base += KCH) {
                if (base != ks0) load_group(fa, fb, base);
                multiply_group(fa, fb, base);
            }
        }
        // partial sums of the wavefronts, added in wavefront order
        red[slot_of_block][wave][0][lane] = accA;
        red[slot_of_block][wave][1][lane] = accB;
        __syncthreads();

        // the next units' first loads go out before these units' epilogue
        const FusedUnit done = cu;
        const bool done_live = u0 + slot_of_block * blocks < n_units;
        u0 += UNITS * blocks;
        const bool more = u0 < n_units;
        if (more) {
            take_unit(u0 + slot_of_block * blocks);
            load_group(fa, fb, ks0);
            if constexpr (PIPE) load_group(fa2, fb2, ks0 + KCH);
            e_next = epilogue_inputs();
        }

        if (epi_lane && done_live) {
            accA = red[slot_of_block][0][0][lane];
            accB = red[slot_of_block][0][1][lane];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                accA += red[slot_of_block][w][0][lane];
                accB += red[slot_of_block][w][1][lane];
            }
            // lane: token r, rows nA + 4g + i and nB + 4g + i
            if (EPI == FD_EPI_SILU) {
                const int col = done.nA + 4 * g;
                if (col < a.I) {
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float gt = fd_round(accA[i]), up = fd_round(accB[i]);
                        v[i] = gt / (1.f + expf(-gt)) * up;
                    }
                    bf16_t* dst = a.act_out + (size_t)tok * a.I + col;
                    if (col + 4 <= a.I) {
                        *(uint2*)dst = uint2{fd_pack(v[0], v[1]), fd_pack(v[2], v[3])};
                    } else {
                        for (int i = 0; i < 4 && col + i < a.I; ++i) dst[i] = f32_to_bf16(v[i]);
                    }
                }
            } else {
                f32x4_t bA = {0.f, 0.f, 0.f, 0.f}, bB = {0.f, 0.f, 0.f, 0.f};
                if (bias_kind == 2) {
                    bA = e.bias_f[0];
                    bB = e.bias_f[1];
                } else if (bias_kind == 1) {
                    bA = f32x4_t{__uint_as_float(e.bias_h[0].x << 16), __uint_as_float(e.bias_h[0].x & 0xffff0000u),
                                 __uint_as_float(e.bias_h[0].y << 16), __uint_as_float(e.bias_h[0].y & 0xffff0000u)};
                    bB = f32x4_t{__uint_as_float(e.bias_h[1].x << 16), __uint_as_float(e.bias_h[1].x & 0xffff0000u),
                                 __uint_as_float(e.bias_h[1].y << 16), __uint_as_float(e.bias_h[1].y & 0xffff0000u)};
                }
                float xA[4], xB[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    xA[i] = fd_round(accA[i] + bA[i]);
                    xB[i] = fd_round(accB[i] + bB[i]);
                }
                const int slot = a.slots ? tok_slot : -1;
                if (done.head < a.H + a.KVH) {
                    const int half = a.D / 2;
                    const int j0 = ROWS * done.jt + 4 * g;                       // pair index of element 0
                    float y1[4], y2[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        rotate_pair(xA[i], xB[i], e.cos[i], e.sin[i], y1[i], y2[i]);
                    }
                    bf16_t* dst = nullptr;
                    if (done.head < a.H)
                        dst = a.q_out + (size_t)tok * a.H * a.D + (size_t)done.head * a.D + j0;
                    else if (slot >= 0)
                        dst = a.k_pool + ((size_t)slot * a.KVH + (done.head - a.H)) * a.D + j0;
                    if (dst) {
                        *(uint2*)dst = uint2{fd_pack(y1[0], y1[1]), fd_pack(y1[2], y1[3])};
                        *(uint2*)(dst + half) = uint2{fd_pack(y2[0], y2[1]), fd_pack(y2[2], y2[3])};
                    }
                } else if (slot >= 0) {
                    const int vh = done.head - a.H - a.KVH;
                    const int pg = slot >> a.page_shift, in_page = slot & ((1 << a.page_shift) - 1);
                    const int d0 = 2 * ROWS * done.jt + 4 * g;
                    bf16_t* dst = a.v_pool + ((((size_t)pg * a.KVH + vh) * a.D + d0) << a.page_shift) + in_page;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        dst[(size_t)i << a.page_shift] = f32_to_bf16(xA[i]);
                        dst[(size_t)(i + ROWS) << a.page_shift] = f32_to_bf16(xB[i]);
                    }
                }
            }
        }
        if (!more) break;
        __syncthreads();                                                 // the sums have been read: red is free again
    }
}

// Dynamic LDS of a launch: the normed rows.
static int fused_lds_bytes(int M, int K) { return fused_rows(M) * fused_norm_stride(K) * (int)sizeof(bf16_t); }

template <int EPI, int ROWS, bool PIPE, int WAVES, int UNITS, bool PLAIN, bool AHEAD>
static int launch_fused_kernel(const FusedArgs& a, int n_units, int blocks, TmAhead& ahead, hipStream_t stream) {
    const int lds = fused_lds_bytes(a.M, a.K);
    if (lds + (int)sizeof(f32x4_t) * UNITS * WAVES * 2 * 64 > 160 * 1024) return TM_ERR_ARG;
    static int raised = 0;          // largest dynamic LDS size this kernel has been allowed so far
    if (lds > 48 * 1024 && lds > raised) {
        if (hipFuncSetAttribute((const void*)fused_norm_gemm_kernel<EPI, ROWS, PIPE, WAVES, UNITS, PLAIN, AHEAD>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
            return TM_ERR_LAUNCH;
        raised = lds;
    }
    ahead.first = blocks;
    fused_norm_gemm_kernel<EPI, ROWS, PIPE, WAVES, UNITS, PLAIN, AHEAD><<<blocks + (ahead.n ? ahead.blocks : 0), 64 * WAVES * UNITS, lds, stream>>>(
        a, n_units, blocks, ahead);
    TM_CHECK_LAUNCH();
    return TM_OK;
}

template <int EPI, int ROWS, bool PIPE, int WAVES, int UNITS>
static int launch_fused_shape(const FusedArgs& a, int n_units, int blocks, TmAhead& ahead, hipStream_t stream) {
    constexpr int THREADS = 64 * WAVES * UNITS;
    const int share = THREADS / fused_rows(a.M), tpr = share < TM_WAVE ? share : TM_WAVE;
    auto go = [&](auto PLAIN) {
        return ahead.n ? launch_fused_kernel<EPI, ROWS, PIPE, WAVES, UNITS, decltype(PLAIN)::value, true>(a, n_units, blocks, ahead, stream)
                       : launch_fused_kernel<EPI, ROWS, PIPE, WAVES, UNITS, decltype(PLAIN)::value, false>(a, n_units, blocks, ahead, stream);
    };
    if (WAVES == 4 && !a.norm_w_f32 && a.K <= fused_row_vectors(THREADS) * 4 * tpr) return go(std::integral_constant<bool, WAVES == 4>{});
    return go(std::false_type{});
}

// A long K gets 8 wavefronts a unit (shorter K ranges, a faster norm); whether a wavefront's range
// needs more than one register group of loads decides the pipelined variant. With a shorter K a block that has several units
// takes two at a time, so that the second's matrix is on its way with the first's.
template <int EPI, int ROWS>
static int launch_fused(const FusedArgs& a, int n_units, int blocks, TmAhead& ahead, hipStream_t stream) {
    const int ksteps = (a.K + 31) / 32;
    if (a.K >= 2048) {
        return (ksteps + 7) / 8 > FD_KCH ? launch_fused_shape<EPI, ROWS, true, 8, 1>(a, n_units, blocks, ahead, stream)
                                         : launch_fused_shape<EPI, ROWS, false, 8, 1>(a, n_units, blocks, ahead, stream);
    }
    if constexpr (EPI == FD_EPI_SILU) {
        if (n_units > blocks)
            return (ksteps + 3) / 4 > FD_KCH ? launch_fused_shape<EPI, ROWS, true, 4, 2>(a, n_units, blocks, ahead, stream)
                                             : launch_fused_shape<EPI, ROWS, false, 4, 2>(a, n_units, blocks, ahead, stream);
    }
    return (ksteps + 3) / 4 > FD_KCH ? launch_fused_shape<EPI, ROWS, true, 4, 1>(a, n_units, blocks, ahead, stream)
                                     : launch_fused_shape<EPI, ROWS, false, 4, 1>(a, n_units, blocks, ahead, stream);
}

static bool fused_common_ok(int M, int K, const void* resid, const void* W) {
    return M > 0 && M <= 16 && K > 0 && K % 8 == 0 && ((uintptr_t)resid % 16) == 0 && ((uintptr_t)W % 16) == 0;
}

// Rows of a strip of the packed q|k|v matrix that tm_fused_norm_qkv_rope reads: strips of 16 rows where
// they give the chip enough blocks, else of 8; a long K runs one block of 8 wavefronts a CU, and more
// blocks than CUs would mean a second round for a few of them.
extern "C" int tm_fused_qkv_strip_rows(int H, int KVH, int D, int K) {
    const int units16 = (H + 2 * KVH) * (D / 32);
    const bool one_block_a_cu = K >= 2048;
    return (units16 >= 256 || (one_block_a_cu && units16 >= 128)) ? 16 : 8;
}

// q_out[M, H*D], K cache, V cache <- rope(norm(resid) Wqkv^T + b).  Needs M <= 16, D % 32 == 0, a
// rotary table over the whole head, page a power of two. W: the [(H + 2 KVH) D, K] matrix packed in
// strips of tm_fused_qkv_strip_rows(H, KVH, D, K) rows.
int fused_norm_qkv_rope_ahead(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M,
                                      int K, const void* W, const void* bias, int bias_dtype, void* q_out, int H,
                                      int KVH, int D, const float* cos_t, const float* sin_t, const int* positions,
                                      const int* slots, void* k_pool, void* v_pool, int page, TmAhead ahead, hipStream_t stream) {
    if (M == 0) return TM_OK;
    if (!fused_common_ok(M, K, resid, W) || H <= 0 || KVH <= 0 || D <= 0 || D % 32 || !cos_t || !sin_t || !positions ||
        !q_out || ((uintptr_t)q_out % 8) || page <= 0 || (page & (page - 1)) || !(eps > 0.f))
        return TM_ERR_ARG;
    if (slots && (!k_pool || !v_pool)) return TM_ERR_ARG;
    if (bias && ((uintptr_t)bias % 16)) return TM_ERR_ARG;          // read four rows at a time
    FusedArgs a{};
    a.resid = resid; a.norm_w = norm_w; a.norm_w_f32 = norm_w_dtype == TM_F32; a.eps = eps; a.M = M; a.K = K;
    a.W = (const bf16_t*)W; a.bias = bias; a.bias_f32 = bias_dtype == TM_F32;
    a.q_out = (bf16_t*)q_out; a.H = H; a.KVH = KVH; a.D = D; a.cos_t = cos_t; a.sin_t = sin_t;
    a.positions = positions; a.slots = slots; a.k_pool = (bf16_t*)k_pool; a.v_pool = (bf16_t*)v_pool;
    a.page_shift = 0;
    while ((1 << a.page_shift) < page) ++a.page_shift;
    const int units16 = (H + 2 * KVH) * (D / 32);
    const int rows = tm_fused_qkv_strip_rows(H, KVH, D, K);
    a.head_inverse = unit_inverse(D / (2 * rows));
    if (rows == 16) return launch_fused<FD_EPI_QKV, 16>(a, units16, units16, ahead, stream);
    return launch_fused<FD_EPI_QKV, 8>(a, 2 * units16, 2 * units16, ahead, stream);
}

extern "C" int tm_fused_norm_qkv_rope(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M,
                                      int K, const void* W, const void* bias, int bias_dtype, void* q_out, int H,
                                      int KVH, int D, const float* cos_t, const float* sin_t, const int* positions,
                                      const int* slots, void* k_pool, void* v_pool, int page, hipStream_t stream) {
    return fused_norm_qkv_rope_ahead(resid, norm_w, norm_w_dtype, eps, M, K, W, bias, bias_dtype, q_out, H, KVH, D, cos_t, sin_t, positions, slots, k_pool, v_pool, page,
        TmAhead{}, stream);
}

// act[M, I] <- silu(norm(resid) Wg^T) * (norm(resid) Wu^T).  Needs M <= 16. W: Wg [I, K] and Wu [I, K]
// each packed in strips of 16 rows, Wu behind Wg.
int fused_norm_gate_up_silu_ahead(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M,
                                          int K, const void* W, void* act_out, int I, TmAhead ahead, hipStream_t stream) {
    if (M == 0) return TM_OK;
    if (!fused_common_ok(M, K, resid, W) || I <= 0 || !act_out || ((uintptr_t)act_out % 8) || (I % 4) || !(eps > 0.f))
        return TM_ERR_ARG;
    FusedArgs a{};
    a.resid = resid; a.norm_w = norm_w; a.norm_w_f32 = norm_w_dtype == TM_F32; a.eps = eps; a.M = M; a.K = K;
    a.W = (const bf16_t*)W; a.act_out = (bf16_t*)act_out; a.I = I;
    // One round of blocks, every block with the same number of units (as few as leave at most a block a CU), after one
    // norm for all of them: the 0.5B shape's 304 units as 152 blocks of two (a decode step of 8 requests 0.980 to
    // 0.960 ms against 304 blocks of one, of which some CUs held two; 256 blocks of one or two: 0.980), the 7B
    // shape's 1,184 as 237 blocks of five (the same as 256 blocks of four or five).
    const int units = (I + 15) / 16;
    a.up_strip0 = units;
    return launch_fused<FD_EPI_SILU, 16>(a, units, fused_gate_up_blocks(I), ahead, stream);
}

extern "C" int tm_fused_norm_gate_up_silu(const float* resid, const void* norm_w, int norm_w_dtype, float eps, int M,
                                          int K, const void* W, void* act_out, int I, hipStream_t stream) {
    return fused_norm_gate_up_silu_ahead(resid, norm_w, norm_w_dtype, eps, M, K, W, act_out, I,
        TmAhead{}, stream);
}
