// The rules by which a step's kernels are chosen, in one place: the row counts up to which each family of
// matrix-product kernels is preferred, and when the decode attention splits a context over blocks. The step
// program (step_program.hip) is the only code that applies them; the Python side reads the numbers through
// tm_rule() where it sizes a buffer or checks an argument, and never decides by them.
#pragma once
#include <stddef.h>

// --- matrix products (bfloat16) ----------------------------------------------------------------------
// up to this many rows the kernels that stream the matrix once win: the products over packed matrices with
// the layer's epilogue (bias, rotary + cache write, SiLU*up, residual add), and the ones that start at the norm
constexpr int TM_SKINNY_ROWS = 16;
// ... while the model is narrow. They keep all of K of every row in LDS (or re-read the rows per block); beyond a
// width of 1,024 the products that stream the matrix through windows of K (gemm_stream.hip, with the partial sums
// of the output and down projections added by the next norm) take over at fewer rows, the wider the earlier.
// Measured on an MI355X, a decode step (ms) with this family against the stream family: width 896 (0.5B shape)
// 16 rows 1.16 against 1.23; width 1,536 (12 layers of 8,960) 8 rows 0.82 against 0.86, 16 rows 0.95 against 0.92;
// width 2,048 (12 layers of 11,008) 4 rows 0.85 against 0.99, 8 rows 0.90 against 1.00, 16 rows 1.10 against 1.06;
// width 3,584 (7B) 1 row 3.38 against 3.53, 4 rows 3.45 against 3.53, 8 rows 3.72 against 3.63, 16 rows 4.42 against
// 3.84; width 5,120 (32B, 16 layers) 1 row 3.64 against 3.49, 4 rows 3.80 against 3.44, 8 rows 4.10 against 3.56,
// 16 rows 4.92 against 3.81. The two families do not mix within a layer: the kernels that start at the norm need the
// residual stream complete, the stream family leaves partial sums for the norm.
inline int tm_skinny_rows(int hidden) { return hidden <= 1024 ? TM_SKINNY_ROWS : hidden < 3072 ? 8 : hidden < 4096 ? 4 : 0; }
// ... and the two of them that start at the norm (q|k|v, gate|up) at most to 8 rows: with 9 to 16 rows in LDS a CU
// holds one block (0.5B shape, 16 rows: 1.195 ms a step against 1.156 with the panel kernels behind a norm of its own)
inline int tm_from_norm_rows(int hidden) { const int s = tm_skinny_rows(hidden); return s < 8 ? s : 8; }
// q|k|v keeps the normed input in LDS behind a norm of its own up to this many rows where it fits (a width of at
// most 1,024): its matrix is small enough that the copy of the input is most of any kernel's work (measured at the
// 0.5B shape, 16 / 32 / 64 rows: 3.7 / 3.8 / 4.4 us against 5.5 / 6.6 / 8.4 streamed). gate|up had such a kernel too; the stream product, with
// the tiles of tokens dealt to two groups of blocks beyond 32 rows, was as fast or faster at every row count while the kernel took twice its
// present time (0.5B shape, a decode step of 12 / 24 / 32 / 48 requests: 1.07 / 1.29 / 1.34 / 1.54 ms against 1.08 / 1.32 / 1.38 / 1.54 ms).
constexpr int TM_PANEL_QKV_ROWS = 64;
// up to this many rows the products stream the packed matrix once for several row tiles, with their epilogues
constexpr int TM_STREAM_ROWS = 64;
// ... except gate|up where a 64-column tile for each CU covers the matrix: the tiled product over the row-major matrix then
// runs in one round with 64 KB of the matrix on their way into each CU. Streamed to tiled, cold matrices, 17 / 64 rows, us:
// 896 -> 2 x 4,864 9.0 / 11.9 to 7.4 / 7.7; 2,048 -> 2 x 5,632 14.4 / 20.8 to 13.0 / 14.2; 3,072 -> 2 x 8,192 (256 tiles)
// 22.7 / 34.6 to 20.4 / 21.5; beyond a tile a CU 1,536 -> 2 x 8,960 16.2 / 19.4 to 15.9 / 22.8, 3,584 -> 2 x 18,944 48.4 / 52.9
// to 62.1 / 66.6.
constexpr int TM_TILE_FEW_COLUMNS = 64 * 256;
// Output and down projections run tiled, K in parts, beyond so many rows: beyond the rows of the kernels that start at the norm
// at widths from 3,072, beyond 16 at smaller ones, and at widths above 4,096 only beyond the streamed products' 64. Against the
// streamed product (the library's for 896 -> 896) with the norm that adds the parts, 8 / 64 rows, us: 896 -> 896 10.4 (of the
// product alone) to 7.2 / 7.8; 4,864 -> 896 10.5 / 14.7 to 8.6 / 10.5; 2,048 -> 2,048 10.4 / 14.5 to 8.9 / 10.3; 3,584 -> 3,584
// 12.9 / 19.0 to 11.5 / 13.4; 18,944 -> 3,584 31.0 / 38.6 to 29.5 / 32.1. In a step of 9 rows the down projections of widths
// 1,536 and 2,048 (K 8,960 and 11,008) were 1.3 and 1.9 us slower tiled, with 24 rows level: hence 16 there. A layer of whole
// steps of 5 / 17 / 40 / 64 single tokens, streamed to tiled: width 3,584 122.7 / 130.1 / 144.2 / 156.1 to 122.7 / 127.7 / 140.0 /
// 150.4; 4,096 (14,336 wide inside) 119.2 / 132.9 / 153.9 / 169.1 to 119.2 / 131.4 / 149.3 / 160.9; 5,120 198.5 / 210.7 / 232.0 /
// 253.2 to 201.3 / 214.2 / 234.0 / 251.6 (the products level, the sums of more parts to add): hence the line behind 4,096.
inline int tm_split_rows(int hidden) { return hidden < 3072 ? TM_SKINNY_ROWS : hidden <= 4096 ? 4 : TM_STREAM_ROWS; }
// (what that does not take, such as a projection with a bias, is streamed where splitting its K over groups of blocks pays:
// tm_stream_linear_parts in gemm_stream.hip; else it is the library's)
// Plain products of prompts that run tiled in place of the library's untimed choice, in three ranges of sizes where that is the better one (cold
// matrices, time of the tiled product over the library's, 60 sizes drawn from each range, any / multiples of 64: mean, worst):
//   256 to 2,560 rows, 512 to 2,048 columns, K below 1,280      0.81, 1.09 / 0.84, 1.09
//   640 to 1,024 rows, up to 1,024 columns, K up to 2,304       0.80, 1.00 / 0.88, 1.02
//   1,200 to 2,048 rows, 1,360 to 2,048 columns, K up to 2,304  0.86, 1.04 / 0.93, 1.06
// and a call takes 8.6 us of the host for the library's 14.2. Beyond them the library is better as often as not, by up to a third: 4,096 -> 512 at
// 300 / 1,000 rows 11.0 / 14.8 us to 15.5 / 16.9, 4,096 -> 1,024 at 300 / 3,001 15.2 / 31 to 18.5 / 35.8, 1,792 -> 2,560 at 500 1.33
// times its time, 2,048 -> 1,360 at 777 to 1,024 1.11 to 1.18, 1,536 -> 4,096 at 1,200 1.14; also 768 -> 3,072 12.5 to 13.2 and 14.3 to 15.8 at
// 1,500 and 2,048 rows, 4,864 -> 896 24.6 to 28.2 at 1,500.
inline bool tm_tile_plain(int M, int N, int K) {
    if (K < 1024 || N < 512) return false;
    return (M >= 256 && M <= 2560 && N <= 2048 && K < 1280) || (M >= 640 && M <= 1024 && N <= 1024 && K <= 2304) ||
           (M >= 1200 && M <= 2048 && N >= 1360 && N <= 2048 && K <= 2304);
}
// most rows one launch of the skinny product takes at all
constexpr int TM_SKINNY_MAX_ROWS = 64;
// most rows the 32-bit matrix-vector product takes
constexpr int TM_GEMV_F32_ROWS = 16;

// Does the kernel for wide products of few bfloat16 rows (gemv_bf16.hip) take an output head from the library? Up to eight rows at every size that it has (from
// 16,384 x 256 to 256,000 x 8,192 the library takes 0.98 to 2.2 times its time, 1.3 on the mean); with more, K of 8,192 is 10 to 20% slower (128,256 rows: 357 to 424 us),
// and K from 3,584 to 5,120 up to 12% in heads of less than 65,536 (50,304 x 5,120: 95 to 107; 65,536 x 5,120 and 151,936 x 5,120 2 and 18% faster).
inline bool tm_head_few(int M, int N, int K) { return M <= 8 || K <= 3072 || (N >= 65536 && K <= 5120); }

// And the tiled kernel, of 17 to 64 rows? It adds all of K up in one chain and has a block a column of tiles, so where these are few and K is long the library, which
// then cuts K, is faster and its error against 64 bits half as large: up to 4,096 columns by K of 768 and more. The tiles' time over the library's and
// the largest of 17, 40 and 64 rows, over 15 widths from 512 to 200,064, cold matrices (up to 4,096 columns K of 1,024 is the library's at 17 rows only):
//   K up to 512             0.46 to 0.98, 24,576 columns at 64 rows 1.05      512 to 4,096 columns, K 2,304 to 6,144    1.0 to 2.9
//   K 768 to 1,024          from 4,096 columns on 0.33 to 0.98, 24,576 and 50,304 columns at 64 rows 1.02 to 1.04
//   K 1,152 to 6,144        8,192 to 50,304 columns 0.62 to 1.4, level on the mean from 16,384 on; from 65,536 on 0.52 to 1.02, 0.88 on the mean
// us, library / tiles, 17 / 33 / 64 rows: 151,936 x 896 65 / 53, 70 / 55, 74 / 64; 151,936 x 2,048 147 / 121, 153 / 129, 158 / 137; 152,064 x 3,584
// 244 / 193, 201 / 201, 218 / 214; 152,064 x 5,120 331 / 274, 293 / 286, 310 / 309; 32,000 x 1,024 24 / 14, 25 / 15, 25 / 16; 200,064 x 3,072 381 / 228, 264 / 241,
// 285 / 258; 262,144 x 1,152 127 / 116, 142 / 124, 147 / 139. 256,000 x 2,304 would be 1 to 4% slower. K of 8,192 is level. From 8,192 columns on the errors are the same
// (128,256 columns alone, from K of 1,536 on, 5 to 9% larger). At 96 and 128 rows the tiles take 0.86 to 1.03 of the library's time. Matrices of 2 GB and more stay
// the library's.
inline bool tm_head_tiled(int M, int N, int K) {
    if (M <= 16 || M > 64 || (long long)N * K >= 1LL << 30) return false;
    return K <= 512 || (K <= 1024 && N >= 4096) || (K <= 6144 && N >= 65536 && (N <= 204800 || K < 2048));
}

// --- decode attention ---------------------------------------------------------------------------------
constexpr int TM_DECODE_CHUNK = 256;        // keys per block of the split decode attention
constexpr int TM_DECODE_F32_CHUNK = 128;    // the same in the 32-bit path, whose contexts are always split below that many pairs
constexpr int TM_DECODE_SPLIT_PAIRS = 192;  // below this many (request, kv head) pairs the split kernels run

inline int tm_decode_chunks(int max_context) { return (max_context + TM_DECODE_CHUNK - 1) / TM_DECODE_CHUNK; }

// Does a decode step of `requests` single tokens split its contexts over blocks (and need the scratch
// memory for their partial results), where the whole kernel below does not take it?
inline bool tm_decode_splits(int requests, int kv_heads, int max_context) {
    return requests * kv_heads < TM_DECODE_SPLIT_PAIRS && tm_decode_chunks(max_context) > 1;
}

// Does one block take all of a (request, kv head)'s context (attn_decode_whole_kernel; asked before the other)? Where there are few pairs two launches
// less a trip to memory stand against one CU's share of the caches, where there are many the chunks would share CUs anyway, and against
// the block kernel (one chunk, or 192 pairs and more) it merges in one pass. max_context is the step's: the longest context of an eager step, and
// of a replayed one the longest that the engine allows (max_model_len), since a graph serves whatever contexts come: with 2,048 allowed no replayed
// step below 192 pairs takes this kernel (0.5B shape, one request of 300 keys 640 us a step for 613, 64 of up to 1,021 sampled 1,218 for 1,188).
// The whole kernel's time over the split kernels', of 1 to 64 requests at 300 / 400 / 512 / 576 / 700 / 768 / 1,024 keys, the least and the most of
//   1 to 64 pairs, D 32     0.72 to 0.85, 0.73 to 0.85, 0.72 to 0.88, 0.77 to 0.94, 0.77 to 0.96, 0.77 to 1.01, 0.85 to 1.17
//                  D 64     0.71 to 0.84, 0.73 to 0.87, 0.74 to 0.90, 0.82 to 1.00, 0.87 to 1.04, 0.87 to 1.08, 1.00 to 1.18
//                  D 96     0.73 to 0.88, 0.79 to 0.92, 0.83 to 1.01, 0.93 to 1.16, 0.99 to 1.22, 1.02 to 1.25, 1.23 to 1.58
//                  D 128    0.74 to 0.84, 0.81 to 0.98, 0.86 to 1.06, 0.95 to 1.12, 1.03 to 1.23, 1.07 to 1.32, 1.28 to 1.67
//   96 and 128,    D 32     0.74 to 0.84, 0.75 to 0.84, 0.75 to 0.84, 0.73 to 0.81, 0.78 to 0.87, 0.78 to 0.88, 0.88 to 0.97 (1,280 keys 0.88 to 0.99)
//                  D 64     0.78 to 0.87, 0.78 to 0.89, 0.79 to 0.90, 0.76 to 0.87, 0.79 to 0.88, 0.81 to 0.92, 0.88 to 1.00 (1,280 keys 0.93 to 1.04)
//                  D 96     0.79 to 0.89, 0.84 to 0.93, 0.91 to 1.01, 0.82 to 0.91, 0.88 to 0.96, 0.89 to 0.97, 1.10 to 1.21
//                  D 128    0.81 to 0.90, 0.89 to 0.97, 0.90 to 0.98, 0.80 to 0.89, 0.90 to 0.97, 0.92 to 0.98, 1.08 to 1.18
// (one, five, seven and 16 heads a kv head; one head is the worst almost everywhere). us, split / whole: one request of 14 heads over 2 of 64, 300 / 700 keys
// 6.7 / 5.2, 6.8 / 6.7. Below 96 pairs the lines lie lower than these alone say: the split kernels' blocks leave room for matrices to be brought ahead of the
// products behind them, and the whole kernel's do not. Steps with contexts of up to 630 keys allowed 694, us, split / whole: the 0.5B shape, 1 / 4 / 16 / 40 requests
// 638 / 659, 658 / 681, 938 / 928, 996 / 992; 7B, of 440 allowed 504, 2 / 12 requests 3,117 / 3,108, 3,207 / 3,198. Against the block kernel, where its keys were loaded in the product's order throughout, by pairs:
//   256,           D 64   300 / 700 / 1,085                    8.2 / 10.9 / 15.8 to 6.9 / 9.8 / 14.3
//   192 and 400,   D 128  the same                             11.5 / 17.9 / 25.2 and 21.5 / 34.7 / 46.6 to 8.3 / 14.4 / 21.9 and 14.6 / 27.0 / 40.2
//   512,           D 64   400 / 700 / 1,000 / 1,280, 16 heads a kv head   12.4 / 20.3 / 27.2 / 32.1 to 11.0 / 18.0 / 25.1 / 32.9
constexpr int TM_DECODE_MANY_PAIRS = 96;
constexpr int TM_DECODE_WHOLE_KEYS = 1280;
constexpr size_t TM_DECODE_WHOLE_LDS = 160 * 1024;
// its LDS: of the four runs of every chunk the maximum and sum of 16 heads and the values of the heads there are, and the former of every chunk
inline size_t tm_decode_whole_lds(int chunks, int group, int head_size) { return (size_t)chunks * (32 + 4 * (32 + group * (head_size + 4))) * 4; }

// From TM_DECODE_SPLIT_PAIRS pairs on: keys up to which a request is attended in the whole kernel's order, whatever the contexts beside it are (the
// block kernel does so too, and takes longer contexts its own way), so that no request's bits hang on its neighbours' lengths, nor a replayed
// step's on the engine's longest. As many chunks as leave the block kernel the blocks a CU that its registers do: two at head size 64, else one.
inline int tm_decode_own_keys(int group, int head_size) {
    const size_t room = head_size == 64 ? TM_DECODE_WHOLE_LDS / 2 : TM_DECODE_WHOLE_LDS;
    const int keys = (int)(room / tm_decode_whole_lds(1, group, head_size)) * TM_DECODE_CHUNK;
    return keys < TM_DECODE_WHOLE_KEYS ? keys : TM_DECODE_WHOLE_KEYS;
}
inline bool tm_decode_whole(int requests, int heads, int kv_heads, int head_size, int max_context) {
    const int pairs = requests * kv_heads;
    if (pairs >= TM_DECODE_SPLIT_PAIRS) return max_context <= tm_decode_own_keys(heads / kv_heads, head_size);
    if (tm_decode_whole_lds(tm_decode_chunks(max_context), heads / kv_heads, head_size) > TM_DECODE_WHOLE_LDS) return false;
    if (pairs >= TM_DECODE_MANY_PAIRS) return max_context <= (head_size <= 64 ? TM_DECODE_WHOLE_KEYS : 768);
    return max_context <= (head_size <= 32 ? 768 : head_size <= 64 ? 576 : 400);
}

// Do a mixed step's prompt portions, of n_tiles tiles, have its decoded tokens beside them in one launch (attn_prefill_mfma_kernel with DECODES)?
// The whole kernel's rule does not hold here: what its blocks take longer than the split kernels' they take beside the portions'. Of two blocks a CU the
// registers hold one, so as many pairs as CUs are the most; contexts (in a replayed step the engine's limit: with 2,048 allowed two launches, and 30 of 1,000
// beside 2 of 241 take 1,752 us for 1,613) end where a block's eight wavefronts have three rounds of keys (16 of 1,500 keys
// beside 1 portion of 100 tokens, the least there is to gain: 12.8 to 13.0 us; beside 2 of 256 14.3 to 13.0); where the pairs are so many that longer
// ones are added up in another order, they end there.
constexpr int TM_DECODE_BESIDE_LDS = 139264, TM_DECODE_BESIDE_KEYS = 1536;
inline bool tm_prefill_takes_decodes(int requests, int heads, int kv_heads, int head_size, int max_context) {
    return requests > 0 && head_size <= 64 && max_context <= TM_DECODE_BESIDE_KEYS && requests * kv_heads <= 256 &&
           (requests * kv_heads < TM_DECODE_SPLIT_PAIRS || max_context <= tm_decode_own_keys(heads / kv_heads, head_size)) &&
           tm_decode_whole_lds(tm_decode_chunks(max_context), heads / kv_heads, head_size) <= TM_DECODE_BESIDE_LDS;
}

// --- prefill attention (bfloat16) ---------------------------------------------------------------------
// Two kernels: one whose wavefronts each load their own key blocks and split a tile's keys among them (many
// short chains: best for short prompts and for small head sizes), and one that stages a tile's keys and values
// through LDS once for all query heads of a kv head (twice the rate at head sizes above 64 from about a thousand
// tokens on, where the first is held back by one wavefront a SIMD). The second needs at least three wavefronts'
// worth of heads (two heads a wavefront) to fill a CU, and a launch of at least a block a CU. us, first / second, at 160, 192, 256, 320 and 512 of its blocks:
// 28 heads over 4 of 128 25.5 / 26.5, 29.1 / 30.0, 38.6 / 37.5, 56.3 / 46.5, 100 / 69; 40 over 8 of 128 15.3 / 16.9, 20.7 / 18.6, 24.9 / 22.4, 32.2 / 26.7, 55.9 / 38.9; 16 over 1
// of 128 84 / 94, 105 / 111, 168 / 144, 249 / 178, 589 / 301. With two kv heads of five to eight heads the first is, since its keys are loaded as rows, the better one
// further on (12 over 2 of 96 19.0 / 37.4, 28.3 / 43.7, 38.9 / 56.1, 52.5 / 69.1, 108 / 107; 16 over 2 of 128 33.2 / 44.4, 39.8 / 51.8, 55.3 / 66.2, 82.6 / 81.7, 168 / 126);
// the line has stayed for what a prompt gives: the two kernels differ by rounding.
inline bool tm_prefill_shares_keys(int D, int H, int KVH, int n_tiles) {
    const int G = H / KVH;
    return D > 64 && G >= 5 && G <= 16 && (long long)n_tiles * KVH >= 256;
}

// The split-keys kernel at head sizes up to 64 takes two heads a wavefront instead of four while the blocks that
// gives are no more than the chip runs at once (one a CU).
constexpr int TM_PREFILL_ONE_ROUND = 256;
