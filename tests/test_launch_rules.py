"""How launches hand out their work, as the library says on the host."""
import ctypes
import struct

import pytest

from tokenmill_amd.csrc import build
from tokenmill_amd.hip.library import library

THREADS = 2 ** 32                       # a dimension of a launch has fewer


# (query heads, kv heads, head size, wavefronts of a block)
@pytest.mark.parametrize("H,KVH,D,waves", [(2, 1, 128, 2), (28, 4, 128, 4), (40, 8, 128, 4), (16, 1, 96, 8), (48, 4, 128, 8), (12, 2, 64, 4)])
def test_a_dealt_launch_fits_the_grid(H, KVH, D, waves):
    """Pieces dealt out stand in the grid's x; tables beyond what that holds are taken by tiles and kv heads, as they were before pieces were dealt, or in pairs where
    eight wavefronts a block fill the chip with them."""
    lib, most = library(), (THREADS // (64 * waves) - 1) // KVH
    order = lambda n: lib.tm_attn_prefill_shared_order(*map(ctypes.c_int, (H, KVH, D, n)))
    assert order(256 // KVH) == 0 and order(256 // KVH + 1) == 2
    for n in [*range(1, 4000, 3), *range(most - 300, most + 300), 2 ** 31 - 1]:
        folded = -(-n // 2) * KVH
        pairs = waves == 8 and n * KVH > 256 and 100 * folded >= 97 * 256 * -(-folded // 256)
        assert order(n) == (1 if pairs else 2 if 256 // KVH < n <= most else 0), n


@pytest.mark.parametrize("H,KVH,D,heads,waves", [(14, 2, 64, 4, 8), (16, 16, 64, 1, 8), (32, 8, 128, 2, 4), (12, 2, 96, 2, 4), (640, 320, 64, 1, 8)])
def test_an_order_of_pieces_fits_the_grid(H, KVH, D, heads, waves):
    lib, columns = library(), KVH * -(-(H // KVH) // heads)
    order = lambda n: lib.tm_attn_prefill_order(*map(ctypes.c_int, (H, KVH, D, heads, n)))
    for n in [*range(1, 3000, 7), *(THREADS // (64 * waves) // columns + d for d in range(-400, 400)), 2 ** 31 - 1]:
        if order(n) == 2:
            assert n * columns * 64 * waves < THREADS
        elif n * columns <= 256:
            assert order(n) == 0
    assert any(order(n) == 2 for n in range(1, 3000))


# (columns, K, rows at which neighbouring lanes load side by side) of the 32-bit product of few rows
@pytest.mark.parametrize("N,K,rows", [(4096, 768, range(1, 17)), (4096, 896, range(5, 17)), (4096, 1536, range(5, 17)), (4096, 1568, range(2, 17)), (3552, 1536, range(1, 17)),
                                      (6144, 704, range(1, 17)), (6144, 768, range(5, 17)), (6144, 896, range(5, 17)), (6144, 928, range(1, 17)), (32768, 896, []),
                                      (32800, 896, [16]), (151936, 896, [16]), (151936, 928, range(1, 17)), (9728, 912, []), (1536, 144, range(1, 17)), (1536, 176, []),
                                      (1536, 496, []), (1536, 528, range(1, 17)), (1536, 192, range(1, 17)), (8224, 176, range(1, 17))])
def test_lanes_of_a_32_bit_product_load_side_by_side_where_that_pays(N, K, rows):
    """Both sides of each line: rows that are no whole lines, two groups of steps a wavefront, one row of a block alone on its CU."""
    assert [m for m in range(1, 17) if library().tm_gemv_f32_turns(*map(ctypes.c_int, (m, N, K)))] == list(rows)


# (columns, K, row stride, tokens at which the activations' pieces change lanes) of the packed product of few tokens: strips of 4, 8 and 16 rows
@pytest.mark.parametrize("N,K,lda,tokens", [(896, 4864, 4864, [3, 4, 6, 7, 8, *range(12, 17)]), (896, 4864, 4872, []), (896, 4856, 4864, [3, 4, 6, 7, 8, *range(12, 17)]),
                                            (896, 4856, 4856, []), (896, 2016, 2016, []), (1536, 2048, 2048, range(4, 17)), (1536, 2016, 2016, []),
                                            (3584, 2048, 2048, range(6, 17)), (3584, 2016, 2016, range(10, 17)), (3584, 512, 512, range(10, 17)), (3584, 480, 480, []),
                                            (3584, 904, 904, []), (4096, 4096, 4096, range(10, 17))])
def test_activations_change_lanes_where_that_pays(N, K, lda, tokens):
    """Both sides of each line: a short K, places without a token, rows that are no whole pieces of 64 bytes."""
    assert [m for m in range(1, 17) if library().tm_skinny_turns(*map(ctypes.c_int, (m, N, K, lda)))] == list(tokens)


# (token tiles, wavefronts a unit, units a block), k-steps a wavefront at which a round has eight of them
@pytest.mark.parametrize("shape,eight", [((1, 8, 1), [6, 7, 8, *range(13, 40)]), ((1, 4, 2), [6, 7, 8, *range(9, 40)]), ((1, 2, 8), range(6, 40)), ((2, 8, 1), []), ((3, 8, 1), []),
                                         ((2, 4, 2), [5, 6, 7, 8, *range(13, 17), *range(21, 40)]), ((4, 2, 4), [5, 6, 7, 8, *range(13, 17), *range(21, 40)]), ((4, 2, 5), [])])
def test_rounds_of_a_streamed_product_have_eight_steps_where_that_pays(shape, eight):
    """Both sides of each line: a second round for a few steps, two tiles of tokens with eight wavefronts a unit, more wavefronts than have the registers."""
    assert [per for per in range(1, 40) if library().tm_stream_round(*map(ctypes.c_int, (*shape, per))) == 8] == list(eight)


# (rows, columns, K, the first table's tile, the one that runs): a tile between the table's on both sides of what says that it may be taken
@pytest.mark.parametrize("M,N,K,table,runs", [(264, 7536, 7808, 6, 6), (231, 9096, 1728, 6, 11), (750, 3120, 4416, 6, 6), (3651, 1288, 5248, 5, 5), (3104, 1392, 11392, 5, 5),
                                              (615, 9832, 1280, 4, 14), (311, 10144, 9920, 6, 6), (287, 11024, 2048, 7, 12), (3562, 544, 1408, 8, 8), (2325, 1160, 384, 10, 11),
                                              (1605, 3072, 832, 5, 13), (2322, 1672, 1472, 5, 12)])
def test_tiles_between_are_taken_where_they_pay(M, N, K, table, runs):
    args = [ctypes.c_int(x) for x in (M, N, K, 1)]
    assert (library().tm_gemm_tile_shape(*args), library().tm_gemm_tile_picked(*args)) == (table, runs)


def test_the_decode_attentions_pair_of_kernels_begins_at_multiples_of_8_kib():
    """Where they lie in their code object is worth 2% of a step, so it does not hang on what stands before them. Read from the code objects' symbol tables."""
    library()                                       # built if it is not there
    data, found, at = build.find_library().read_bytes(), {}, 0
    while (at := data.find(b"\x7fELF\x02", at)) >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:           # EM_AMDGPU
            table, = struct.unpack_from("<Q", data, at + 40)
            size, count = struct.unpack_from("<HH", data, at + 58)
            sections = [struct.unpack_from("<IIQQQQI", data, at + table + size * i) for i in range(count)]
            for _, kind, _, _, offset, length, link in sections:
                for s in range(offset, offset + length, 24) if kind == 11 else ():      # SHT_DYNSYM
                    name, info, _, _, value, _ = struct.unpack_from("<IBBHQQ", data, at + s)
                    start = at + sections[link][4] + name
                    if info & 15 == 2:                                                  # STT_FUNC
                        found[data[start:data.index(b"\0", start)].decode()] = value
        at += 4
    pair = {name: value for name, value in found.items() if "attn_decode_split_kernel" in name or "attn_decode_merge_kernel" in name}
    assert len(pair) == 4 * 2 + 1 and not any(value % 8192 for value in pair.values()), pair
