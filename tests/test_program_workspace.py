"""What a step's workspace holds (csrc/step_program.hip, tm_program_workspace_bytes): asked of the library on the host, no kernel runs."""
from __future__ import annotations

import pytest

from tokenmill_amd.hip import abi

HIDDEN, LIMIT = 896, 32768
F32, BF16 = 0, 1


def _attention_program(dtype, heads, kv_heads, head_dim, page=16):
    lib = abi.bound()
    place = 4096                                                # (never read)
    op = abi.TmAttentionOp(qkv=abi.TmLinear(w=place, N=(heads + 2 * kv_heads) * head_dim, K=HIDDEN, dtype=dtype, bias_dtype=-1),
                           o=abi.TmLinear(w=place, N=HIDDEN, K=heads * head_dim, dtype=dtype, bias_dtype=-1), k_pool=place, v_pool=place, H=heads,
                           KVH=kv_heads, D=head_dim, scale=1.0, page=page)
    p = lib.tm_program_create(dtype, HIDDEN)
    assert lib.tm_program_add_attention(p, op) == 0
    return lib, p


def _grows_by(dtype, heads, kv_heads, head_dim, requests, context, page=16):
    """Bytes that a limit of ``context`` adds to a step of single tokens over a limit that no chunk is needed for."""
    lib, p = _attention_program(dtype, heads, kv_heads, head_dim, page)
    grown = lib.tm_program_workspace_bytes(p, requests, requests, requests, context)
    none = lib.tm_program_workspace_bytes(p, requests, requests, 0, 0)
    lib.tm_program_destroy(p)
    return grown - none


def _chunked(heads, head_dim, requests, chunks):
    up = lambda n: -(-n // 256) * 256
    return up(requests * heads * head_dim * chunks * 4) + up(requests * heads * chunks * 8)


@pytest.mark.parametrize("dtype,requests,chunk,taken", [(F32, 1, 128, True), (F32, 95, 128, True), (F32, 96, 128, False), (F32, 256, 128, False),
                                                        (BF16, 1, 256, True), (BF16, 95, 256, True), (BF16, 96, 256, False), (BF16, 256, 256, False)])
def test_partial_results_of_the_decode_attention_have_room_only_where_a_kernel_writes_them(dtype, requests, chunk, taken):
    """Beyond 192 (request, kv head) pairs no kernel splits a context: 256 requests under 32,768 tokens would hold 235 MB in 32-bit."""
    assert _grows_by(dtype, 14, 2, 64, requests, LIMIT) == (_chunked(14, 64, requests, LIMIT // chunk) if taken else 0)


@pytest.mark.parametrize("heads,kv_heads,head_dim,page", [(14, 2, 96, 16), (14, 2, 64, 8), (34, 2, 64, 16)])
def test_shapes_that_the_32_bit_kernel_does_not_take_hold_no_room_for_it(heads, kv_heads, head_dim, page):
    assert _grows_by(F32, heads, kv_heads, head_dim, 8, LIMIT, page) == 0


def test_one_chunk():
    """In 32-bit a single chunk passes through the partial results too, in bfloat16 it does not."""
    assert _grows_by(F32, 14, 2, 64, 8, 100) == _chunked(14, 64, 8, 1) and _grows_by(BF16, 14, 2, 64, 8, 256) == 0


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_partial_sums_have_the_room_of_the_projection_with_most_parts(dtype):
    """However many layers there are and whichever comes first: 896 -> 896 and 4,864 -> 896 are cut into different numbers of parts."""
    lib, place = abi.bound(), 4096
    parts = lambda T, K: (lib.tm_tile_linear_parts if dtype == BF16 else lib.tm_tile_f32_parts)(T, HIDDEN, K)      # noqa: E731

    def program(layers):
        p = lib.tm_program_create(dtype, HIDDEN)
        for inside in layers:
            lin = lambda n, k: abi.TmLinear(w=place, N=n, K=k, dtype=dtype, bias_dtype=-1)                          # noqa: E731
            assert lib.tm_program_add_feed_forward(p, abi.TmFfnOp(gate_up=lin(2 * inside, HIDDEN), down=lin(HIDDEN, inside), I=inside)) >= 0
        return p

    first, many, other = program([4864, 896]), program([896, 4864] * 12), program([896])
    for T in (65, 300, 1000, 2048):
        assert parts(T, 4864) > parts(T, 896) or dtype == BF16
        sizes = [lib.tm_program_workspace_bytes(p, T, 1, 0, 0) for p in (first, many, other)]
        size, up = 4 if dtype == F32 else 2, lambda n: -(-n // 256) * 256
        widest = up(T * 2 * 4864 * size) + up(T * 4864 * size) - up(T * 2 * 896 * size) - up(T * 896 * size)
        more = max(parts(T, 4864), parts(T, 896)) - parts(T, 896)
        assert sizes[0] == sizes[1] == sizes[2] + widest + up(more * T * HIDDEN * 4)
    for p in (first, many, other):
        lib.tm_program_destroy(p)
