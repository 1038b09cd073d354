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
