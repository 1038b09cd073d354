"""Decoded tokens attended in the launch of prompt portions: the bits of the two launches, where the decoded tokens fill less than a layer of the
grid, exactly one and several, with one, two and four heads a wavefront, folded tables, windows, kept keys, caps, sinks, gates."""
from __future__ import annotations

import ctypes

import pytest
import torch

from tokenmill_amd.hip.library import library

pytestmark = pytest.mark.gpu
P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
PAGE = 16


def _ptr(t):
    return P(t.data_ptr() if t is not None else None)


@pytest.mark.parametrize("extras", ["plain", "window+keep", "cap+sink+gate"])
@pytest.mark.parametrize("H,KVH,D,portions,contexts", [
    (14, 2, 64, [(482, 241), (482, 241)], [1000, 17, 256, 257, 640]),     # four heads a wavefront
    (14, 2, 64, [(0, 40)], [1, 64, 65, 1536]),                            # two heads; the longest context
    (14, 2, 64, [(3, 5)], list(range(1, 130, 2))),                        # more pairs than a layer of the grid has blocks
    (4, 4, 64, [(0, 17)], [300, 5]),                                      # exactly a layer; one head
    (4, 2, 32, [(100, 33), (0, 1)], [700] * 3),
    (14, 2, 64, [(0, 2100)], [900, 33]),                                  # a folded table
])
def test_bits_of_the_two_launches(H, KVH, D, portions, contexts, extras):
    lib, g = library(), torch.Generator(device="cuda").manual_seed(H + D + len(contexts))
    lens = [a + b for a, b in portions] + contexts
    R, S, W = len(lens), len(contexts), -(-max(lens) // PAGE)
    tokens = sum(b for _, b in portions)
    k = torch.randn(R * W, PAGE, KVH, D, generator=g, device="cuda").bfloat16()
    v = torch.randn(R * W, KVH, D, PAGE, generator=g, device="cuda").bfloat16()
    table = torch.randperm(R * W, generator=g, device="cuda").int().view(R, W)
    ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
    q = torch.randn(tokens + S, H * D, generator=g, device="cuda").bfloat16()
    tiles, row = [], 0
    for s, (before, n) in enumerate(portions):
        tiles += [(s, row + i, min(16, n - i), before + i) for i in range(0, n, 16)]
        row += n
    tiles = torch.tensor(sorted(tiles, key=lambda t: -t[3]), dtype=torch.int32, device="cuda")
    window, keep = (200, 20) if extras == "window+keep" else (0, 0)
    full = extras == "cap+sink+gate"
    cap, sink = (30.0, torch.randn(H, generator=g, device="cuda")) if full else (0.0, None)
    gate = torch.randn(tokens + S, H * D, generator=g, device="cuda").bfloat16() if full else None
    chunks = -(-max(contexts) // 256)
    two, one = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    pools = (_ptr(k), _ptr(v))
    ends = (I(H), I(KVH), I(D), I(PAGE), F(D ** -0.5), I(window), I(keep), F(cap), _ptr(sink))
    gate_d = gate[tokens:] if full else None
    stream = P(torch.cuda.current_stream().cuda_stream)
    assert lib.tm_attn_prefill_mfma_cap(_ptr(q), I(H * D), _ptr(two), I(H * D), *pools, _ptr(table), I(W), _ptr(tiles), I(len(tiles)), *ends, _ptr(gate),
                                        I(H * D), stream) == 0
    assert lib.tm_attn_decode_whole(_ptr(q[tokens:]), I(H * D), _ptr(two[tokens:]), I(H * D), *pools, _ptr(table[len(portions):]), I(W),
                                    _ptr(ctx[len(portions):]), I(chunks), I(S), *ends, _ptr(gate_d), I(H * D), stream) == 0
    assert lib.tm_attn_prefill_decodes(_ptr(q), I(H * D), _ptr(one), I(H * D), *pools, _ptr(table), I(W), _ptr(tiles), I(len(tiles)), _ptr(q[tokens:]),
                                       _ptr(one[tokens:]), _ptr(table[len(portions):]), _ptr(ctx[len(portions):]), I(chunks), I(S), *ends, _ptr(gate),
                                       _ptr(gate_d), I(H * D), stream) == 0
    assert not one.isnan().any() and torch.equal(one, two)


@pytest.mark.parametrize("n", [1040, 1740, 2048])
def test_bits_of_the_two_launches_in_every_order_of_the_pieces(n):
    """Dealt out, and folded below and at a block a CU."""
    test_bits_of_the_two_launches(14, 2, 64, [(0, n)], [900, 33], "plain")


def test_what_the_launch_does_not_take_is_refused():
    lib = library()
    t = torch.zeros(1 << 16, dtype=torch.bfloat16, device="cuda")
    i = torch.zeros(64, dtype=torch.int32, device="cuda")

    def call(D=64, chunks=1, n=1, tiles=1, offset=0, H=14):
        return lib.tm_attn_prefill_decodes(_ptr(t), I(H * D), _ptr(t), I(H * D), _ptr(t), _ptr(t), _ptr(i), I(1), _ptr(i), I(tiles), _ptr(t), P(t.data_ptr() + offset),
                                           _ptr(i), _ptr(i), I(chunks), I(n), I(H), I(2), I(D), I(PAGE), F(0.1), I(0), I(0), F(0), _ptr(None), _ptr(None),
                                           _ptr(None), I(0), P(torch.cuda.current_stream().cuda_stream))

    for wrong in (dict(D=128), dict(chunks=17), dict(chunks=0), dict(n=0), dict(n=40000), dict(tiles=0), dict(offset=4), dict(H=34)):
        assert call(**wrong) != 0, wrong
