"""The bfloat16 attention of prompt portions that splits keys: one, two and more heads of a kv head a wavefront give a head the same bits."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("n,window,softcap", [(1, 0, 0.0), (17, 0, 0.0), (333, 0, 0.0), (333, 70, 0.0), (260, 0, 20.0), (2100, 0, 0.0)])
def test_a_heads_bits_do_not_depend_on_the_heads_beside_it(D, n, window, softcap):
    from tokenmill_amd.hip import ops

    H, page = 7, 16
    g = torch.Generator(device=DEV).manual_seed(n + D)
    pages = -(-n // page)
    q = torch.randn(n, H * D, generator=g, device=DEV).to(BF)
    k, v = torch.randn(pages, page, 1, D, generator=g, device=DEV).to(BF), torch.randn(pages, 1, D, page, generator=g, device=DEV).to(BF)
    tables = torch.randperm(pages, generator=torch.Generator().manual_seed(n)).int().to(DEV).view(1, -1)
    tiles = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)

    def attend(lo, hi):
        out = torch.full((n, (hi - lo) * D), 3.0, dtype=BF, device=DEV)
        ops.attn_prefill_mfma(q[:, lo * D:hi * D].contiguous(), out, k, v, tables, tiles, hi - lo, 1, D, D ** -0.5, window, softcap=softcap)
        return out.view(n, hi - lo, D)

    every = attend(0, H)
    for lo, hi in ((0, 1), (6, 7), (2, 4), (3, 6)):
        assert torch.equal(attend(lo, hi), every[:, lo:hi]), (lo, hi)
    keys, values = k[tables[0].long()].view(-1, D)[:n].double(), v[tables[0].long()].permute(0, 3, 1, 2).reshape(-1, D)[:n].double()
    s = torch.einsum("qhd,kd->hqk", q.view(n, H, D).double(), keys) * D ** -0.5
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    far = torch.arange(n, device=DEV)[:, None] - torch.arange(n, device=DEV)
    s = s.masked_fill((far < 0) | (far >= (window or n)), float("-inf"))
    want = torch.einsum("hqk,kd->qhd", s.softmax(-1), values)
    # weights and results are rounded to 8 bits: 2^-9 of the largest value each, the capped score's fast tanh adds below that
    assert (every.double() - want).abs().max() < 3 * 2.0 ** -9 * values.abs().max()


@pytest.mark.parametrize("shared,D,KVH,tiles", [(True, 96, *case) for case in ((4, 64), (4, 65), (3, 86), (2, 255), (3, 170), (4, 128), (3, 171), (16, 47),
                                                                              (257, 1), (257, 2))]
                         + [(False, D, *case) for D in (64, 96) for case in ((4, 65), (4, 108), (4, 109), (4, 128), (4, 129), (4, 217), (3, 87), (257, 2))])
def test_every_piece_of_a_launch_is_somebodys(shared, D, KVH, tiles, G=2):
    """From 257 pieces (tile, kv head, its heads) on a launch's blocks take them dealt out over all heads, in reverse among the second 256 (the
    shared-keys kernel), or dealt or a tile from either end of the table (the other): the same bits as calls on parts of the table so few that every
    block takes the piece of its own place."""
    from tokenmill_amd.hip import ops

    page, n = 16, 16 * tiles - 3
    H = KVH * G
    g = torch.Generator(device=DEV).manual_seed(tiles)
    q = torch.randn(n, H * D, generator=g, device=DEV).to(BF)
    k, v = torch.randn(tiles, page, KVH, D, generator=g, device=DEV).to(BF), torch.randn(tiles, KVH, D, page, generator=g, device=DEV).to(BF)
    tables = torch.arange(tiles, dtype=torch.int32, device=DEV).view(1, -1)
    table = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)

    def attend(rows, heads, out):
        lo, hi = heads
        ops.attn_prefill_mfma(q.view(n, H, D)[:, lo * G:hi * G].reshape(n, -1), out, k[:, :, lo:hi].contiguous(), v[:, lo:hi].contiguous(),
                              tables, table[rows], (hi - lo) * G, hi - lo, D, D ** -0.5, 0, shared=shared)

    dealt = torch.full((n, H * D), 3.0, dtype=BF, device=DEV)
    attend(slice(0, tiles), (0, KVH), dealt)
    wide = min(KVH, 128)
    for lo in range(0, KVH, wide):
        heads = (lo, min(lo + wide, KVH))
        part = torch.full((n, (heads[1] - lo) * G * D), 3.0, dtype=BF, device=DEV)
        for t in range(0, tiles, 256 // wide):
            attend(slice(t, t + 256 // wide), heads, part)
        assert torch.equal(part.view(n, -1), dealt.view(n, KVH, -1)[:, lo:heads[1]].reshape(n, -1))


@pytest.mark.parametrize("D,KVH,G,tiles", [(96, 1, 10, 257), (96, 1, 10, 400), (128, 2, 16, 256), (128, 1, 9, 513), (96, 2, 5, 200), (128, 4, 7, 128)])
def test_every_piece_of_a_launch_of_many_heads_is_somebodys(D, KVH, G, tiles):
    """Blocks of four wavefronts, whose second 256 pieces stand in reverse, and of eight, whose pieces do not."""
    test_every_piece_of_a_launch_is_somebodys(True, D, KVH, tiles, G)


# (head size, kv heads, heads of each, tokens, page, window, softcap, shared keys) and what the bits of the result add up to (bits_of_a_prompt)
BITS = {
    (32, 2, 3, 300, 16, 0, 0.0, False): 273273644921,
    (64, 2, 7, 33, 16, 0, 0.0, False): 903370577692,
    (64, 2, 7, 700, 64, 0, 0.0, False): 263496069408,
    (64, 1, 4, 333, 32, 70, 0.0, False): 291748353217,
    (96, 2, 3, 260, 16, 0, 20.0, False): 543656972435,
    (128, 4, 2, 500, 16, 0, 0.0, False): 767424335260,
    (96, 2, 5, 260, 16, 0, 0.0, True): 154814135182,
    (128, 4, 7, 500, 32, 90, 0.0, True): 16163658554,
}


def bits_of_a_prompt(D, KVH, G, n, page, window, softcap, shared):
    """Attention over numbers made from their places; its bits weighted and added up modulo 2^40."""
    from tokenmill_amd.hip import ops

    def numbers(*size, seed):
        i = torch.arange(torch.Size(size).numel()) * 2654435761 + seed * 40503
        i = (i ^ (i >> 13)) * 1103515245 % 2 ** 31
        return ((i >> 8) % 4096 - 2048).float().div(800).view(size).to(BF).to(DEV)

    pages, H = -(-n // page), KVH * G
    out = torch.empty(n, H * D, dtype=BF, device=DEV)
    tables = torch.arange(pages - 1, -1, -1, dtype=torch.int32, device=DEV).view(1, -1)
    tiles = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)
    ops.attn_prefill_mfma(numbers(n, H * D, seed=1), out, numbers(pages, page, KVH, D, seed=2), numbers(pages, KVH, D, page, seed=3), tables, tiles,
                          H, KVH, D, D ** -0.5, window, softcap=softcap, shared=shared)
    bits = out.view(torch.int16).long().flatten().cpu()
    return int((bits * (torch.arange(bits.numel()) % 1000003 + 1)).sum()) % 2 ** 40


@pytest.mark.parametrize("case", BITS)
def test_the_bits_of_a_prompt_stay(case):
    """The order in which keys are added up, within a block of the matrix unit too, is part of what a prompt gives: the same numbers by any way the
    keys and values are loaded. Which keys of a block stand in which place shows in the last bits alone, and nowhere else."""
    assert bits_of_a_prompt(*case) == BITS[case]


@pytest.mark.parametrize("D,KVH,G", [(32, 2, 3), (64, 2, 7), (64, 2, 2), (96, 3, 2), (96, 3, 1), (128, 2, 4)])
@pytest.mark.parametrize("n", [31, 300])
def test_the_size_of_a_page_changes_no_bit(D, KVH, G, n):
    """Values come in other pieces out of pages of 16 than out of longer ones."""
    from tokenmill_amd.hip import ops

    g = torch.Generator(device=DEV).manual_seed(D + n)
    H, most = KVH * G, 64 * -(-n // 64)
    q, k, v = (torch.randn(m, heads, D, generator=g, device=DEV).to(BF) for m, heads in ((n, H), (most, KVH), (most, KVH)))
    tiles = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)
    got = []
    for page in (16, 32, 64):
        out = torch.full((n, H * D), 3.0, dtype=BF, device=DEV)
        tables = torch.arange(most // page, dtype=torch.int32, device=DEV).view(1, -1)
        ops.attn_prefill_mfma(q.view(n, -1), out, k.view(-1, page, KVH, D), v.view(-1, page, KVH, D).permute(0, 2, 3, 1).contiguous(), tables, tiles, H, KVH, D,
                              D ** -0.5, 0)
        got.append(out)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
