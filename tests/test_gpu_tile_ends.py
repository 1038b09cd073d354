"""How the tiled products end: blocks whose last tile has nothing behind it to load, with K just as deep as the ring and with several
tiles a block, and the head of a unit of columns without a division."""
from __future__ import annotations

import pytest
import torch

gpu = pytest.mark.gpu


# (tile, M, N, K): a tile a block, then, where the rule has such sizes (the first eleven tiles), several with a last round that is not full; K as deep as the ring
# (256 for rings of four buffers, 320 for five, 512 for eight; no K is as short as rings of two or three), a step deeper, and longer
SIZES = [(0, 482, 21800, 256), (0, 904, 26168, 256), (0, 897, 26200, 320), (1, 385, 22488, 256), (1, 770, 26160, 256), (1, 776, 26176, 320),
         (2, 353, 21784, 256), (2, 802, 22056, 256), (2, 802, 21768, 320),
         (3, 259, 25840, 256), (3, 513, 27352, 256), (3, 257, 22184, 320), (3, 517, 26264, 320), (3, 516, 26224, 896),
         (4, 229, 26464, 256), (4, 514, 23664, 256), (4, 226, 23592, 320), (4, 515, 21848, 320), (4, 513, 21848, 896),
         (5, 162, 26848, 256), (5, 457, 21824, 256), (5, 323, 13368, 320), (5, 643, 26360, 320), (5, 642, 26176, 896),
         (6, 229, 15064, 256), (6, 97, 26448, 320), (6, 65, 21520, 896), (7, 162, 20408, 256), (7, 99, 15352, 320), (7, 33, 27720, 896),
         (8, 22, 8, 256), (8, 29, 8, 320), (8, 2961, 1288, 320), (8, 34, 28320, 512), (9, 20, 8, 512), (9, 27, 8, 576), (9, 19, 8, 896),
         (10, 17, 16544, 256), (10, 66, 22192, 256), (10, 65, 22336, 320), (10, 66, 22176, 512),
         (11, 258, 10416, 320), (11, 2932, 832, 384), (11, 199, 8288, 896), (12, 2127, 2200, 256), (12, 2756, 1672, 256), (12, 129, 28272, 320), (12, 145, 21800, 512),
         (12, 259, 14008, 896), (13, 867, 6424, 256), (13, 369, 11176, 896), (14, 193, 28552, 256), (14, 193, 24744, 320), (14, 198, 25824, 896)]


@gpu
@pytest.mark.parametrize("shape,M,N,K", SIZES)
def test_the_last_tile_of_every_block(shape, M, N, K):
    from tokenmill_amd.hip import ops
    from tokenmill_amd.hip.library import library

    assert library().tm_gemm_tile_picked(M, N, K, 1) == shape
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    out = torch.full((M, N), float("nan"), device="cuda")
    ops.tile_linear(a, w, out)
    want = a.double() @ w.double().T
    # one chain of K / 8 additions of products of size K ** -0.5: below 2^-24 of some 2 K ** 0.5, K / 8 times at the worst
    assert ((out.double() - want).abs() <= 2.0 ** -24 * (K / 8) * 4).all()


def test_a_units_head_without_a_division():
    """unit_inverse and unit_head of csrc/fused_common.h: the host's inverse and the kernel's upper half of a 64-bit product, as numbers."""
    for d in range(1, 17):
        inverse = ((1 << 31) + d - 1) // d
        assert inverse < 1 << 32
        for u in [*range(0, 70000), 10 ** 7, 10 ** 7 + d - 1]:
            assert ((2 * u + 1) * inverse) >> 32 == u // d
