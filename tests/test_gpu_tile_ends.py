"""How the tiled products end: blocks whose last tile has nothing behind it to load, with K just as deep as the ring and with several
tiles a block, and the head of a unit of columns without a division."""
from __future__ import annotations

import pytest
import torch

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("K", [256, 320, 896])
@pytest.mark.parametrize("shape", range(11))
def test_the_last_tile_of_every_block(shape, K):
    from tokenmill_amd.hip import ops
    from tokenmill_amd.hip.library import library

    lib = library()
    sizes = [(M, N) for M in (66, 97, 130, 261, 515, 700, 1030, 1500, 2049, 4097) for N in (72, 904, 1800, 3592, 9720, 20000)
             if lib.tm_gemm_tile_shape(M, N, K, 1) == shape]
    if not sizes:
        pytest.skip("no size of these runs with this tile")
    for M, N in {sizes[0], sizes[-1]}:                  # a tile a block; where the rule has such sizes, several
        g = torch.Generator(device="cuda").manual_seed(M + N)
        a = torch.randn(M, K, generator=g, device="cuda").bfloat16()
        w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
        out = torch.full((M, N), float("nan"), device="cuda")
        ops.tile_linear(a, w, out)
        want = a.double() @ w.double().T
        # one chain of K / 8 additions of products of size K ** -0.5: below 2^-24 of some 2 K ** 0.5, K / 8 times at the worst
        assert ((out.double() - want).abs() <= 2.0 ** -24 * (K / 8) * 4).all(), (M, N)


def test_a_units_head_without_a_division():
    """unit_inverse and unit_head of csrc/fused_common.h: the host's inverse and the kernel's upper half of a 64-bit product, as numbers."""
    for d in range(1, 17):
        inverse = ((1 << 31) + d - 1) // d
        assert inverse < 1 << 32
        for u in [*range(0, 70000), 10 ** 7, 10 ** 7 + d - 1]:
            assert ((2 * u + 1) * inverse) >> 32 == u // d
