"""Plain products of prompts through the tiled kernel, in either type, against 64 bits: rows and columns that fill no tile, and
both sides of the line up to which they run in place of the library's."""
from __future__ import annotations

import pytest
import torch

from tokenmill_amd.hip import ops
from tokenmill_amd.parts.linear import Linear

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16
SIZES = [(65, 8, 256), (77, 2432, 320), (333, 4864, 256), (257, 9728, 448), (512, 9728, 896), (1000, 2048, 2048), (1025, 40, 256), (2048, 9728, 896), (4001, 1360, 1024),
         (2000, 4096, 1792), (33, 1000, 1024), (5, 648, 512), (1500, 2048, 512), (2048, 1536, 512)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("out_dtype", [BF, torch.float32])
def test_plain_product(M, N, K, out_dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    wide = torch.randn(M, K + 64, generator=g, device=DEV).to(BF)
    a, w = wide[:, :K], (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)
    out = torch.full((M + 1, N), 7.0, dtype=out_dtype, device=DEV)
    ops.tile_linear(a, w, out[:M])
    want = a.double() @ w.double().T
    # the sum's own error (32-bit, K products of K ** -0.5 against unit values), and one rounding to 8 bits
    bound = 1e-6 * want.abs().max() + (2.0 ** -8 * want.abs() if out_dtype == BF else 0)
    assert ((out[:M].double() - want).abs() <= bound + 1e-6).all() and (out[M] == 7).all()


@pytest.mark.parametrize("M", [255, 256, 1500, 3072, 3073])
@pytest.mark.parametrize("N,K", [(512, 1024), (4096, 1024), (1360, 4096), (4104, 1024)])
def test_a_linear_on_both_sides_of_the_line(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M)
    lin = Linear(K, N, "w", bias=False)
    lin.load({"w.weight": (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)}, "")
    lin.prepare(False)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF)
    want = x.double() @ lin.weight.double().T
    for out_dtype in (BF, torch.float32):
        got = lin.forward(x, out_dtype=out_dtype)
        assert (got.double() - want).norm() < (2.0 ** -8 if out_dtype == BF else 1e-6) * want.norm()
        tiled = torch.empty_like(got)
        if 256 <= M <= 3072 and N <= 4096:
            assert torch.equal(got, ops.tile_linear(x, lin.weight, tiled))
