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


@pytest.mark.parametrize("N,K,tiled", [(512, 1024, {256, 640, 1024, 1200, 2048, 2560}), (504, 1024, set()), (512, 960, set()),
                                       (2048, 1216, {256, 640, 1024, 1200, 2048, 2560}), (2056, 1216, set()), (1024, 2304, {640, 1024}), (512, 4096, set()),
                                       (1360, 2304, {1200, 2048}), (1024, 2368, set()), (1032, 1280, set()), (2056, 2304, set()), (4096, 1024, set())])
def test_a_linear_on_both_sides_of_the_lines(N, K, tiled):
    """The ranges of rows that a plain product of each size runs tiled in: at their ends and one beyond."""
    from tokenmill_amd import profiling

    g = torch.Generator(device=DEV).manual_seed(N)
    lin = Linear(K, N, "w", bias=False)
    lin.load({"w.weight": (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)}, "")
    lin.prepare(False)
    for M in (255, 256, 639, 640, 1024, 1025, 1199, 1200, 2048, 2049, 2560, 2561):
        x = torch.randn(M, K, generator=g, device=DEV).to(BF)
        want = x.double() @ lin.weight.double().T
        for out_dtype in (BF, torch.float32):
            with profiling.collect() as seen:
                got = lin.forward(x, out_dtype=out_dtype)
            ran = any("gemm_tile_kernel" in name for name in seen["kernels"])
            inside = M in tiled or (len(tiled) == 6 and M in (639, 1025, 1199, 2049))
            assert ran == inside, (M, seen["kernels"])
            assert (got.double() - want).norm() < (2.0 ** -8 if out_dtype == BF else 1e-6) * want.norm()
            if inside:
                assert torch.equal(got, ops.tile_linear(x, lin.weight, torch.empty_like(got)))


@pytest.mark.parametrize("N,K,tiled", [(32000, 1024, True), (16384, 256, True), (32004, 1024, False), (32000, 1056, False), (204808, 2048, False), (204808, 1984, True),
                                         (264, 512, True), (4088, 576, False), (4096, 1024, True), (4096, 1088, False), (65528, 1088, False), (65536, 1088, True),
                                         (65536, 6144, True), (65536, 6208, False), (541200, 1984, True), (541208, 1984, False)])
def test_an_output_head_on_both_sides_of_the_lines(N, K, tiled):
    """Rows of a head that the tiled kernel takes from the library: their ends and one beyond, sizes it does not have; a row does not depend on the others."""
    from tokenmill_amd import profiling

    g = torch.Generator(device=DEV).manual_seed(N)
    lin = Linear(K, N, "w", bias=False, library_first=True)
    lin.load({"w.weight": (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)}, "")
    lin.prepare(False)
    x = torch.randn(65, K, generator=g, device=DEV).to(BF)
    want, got = x.double() @ lin.weight.double().T, {}
    for M in (16, 17, 33, 64, 65):
        with profiling.collect() as seen:
            got[M] = lin.forward(x[:M], out_dtype=torch.float32)
        assert any("gemm_tile_kernel" in name for name in seen["kernels"]) == (tiled and 16 < M <= 64), (M, seen["kernels"])
        assert (got[M].double() - want[:M]).norm() < 1e-6 * want[:M].norm()
    if tiled:
        assert torch.equal(got[64][:17], got[17]) and torch.equal(got[64][:33], got[33])
