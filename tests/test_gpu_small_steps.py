"""The products of steps of at most 16 tokens at the edges of how they share a tile: every strip height with every number of
tokens a tile holds, K around whole ranges, values that are no numbers."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from tokenmill_amd.hip import ops as o
    return o


@pytest.mark.parametrize("N", [897, 1540, 3076])                     # strips of 4, 8 and 16 rows, the last one not full
@pytest.mark.parametrize("K", [8, 40, 904, 2040, 2056, 4864])
def test_few_tokens_against_64_bits_and_against_many_tokens(ops, N, K):
    torch.manual_seed(K + N)
    a = torch.randn(20, K, device=DEV).to(BF)
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).to(BF)
    packed = ops.pack_weight(w, ops.skinny_strip_rows(N, K))
    exact = a.double() @ w.double().T
    many = torch.empty(20, N, dtype=torch.float32, device=DEV)       # the kernel of more than 16 rows: its own wavefronts split K
    ops.gemm_skinny(a, w, None, many)
    resid = torch.randn(20, N, device=DEV)
    for M in (1, 4, 5, 8, 9, 16):
        out, acc = torch.empty(M, N, dtype=torch.float32, device=DEV), resid[:M].clone()
        ops.gemm_skinny(a[:M], packed, None, out)
        # 32-bit sums of K products of about K ** -0.5: the sum of their magnitudes is below 2 K ** 0.5, each addition rounds by 6e-8 of
        # a partial sum, in chains of at most K / 4
        assert (out - exact[:M]).abs().max() < 6e-8 * 2 * K ** 0.5 + 6e-8 * exact.abs().max() * 8
        wide = torch.randn(M, K + 24, device=DEV).to(BF)
        wide[:, :K] = a[:M]
        again = torch.empty(M, N, dtype=torch.float32, device=DEV)
        ops.gemm_skinny(wide[:, :K], w, None, again)
        assert torch.equal(out, again) and torch.equal(out, many[:M])
        ops.gemm_skinny(a[:M], packed, None, None, accum=acc)
        assert torch.equal(acc, resid[:M] + out.to(BF).float())


@pytest.mark.parametrize("M", [3, 7, 12])
@pytest.mark.parametrize("N", [896, 1536])
def test_what_is_no_number_stays_with_its_token_and_its_row(ops, M, N):
    K = 4864
    torch.manual_seed(M)
    a = torch.randn(M, K, device=DEV).to(BF)
    w = (torch.randn(N, K, device=DEV) * 0.02).to(BF)
    a[1, 3001], w[5, 77], w[6, 4863] = float("inf"), float("nan"), float("-inf")
    want = a.double() @ w.double().T
    out = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops.gemm_skinny(a, ops.pack_weight(w, ops.skinny_strip_rows(N, K)), None, out)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    assert out[:, 5].isnan().all() and out[0].isfinite().sum() == N - 2


@pytest.mark.parametrize("norm32", [False, True])
@pytest.mark.parametrize("M,K,I", [(1, 8, 16), (4, 1024, 4872), (5, 1032, 4872), (8, 904, 12296), (9, 520, 64), (2, 2040, 8200)])
def test_gate_up_behind_its_norm_at_the_edges_of_its_rounds(ops, M, K, I, norm32):
    """Rows that one round of loads covers and not, units in one and several rounds of two, norm weights of either type."""
    torch.manual_seed(K)
    resid = torch.randn(M, K, device=DEV) * 2
    nw = torch.rand(K, device=DEV) + 0.5
    nw = nw if norm32 else nw.to(BF)
    w = (torch.randn(2 * I, K, device=DEV) * K ** -0.5).to(BF)
    x = resid.double()
    n = (x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)).to(BF).double()
    x = (nw.double() * n).to(BF).double()
    gate, up = (x @ w.double().T).chunk(2, -1)
    want = torch.nn.functional.silu(gate) * up
    out = torch.empty(M, I, dtype=BF, device=DEV)
    ops.fused_norm_gate_up_silu(resid, nw, 1e-6, ops.pack_weight(w, 16, [I, I]), out)
    # gate, up and the result are rounded to 8 bits, and an element of x may round the other way
    assert (out.double() - want).abs().max() < 3 * 2.0 ** -8 * want.abs().max()
    assert ((out.double() - want).norm() / want.norm()) < 2.0 ** -7
