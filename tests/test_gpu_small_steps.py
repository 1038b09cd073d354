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


@pytest.mark.parametrize("N", [388, 1540, 3076])                     # strips of 4, 8 and 16 rows
@pytest.mark.parametrize("K", [456, 640, 776, 1000, 1160, 1416, 2040, 2056, 2824, 3080, 3592, 4104, 4616, 5640, 6152, 12296])
def test_every_depth_of_a_round(ops, N, K):
    """Ranges of 4 to 16 k-steps in four parts and of 5 to 25 in sixteen, one to three rounds of each depth there is a kernel for."""
    torch.manual_seed(K + N)
    a = torch.randn(17, K, device=DEV).to(BF)
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).to(BF)
    packed = ops.pack_weight(w, ops.skinny_strip_rows(N, K))
    many = torch.empty(17, N, dtype=torch.float32, device=DEV)       # the kernel of more than 16 rows
    ops.gemm_skinny(a, w, None, many)
    assert (many - a.double() @ w.double().T).abs().max() < 1e-4
    for M in (3, 8, 16):
        for matrix in (packed, w):
            out = torch.empty(M, N, dtype=torch.float32, device=DEV)
            ops.gemm_skinny(a[:M], matrix, None, out)
            assert torch.equal(out, many[:M]), (M, matrix is w)


@pytest.mark.parametrize("N,K", [(897, 4856), (1540, 2056), (3076, 2056), (3076, 904), (4100, 2056)])
def test_every_number_of_few_tokens(ops, N, K):
    """Activations whose pieces change lanes behind their loads and those that do not, on both sides of each line between them: a token's bits are one."""
    torch.manual_seed(K + N)
    a = torch.randn(16, K, device=DEV).to(BF)
    packed = ops.pack_weight((torch.randn(N, K, device=DEV) * K ** -0.5).to(BF), ops.skinny_strip_rows(N, K))
    outs = [ops.gemm_skinny(a[:M], packed, None, torch.full((M, N), float("nan"), device=DEV)) for M in range(1, 17)]
    for M, out in enumerate(outs, 1):
        assert torch.equal(out, outs[15][:M]), M


@pytest.mark.parametrize("N", [388, 1540, 3076, 4100])
@pytest.mark.parametrize("K", [456, 512, 904, 2040, 2056, 2824, 3592, 4616, 6152, 12296])
def test_rows_of_whole_pieces_have_the_bits_of_others(ops, N, K):
    """Activations change lanes where their rows lie in whole pieces of 64 bytes, at every depth of a round; the others, and those that begin
    beside a piece, do not."""
    torch.manual_seed(K + N)
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).to(BF)
    packed = ops.pack_weight(w, ops.skinny_strip_rows(N, K))
    room = torch.randn(17, -(-K // 32) * 32 + 32, device=DEV).to(BF)
    room[:, K:] = float("nan")                                       # what lies behind a row is nobody's
    rows, beside = room[:16, :K], torch.empty_like(room)[:16, 8:8 + K]
    beside.copy_(rows)
    assert rows.stride(0) % 32 == 0 and rows.data_ptr() % 64 == 0 and beside.data_ptr() % 64
    for M in range(1, 17):
        outs = [ops.gemm_skinny(x[:M], packed, None, torch.full((M, N), float("nan"), device=DEV)) for x in (rows, beside, rows[:M].contiguous())]
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), M
    # products of two bfloat16 are exact in 32 bits: what is left is one rounding of at most the sum of the magnitudes an addition
    assert ((outs[0].double() - rows.double() @ w.double().T).abs() <= K * 2.0 ** -24 * (rows.double().abs() @ w.double().abs().T)).all()


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


@pytest.mark.parametrize("norm32", [False, True])
@pytest.mark.parametrize("K", [136, 904, 1032, 2040])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_gate_up_of_a_token_has_the_same_bits_whatever_the_matrix_height(ops, M, K, norm32):
    """A block with one unit and one with two at a time (narrow and wide results) add a row's squares in the same order. Rows of ties: their
    elements times the norm's factor lie within a last bit of the middle of two bfloat16 numbers, so the factor's last bit shows."""
    g = torch.Generator(device=DEV).manual_seed(M + K)
    narrow, wide = 64, 4872
    w = (torch.randn(2, wide, K, generator=g, device=DEV) * K ** -0.5).to(BF)
    few = ops.pack_weight(w[:, :narrow].reshape(2 * narrow, K), 16, [narrow, narrow])
    many = ops.pack_weight(w.view(2 * wide, K), 16, [wide, wide])
    nw = torch.rand(K, generator=g, device=DEV) + 0.5
    nw = nw if norm32 else nw.to(BF)
    for _ in range(8):
        resid = 0.5 + (2 * torch.randint(0, 128, (M, K), generator=g, device=DEV).double() + 1) / 512
        resid[:, 5] = (K * (1 - 1e-6) - (resid * resid).sum(-1) + resid[:, 5] ** 2).sqrt()         # the factor is 1
        resid = resid.float()
        a, b = torch.empty(M, narrow, dtype=BF, device=DEV), torch.empty(M, wide, dtype=BF, device=DEV)
        ops.fused_norm_gate_up_silu(resid, nw, 1e-6, few, a)
        ops.fused_norm_gate_up_silu(resid, nw, 1e-6, many, b)
        assert torch.equal(a, b[:, :narrow])


@pytest.mark.parametrize("bias_dtype", [torch.float32, BF, None])
@pytest.mark.parametrize("M,K,H,KVH,D", [(9, 8, 2, 1, 32), (16, 1000, 14, 2, 64), (17, 1024, 3, 1, 64), (33, 904, 66, 1, 128), (48, 776, 4, 2, 96), (64, 936, 14, 2, 64),
                                         (49, 40, 70, 1, 128)])
def test_qkv_of_9_to_64_rows_at_the_edges_of_what_a_wavefront_brings(ops, M, K, H, KVH, D, bias_dtype):
    """Rows that end inside a piece of 64 lanes and inside a k-step, ranges of k that some wavefronts do not have, one unit a block and more
    (more units than CUs), a token whose numbers are none."""
    torch.manual_seed(M + K)
    N = (H + 2 * KVH) * D
    x, w = torch.randn(M, K, device=DEV).to(BF), (torch.randn(N, K, device=DEV) * K ** -0.5).to(BF)
    x[3, K - 1] = float("inf")
    b = None if bias_dtype is None else torch.randn(N, device=DEV).to(bias_dtype)
    angle = torch.rand(40, D // 2, device=DEV) * 6
    positions = torch.randint(0, 40, (M,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(5 * 16)[:M].to(torch.int32).to(DEV)
    kp, vp = torch.zeros(5, 16, KVH, D, dtype=BF, device=DEV), torch.zeros(5, KVH, D, 16, dtype=BF, device=DEV)
    out = torch.empty(M, H * D, dtype=BF, device=DEV)
    assert ops.panel_fits(M, K)
    ops.panel_qkv_rope(x, ops.pack_weight(w, ops.fused_qkv_strip_rows(H, KVH, D, K)), b, out, H, KVH, D, angle.cos(), angle.sin(), positions, slots, kp, vp)
    y = x.double() @ w.double().T + (0 if b is None else b.double())
    y = y.to(BF).double().view(M, H + 2 * KVH, D)
    c, s = angle.double().cos()[positions.long()][:, None], angle.double().sin()[positions.long()][:, None]
    lo, hi = y[:, :H + KVH].chunk(2, -1)
    turned = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    at = slots.long()
    got = torch.cat([out.view(M, H, D), kp.view(-1, KVH, D)[at], vp.permute(0, 3, 1, 2).reshape(-1, KVH, D)[at]], 1).double()
    want = torch.cat([turned, y[:, H + KVH:]], 1)
    rest = [t for t in range(M) if t != 3]
    assert not got[3, :H + KVH].isfinite().any() and got[rest].isfinite().all()
    # a projection may round the other way (2^-7 of itself, in both terms of a rotation), and the result is rounded (2^-8)
    scale = torch.cat([torch.cat([lo.abs() + hi.abs()] * 2, -1), y[:, H + KVH:].abs()], 1)[rest]
    assert ((got[rest] - want[rest]).abs() <= 2.0 ** -6 * scale + 1e-5).all()


@pytest.mark.parametrize("norm32", [False, True])
@pytest.mark.parametrize("M,K,H,KVH", [(1, 896, 14, 2), (8, 896, 4, 2), (4, 904, 4, 2), (16, 1544, 4, 2), (3, 2048, 4, 2), (2, 3584, 28, 4)])
def test_an_infinite_norm_weight_gives_infinite_values(ops, M, K, H, KVH, norm32):
    """x has an infinity in one channel: it meets that channel's column of the matrix and nothing else, least of all the zeros that stand
    for k-steps a wavefront does not have."""
    D = 64
    torch.manual_seed(K)
    N = (H + 2 * KVH) * D
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).to(BF)
    packed = ops.pack_weight(w, ops.fused_qkv_strip_rows(H, KVH, D, K))
    angle = torch.rand(40, D // 2, device=DEV)
    positions = torch.arange(M, dtype=torch.int32, device=DEV)
    for at in (3, 37, K // 4, K // 2 + 5, K - 1):
        resid, nw = torch.randn(M, K, device=DEV) + 0.1, torch.rand(K, device=DEV) + 0.5
        nw[at] = float("inf")
        nw = nw if norm32 else nw.to(BF)
        kp, vp = torch.zeros(1, 16, KVH, D, dtype=BF, device=DEV), torch.zeros(1, KVH, D, 16, dtype=BF, device=DEV)
        out = torch.empty(M, H * D, dtype=BF, device=DEV)
        ops.fused_norm_qkv_rope(resid, nw, 1e-6, packed, None, out, H, KVH, D, angle.cos(), angle.sin(), positions, positions, kp, vp)
        x = (resid[:, at:at + 1].sign() * float("inf")).double()
        want = (x @ w[-KVH * D:, at:at + 1].double().T).view(M, KVH, D)
        assert torch.equal(vp[0, :, :, :M].permute(2, 0, 1).double(), want), at
