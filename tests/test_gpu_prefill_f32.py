"""The 32-bit attention of prompt portions where its weights' reference moves rarely, often and not at all, and over grids of one to
several rounds of the chip."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from tokenmill_amd.hip import ops as o
    return o


def attend(ops, q, k, v, H, KVH, D, page, scale):
    n = q.shape[0]
    pages = -(-n // page)
    kp, vp = torch.zeros(pages * page, KVH, D, device=DEV), torch.zeros(pages * page, KVH, D, device=DEV)
    kp[:n], vp[:n] = k, v
    tiles = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)
    out = torch.full((n, H * D), 3.0, device=DEV)
    ops.attn_prefill_f32(q.reshape(n, H * D).contiguous(), out, kp.view(pages, page, KVH, D),
                         vp.view(pages, page, KVH, D).permute(0, 2, 3, 1).contiguous(),
                         torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1), tiles, H, KVH, D, scale, 0)
    return out.view(n, H, D)


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("step", [0.0, 0.05, 0.49, 3.0, -0.3, -8.0])     # how much a key's score exceeds the one before it
@pytest.mark.parametrize("n,H", [(17, 1), (300, 14), (300, 30)])
def test_moving_reference(ops, D, step, n, H):
    torch.manual_seed(n + D)
    q, k, v = (torch.randn(n, h, D, device=DEV) for h in (H, 1, 1))
    q[..., 0], k[..., 0] = D ** 0.5, step * torch.arange(n, device=DEV)[:, None]
    got = attend(ops, q, k, v, H, 1, D, 16, D ** -0.5)
    s = torch.einsum("qhd,kd->hqk", q.double().cpu(), k[:, 0].double().cpu()) * D ** -0.5
    top = s.abs().max()
    s = s.masked_fill(torch.ones(n, n).triu(1).bool(), float("-inf"))
    want = torch.einsum("hqk,kd->qhd", s.softmax(-1), v[:, 0].double().cpu())
    # a score of magnitude S is the running sum of D products that round by up to 2^-24 S each, at random (deviation 2^-24 S / 3^0.5):
    # the difference of two scores is off by at most 5 deviations of 2 D of them, 2^-24 S 4.1 D^0.5, and a result by
    # a quarter of that times the distance of two values, below 8; weights and their sums add 2e-6
    bound = 2 ** -24 * top * 4.1 * D ** 0.5 * 2 + 2e-6
    assert (got.cpu() - want).abs().max() < bound


@pytest.mark.parametrize("D,H,n", [(64, 12, 1008), (64, 12, 1024), (64, 64, 190), (96, 8, 1007), (96, 8, 1024), (128, 32, 255), (128, 32, 257), (80, 32, 400)])
def test_a_tokens_bits_do_not_depend_on_the_launch(ops, D, H, n):
    """From two or three blocks a CU on keys and values change lanes behind their loads: the bits of launches with fewer heads, and so fewer blocks."""
    torch.manual_seed(n)
    q, k, v = torch.randn(n, H, D, device=DEV), torch.randn(n, 2, D, device=DEV), torch.randn(n, 2, D, device=DEV)
    full = attend(ops, q, k, v, H, 2, D, 16, D ** -0.5)
    few = attend(ops, q[:, [0, H - 1]], k, v, 2, 2, D, 16, D ** -0.5)
    assert torch.equal(full[:, [0, H - 1]], few)
    s = torch.einsum("qhd,khd->hqk", q[:, [0, H - 1]].double(), k.double()) * D ** -0.5
    want = torch.einsum("hqk,khd->qhd", s.masked_fill(torch.ones(n, n, device=DEV).triu(1).bool(), float("-inf")).softmax(-1), v.double())
    assert (full[:, [0, H - 1]] - want).abs().max() < 2 ** -24 * s.abs().max() * 4.1 * D ** 0.5 * 2 + 2e-6      # (the bound above)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_no_number_reaches_those_that_see_it(ops, bad):
    torch.manual_seed(1)
    n, H, D = 100, 2, 64
    q, k, v = (torch.randn(n, h, D, device=DEV) for h in (H, 1, 1))
    q[..., 0] = q[..., 0].abs() + 1
    k[70, 0, 0] = bad
    got = attend(ops, q, k, v, H, 1, D, 16, D ** -0.5)
    assert got[:70].isfinite().all() and not got[70:].isfinite().any()
    k[70, 0, 0] = float("-inf")                                          # a key of weight zero
    got = attend(ops, q, k, v, H, 1, D, 16, D ** -0.5)
    k[70, 0, 0] = -1e6
    assert torch.equal(got, attend(ops, q, k, v, H, 1, D, 16, D ** -0.5))


def test_weights_over_the_whole_range_of_the_exponential(ops):
    """Token t sees keys of score 0, among them its block's, so that 0 is the weights' reference, and one key (64) of a score of its own from
    -86 up to where the reference would move, whose value alone is not 0: the result is e^s 2^30 / (t + e^s)."""
    D, n, H = 16, 144, 64
    s = torch.linspace(-86.0, 7.9, (n - 80) * H, device=DEV).view(n - 80, H)
    q, k, v = torch.zeros(n, H, D, device=DEV), torch.zeros(n, 1, D, device=DEV), torch.zeros(n, 1, D, device=DEV)
    q[80:, :, 0], k[64, 0, 0], v[64, 0] = s, 1.0, 2.0 ** 30
    got = attend(ops, q, k, v, H, 1, D, 16, 1.0)[80:].double()
    e = s.double().exp()
    want = (e / (torch.arange(80, n, device=DEV)[:, None] + e) * 2.0 ** 30)[..., None]
    units = ((got - want) / want) * 2.0 ** 24                            # of half a last place
    # the exponential instruction is good to a last place (2 units), its argument, below 1/2, is rounded (0.4 units of the result); the sum, its
    # inverse and the product with it round once each (3)
    assert units.abs().max() <= 6
    # no roundings lean one way over a range: a correction of the wrong size or sign does (by up to 8 units at -86)
    for part in units.flatten().chunk(8):
        assert part.mean().abs() <= 0.5, part.mean()


def test_more_tiles_than_one_launch_holds(ops):
    """A table of 2^18 + 300 tiles at 64 heads (more than 2^32 threads), all the same but for the last, and so one with the last alone."""
    H, D = 64, 16
    g = torch.Generator(device=DEV).manual_seed(3)
    q, kp, vp = (torch.randn(*shape, generator=g, device=DEV) for shape in ((2, H * D), (1, 16, 1, D), (1, 1, D, 16)))
    tables = torch.zeros(1, 1, dtype=torch.int32, device=DEV)
    tiles = torch.tensor([[0, 0, 1, 0]], dtype=torch.int32, device=DEV).repeat((1 << 18) + 300, 1)
    tiles[-1] = torch.tensor([0, 1, 1, 1], device=DEV)
    many, few = torch.full_like(q, 5.0), torch.empty_like(q)
    ops.attn_prefill_f32(q, many, kp, vp, tables, tiles, H, 1, D, 0.25, 0)
    ops.attn_prefill_f32(q, few, kp, vp, tables, tiles[-2:].contiguous(), H, 1, D, 0.25, 0)
    assert torch.equal(many, few)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("window,keep,softcap", [(1, 0, 0.0), (16, 0, 0.0), (64, 0, 9.0), (128, 0, 0.0), (129, 0, 0.0), (40, 88, 0.0), (41, 88, 0.0), (20, 33, 9.0)])
def test_windows_on_both_sides_of_a_short_walk(ops, D, window, keep, softcap):
    """Walks without a block ahead (a window and what is kept beside it of at most 128 keys) and with one."""
    n, H, KVH, page = 300, 6, 2, 16
    g = torch.Generator(device=DEV).manual_seed(window + D)
    q = torch.randn(n, H, D, generator=g, device=DEV)
    pages = -(-n // page)
    k, v = torch.randn(pages, page, KVH, D, generator=g, device=DEV), torch.randn(pages, KVH, D, page, generator=g, device=DEV)
    tables = torch.randperm(pages, generator=torch.Generator().manual_seed(D)).int().to(DEV).view(1, -1)
    tiles = torch.tensor([(0, j, min(16, n - j), j) for j in reversed(range(0, n, 16))], dtype=torch.int32, device=DEV)
    out = torch.full((n, H * D), 3.0, device=DEV)
    ops.attn_prefill_f32(q.view(n, H * D), out, k, v, tables, tiles, H, KVH, D, D ** -0.5, window, softcap=softcap, keep=keep)
    keys = k[tables[0].long()].view(-1, KVH, D)[:n].double().repeat_interleave(H // KVH, 1)
    values = v[tables[0].long()].permute(0, 3, 1, 2).reshape(-1, KVH, D)[:n].double().repeat_interleave(H // KVH, 1)
    s = torch.einsum("qhd,khd->hqk", q.double(), keys) * D ** -0.5
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    place = torch.arange(n, device=DEV)
    far = place[:, None] - place
    s = s.masked_fill((far < 0) | ((far >= window) & (place >= keep)), float("-inf"))
    want = torch.einsum("hqk,khd->qhd", s.softmax(-1), values).reshape(n, H * D)
    # scores are sums of D products of unit size (their roundings 2^-24 D^0.5 of some 10), weights and sums of up to 129 values below 6
    assert (out.double() - want).abs().max() < 2.0 ** -24 * (10 * D ** 0.5 + 200)
