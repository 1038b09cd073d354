"""Add + RMSNorm at the widths where a block's threads, or the groups of four numbers that a thread has, change."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.mark.parametrize("dtype", [BF, torch.float32])
@pytest.mark.parametrize("hidden", [4, 256, 512, 516, 1024, 1028, 2052, 4096, 4100, 5120, 8196, 12288, 16384])
def test_what_is_added_and_normed(hidden, dtype):
    from tokenmill_amd.hip import ops

    g = torch.Generator(device=DEV).manual_seed(hidden)
    T, eps = 5, 1e-6
    x, w = torch.randn(T, hidden, generator=g, device=DEV), (torch.rand(hidden, generator=g, device=DEV) + 0.5).to(dtype)
    delta = torch.randn(T, hidden, generator=g, device=DEV).to(dtype)
    rows = torch.tensor([3, 0], dtype=torch.int32, device=DEV)
    for n in (0, -1, 1, 2, 3, 5, 8):                                 # nothing, a tensor, or so many partial sums
        parts = torch.randn(max(n, 1), T, hidden, generator=g, device=DEV) * 0.3
        added = x
        if n > 0:
            total = parts[0].clone()
            for p in parts[1:]:
                total += p
            added = x + total.to(dtype).float()
        elif n < 0:
            added = x + delta.float()
        d = added.double()
        want = w.double() * (d * torch.rsqrt((d * d).mean(-1, keepdim=True) + eps)).to(dtype).double()
        for pick in (None, rows):
            resid, out = x.clone(), torch.empty(2 if pick is not None else T, hidden, dtype=dtype, device=DEV)
            if n > 0:
                ops.add_rmsnorm_parts(resid, parts, w, eps, out, rows=pick)
            else:
                ops.add_rmsnorm(resid, delta if n < 0 else None, w, eps, out, rows=pick)
            assert torch.equal(resid, added if pick is None else x)
            ref = want if pick is None else want[pick.long()]
            # bfloat16: the first rounding may go the other way (a last place, at most 2^-7 of a number), the second is half of one (2^-8);
            # in 32-bit the factor is off by the sum's rounding, at most 2^-24 for each of 16 terms of a thread and 10 of a block's tree,
            # halved by the root
            bound = 1.6 * 2.0 ** -7 if dtype == BF else 20 * 2.0 ** -24
            assert ((out.double() - ref).abs() <= bound * ref.abs() + 1e-30).all(), (n, pick is None)
