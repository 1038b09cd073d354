"""Top-k beside the bound that the wavefronts' maxima give: as many entries kept as there are shares, one more and one less;
the largest entries all in one share; shares with no number in them."""
import pytest
import torch

from plain import qwen2_plain as P

pytestmark = pytest.mark.gpu
V = 4 * 4096 + 616                                              # five chunks of four shares


def tokens(logits, k, p, us):
    from tokenmill_amd.hip import ops
    R = logits.shape[0]
    out = torch.empty(R, dtype=torch.int32, device="cuda")
    full = lambda x: torch.full((R,), x, device="cuda", dtype=torch.int32 if isinstance(x, int) else torch.float32)   # noqa: E731
    ops.sample_rows(logits.cuda(), full(0.9), full(k), full(p), torch.tensor(us, dtype=torch.float32, device="cuda"), out)
    return out.cpu().tolist()


@pytest.mark.parametrize("p", [1.0, 0.9])
@pytest.mark.parametrize("k", [2, 19, 20, 21, 3000])
@pytest.mark.parametrize("where", ["spread", "one share", "steps", "not numbers"])
def test_top_k_at_the_bound(where, k, p):
    R = 24
    g = torch.Generator().manual_seed(k)
    logits = torch.randn(R, V, generator=g) * 2
    if where == "one share":                                    # the first wavefront's entries of the second chunk: lanes 0 to 63 of every 256
        chunk = -(-V // 5)
        at = torch.cat([torch.arange(chunk + 256 * j, chunk + 256 * j + 64) for j in range(8)])
        logits[:, at] += 12
    elif where == "steps":                                      # ties everywhere
        logits = (logits * 2).round() / 2
    us = [P.uniform_from_counter(3, r) for r in range(R)]
    want, margins = zip(*[P.sample_token(logits[r], 0.9, k, p, 3, r) for r in range(R)])
    if where == "not numbers":                                  # an entry that is none is as good as one of no weight
        hole = torch.rand(R, V, generator=g) < 0.6
        hole[:, :4096] = True
        want, margins = zip(*[P.sample_token(logits[r].masked_fill(hole[r], float("-inf")), 0.9, k, p, 3, r) for r in range(R)])
        logits = logits.masked_fill(hole, float("nan"))
    got = tokens(logits, k, p, us)
    assert all(a == b or m < 1e-4 for a, b, m in zip(got, want, margins))
    assert sum(a == b for a, b in zip(got, want)) >= R - 2
