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


@pytest.mark.parametrize("k", [2, 50, 244, 245, 246, 980])
def test_top_k_at_the_bound_of_the_widest_rows(k):
    """A million entries have 245 chunks, whose maxima are the keys that the bound is looked up among. Entries of whole steps tie
    by the thousand, and every token is among the k that are kept."""
    R, wide = 4, 1_000_000
    g = torch.Generator().manual_seed(k)
    logits = (torch.randn(R, wide, generator=g) * 3).round() / 4
    logits[1, :900_000] = float("nan")                          # most shares without a number
    logits[2] = logits[2].sort().values                         # the largest all in the last shares
    us = [P.uniform_from_counter(3, r) for r in range(R)]
    kept = torch.zeros(R, wide, dtype=torch.bool)
    for r in range(R):
        kept[r, logits[r].nan_to_num(float("-inf")).sort(descending=True, stable=True).indices[:k]] = True
    for u in (us, [0.0] * R, [1.0 - 2.0 ** -24] * R):
        got = tokens(logits, k, 1.0, u)
        assert all(kept[r, t] for r, t in enumerate(got))
        z = torch.where(kept, logits.double() / 0.9, torch.tensor(float("-inf"), dtype=torch.float64)).softmax(1).cumsum(1)
        for r, t in enumerate(got):                             # the token in whose share of the mass u lies, to 32-bit sums of k weights
            assert (z[r, t - 1] if t else 0.0) - 1e-5 <= u[r] <= z[r, t] + 1e-5


@pytest.mark.parametrize("vocab", [V, 151936, 4097, 1 << 20])
@pytest.mark.parametrize("where", ["spread", "one share", "steps", "level", "not numbers", "small"])
def test_lists_give_the_tokens_of_the_launches_over_all_chunks(where, vocab):
    """Rows with k from 1 to beyond what the bound covers, with and without top-p, greedy ones and ones without top-k among them: through lists,
    where thousands of equal entries do not fit one and unbounded rows have none, and without."""
    from tokenmill_amd.hip import ops
    most = ops.sample_list_k(vocab)
    ks = [2, 7, 20, 50, most // 2, most, 1, 0, most + 1, 4 * most + 9]
    R = 3 * len(ks)
    g = torch.Generator().manual_seed(vocab)
    logits = torch.randn(R, vocab, generator=g) * (0.01 if where == "small" else 2)
    if where == "one share":
        chunk = -(-vocab // (-(-vocab // 4096) if vocab <= 256 * 4096 else 256))
        logits[:, torch.cat([torch.arange(chunk + 256 * j, min(vocab, chunk + 256 * j + 64)) for j in range(8) if chunk + 256 * j < vocab])] += 12
    elif where == "steps":
        logits = (logits * 2).round() / 2
    elif where == "level":
        logits = torch.where(torch.rand(R, vocab, generator=g) < 0.3, 1.5, 0.25)
    elif where == "not numbers":
        logits = logits.masked_fill(torch.rand(R, vocab, generator=g) < 0.6, float("nan"))
    logits = logits.cuda()
    f = lambda x: torch.tensor(x, dtype=torch.float32, device="cuda")       # noqa: E731
    rows = [(ks[r % len(ks)], (1.0, 0.9, 0.5)[r // len(ks)]) for r in range(R)]
    args = (f([0.0 if r == 4 else 0.8 for r in range(R)]), torch.tensor([k for k, _ in rows], dtype=torch.int32, device="cuda"), f([p for _, p in rows]),
            f([(r * 0.137) % 1 for r in range(R)]))
    want, got = (torch.full((R,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    ops.sample_rows(logits, *args, want)
    for _ in range(2):                                                       # (the second call finds what the first left in the scratch memory)
        ops.sample_rows(logits, *args, got, small_top_k=True)
        assert got.tolist() == want.tolist()


TOGETHER = ("few of -inf", "many of -inf", "few of the smallest", "one place of -inf", "a larger place of -inf", "steps in one place", "two steps in one place",
            "half raised", "ascending", "descending", "one level", "one above a level", "infinite", "one place of not numbers")


@pytest.mark.parametrize("vocab", [V, 151936, 4097, 1 << 20])
@pytest.mark.parametrize("where", TOGETHER)
def test_lists_of_rows_whose_large_entries_lie_together(where, vocab):
    """Fewer finite entries than k; a level that fills all shares; more entries above the bound than a list holds, in few shares and in most, with the edge
    of top-k inside equal ones or not: the tokens of the launches over all chunks."""
    from tokenmill_amd.hip import ops
    most = ops.sample_list_k(vocab)
    ks = sorted({2, 7, 20, 50, most // 2, most})
    R = 4 * len(ks)
    g = torch.Generator(device="cuda").manual_seed(vocab)
    x = torch.randn(R, vocab, generator=g, device="cuda") * 2
    place = torch.zeros(vocab, dtype=torch.bool, device="cuda")
    place[vocab // 5:vocab // 5 + (min(900, vocab // 3) if where == "one place of -inf" else min(4000, vocab // 2))] = True
    if where.startswith(("few", "many")):
        kept = torch.rand(R, vocab, generator=g, device="cuda").topk(5 if where.startswith("few") else min(700, vocab // 8), 1).indices
        logits = torch.full_like(x, torch.finfo(torch.float32).min if "smallest" in where else float("-inf")).scatter(1, kept, x.gather(1, kept))
    elif "place of -inf" in where:
        logits = x.masked_fill(~place, float("-inf"))
    elif "steps in" in where:
        logits = ((x * (2 if where.startswith("steps") else 0.1)).round() / 2).masked_fill(~place, -9.0)
    elif where == "half raised":
        logits = x + 30 * (torch.arange(vocab, device="cuda") >= vocab // 2)
    elif where in ("ascending", "descending"):
        logits = (torch.arange(vocab, dtype=torch.float32, device="cuda") * (20 / vocab if where == "ascending" else -20 / vocab)).expand(R, vocab).contiguous()
    elif where == "infinite":
        logits = x.masked_fill(place, float("inf"))
    elif where == "one place of not numbers":
        logits = x.masked_fill(~place, float("nan"))
    else:
        logits = torch.full_like(x, 0.5)
        if where.startswith("one above"):
            logits[:, vocab // 3] = 2.0
    f = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")       # noqa: E731
    k = torch.tensor([ks[r % len(ks)] for r in range(R)], dtype=torch.int32, device="cuda")
    p = f([(1.0, 0.95, 0.5, 1e-4)[r // len(ks)] for r in range(R)])
    for u in (0.0, 0.31, 0.77, 1 - 2.0 ** -24):
        args = (f([0.8] * R), k, p, f([u] * R))
        want, got = (torch.full((R,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
        ops.sample_rows(logits, *args, want)
        ops.sample_rows(logits, *args, got, small_top_k=True)
        assert got.tolist() == want.tolist(), u
