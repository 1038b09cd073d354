"""Attention of prompt portions over a shared latent with keys and values per head (csrc/attention_heads.hip) against 64 bits: portions at
the edges of blocks of 64 queries and keys, behind cached tokens, in windows, several of them, beside single tokens; a gate, a sink,
either pairing of the rotation."""
from __future__ import annotations

import types

import pytest
import torch

from tokenmill_amd.parts.attention_latent import LatentAttention
from tokenmill_amd.parts.base import GroupStep, StepContext
from tokenmill_amd.parts.position import RotaryEmbedding

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16

SIZES = {"2k": (4, 128, 64, 128, 256, 512), "1k": (3, 64, 32, 64, 128, 256)}          # heads, Dn, Dr, Dv, Lq, Lk
# (cached tokens, tokens) of each portion, lengths of single tokens' contexts, window
STEPS = [([(0, 2)], [], None), ([(0, 64)], [], 64), ([(0, 65)], [], 30), ([(37, 150)], [], None), ([(300, 129)], [], 100),
         ([(0, 200), (90, 33), (64, 64)], [], 70), ([(10, 100)], [1, 77, 300], 128), ([(0, 500)], [5], 1000)]


def _part(size, sink, gate, half):
    H, Dn, Dr, Dv, Lq, Lk = SIZES[size]
    hidden = 256
    rot = RotaryEmbedding(Dr, 1024, 10000.0, interleaved=not half)
    return LatentAttention(hidden, H, Dn, Dr, Dv, Lq, Lk, 0.09, 1e-5, rotary=rot, output_gate=gate, sink=sink), hidden


def _step(portions, singles, tables, page, window):
    entries = list(portions) + [(c - 1, 1) for c in singles]
    T, S = sum(n for _, n in entries), len(entries)
    pos = torch.cat([torch.arange(a, a + n) for a, n in entries]).int()
    seq = torch.cat([torch.full((n,), s) for s, (_, n) in enumerate(entries)]).int()
    slots = torch.tensor([int(tables[s, p // page]) * page + p % page for s, p in zip(seq.tolist(), pos.tolist())], dtype=torch.int32)
    tiles, row = [], 0
    for s, (a, n) in enumerate(portions):
        tiles += [(s, row + i, min(16, n - i), a + i) for i in range(0, n, 16)]
        row += n
    d = dict(dtype=torch.int32, device=DEV)
    cu = [0]
    for _, n in entries:
        cu.append(cu[-1] + n)
    return StepContext(num_tokens=T, num_seqs=S, token_ids=torch.zeros(T, **d), positions=pos.to(DEV), seq_of_token=seq.to(DEV),
                       cu_q_lens=torch.tensor(cu, **d), context_lens=torch.tensor([a + n for a, n in entries], **d), state_slots=torch.zeros(S, **d),
                       logit_rows=torch.zeros(1, **d), groups=[GroupStep(block_tables=tables.to(DEV), slot_mapping=slots.to(DEV))],
                       q_lens=[n for _, n in entries], start_positions=[a for a, _ in entries], max_q_len=max(n for _, n in entries),
                       max_context_len=max(a + n for a, n in entries), num_decode=len(singles), max_decode_context=max(singles, default=0),
                       prefill_tiles=torch.tensor(tiles, **d).view(-1, 4), portions_known=True)


@pytest.mark.parametrize("size", list(SIZES))
@pytest.mark.parametrize("case", range(len(STEPS)))
@pytest.mark.parametrize("page,sink,gate,half", [(16, False, True, False), (8, True, False, True)])
def test_portions_by_heads(size, case, page, sink, gate, half, monkeypatch):
    from tokenmill_amd.hip import ops
    from tokenmill_amd.parts import attention_latent

    monkeypatch.setattr(attention_latent, "HEADS_SEEN_ROWS", 0)     # few rows too
    portions, singles, window = STEPS[case]
    H, Dn, Dr, Dv, Lq, Lk = SIZES[size]
    torch.manual_seed(case)
    part, hidden = _part(size, sink, gate, half)
    part.window = window
    g = torch.Generator().manual_seed(case)
    tensors = {}
    for name, spec in part.tensor_specs("m.").items():
        t = torch.randn(spec.shape, generator=g) * (0.06 if len(spec.shape) == 2 else 0.3) + (1.0 if spec.init == "ones" else 0.0)
        tensors[name] = t.to(BF).to(DEV)
    part.load(tensors, "m.")
    part.prepare(False)
    entries = list(portions) + [(c - 1, 1) for c in singles]
    pages = [-(-(a + n) // page) for a, n in entries]
    order = torch.randperm(sum(pages) + 3, generator=g)
    tables = torch.zeros(len(entries), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        tables[s, :n] = order[at:at + n].int()
        at += n
    pool = torch.full((len(order), page, 1, Lk + Dr), float("nan"), dtype=BF, device=DEV)       # what nobody wrote is never looked at
    cached = [torch.randn(a, Lk + Dr, generator=g).to(BF).to(DEV) for a, _ in entries]
    for s, (a, _) in enumerate(entries):
        for p in range(a):
            pool[int(tables[s, p // page]), p % page, 0] = cached[s][p]
    cache = types.SimpleNamespace(k=pool, v=None, group=0, write=True)
    step = _step(portions, singles, tables, page, window)
    x = torch.randn(step.num_tokens, hidden, generator=g).to(BF).to(DEV)
    taken = []
    real = ops.attn_heads
    monkeypatch.setattr(ops, "attn_heads", lambda *a, **k: taken.append(1) or real(*a, **k))
    got = part.forward(x, step, cache)
    assert taken
    step.portions_known = False                                     # the same over the latent itself
    other = part.forward(x, step, cache)
    assert len(taken) == 1

    # 64 bits from what the cache holds now
    low = part.down.forward(x, out_dtype=torch.float32).double()
    cq = low[:, :Lq]
    cq = (cq * torch.rsqrt((cq * cq).mean(-1, keepdim=True) + 1e-5) * part.q_norm.double()).to(BF).double()
    q = (cq @ part.uq.weight.double().T).view(-1, H, Dn + Dr)
    cos, sin = (t.double()[step.positions.long()][:, None] for t in (part.rotary.cos, part.rotary.sin))
    r = q[..., Dn:]
    a, b = (r[..., :Dr // 2], r[..., Dr // 2:]) if half else (r[..., 0::2], r[..., 1::2])
    turned = torch.empty_like(r)
    if half:
        turned[..., :Dr // 2], turned[..., Dr // 2:] = a * cos - b * sin, b * cos + a * sin
    else:
        turned[..., 0::2], turned[..., 1::2] = a * cos - b * sin, b * cos + a * sin
    q = torch.cat([q[..., :Dn], turned], -1)
    want = torch.empty(step.num_tokens, H * Dv, dtype=torch.float64, device=DEV)
    row = 0
    for s, (start, n) in enumerate(entries):
        rows = torch.stack([pool[int(tables[s, p // page]), p % page, 0] for p in range(start + n)]).double()
        k = torch.einsum("jc,hdc->hjd", rows[:, :Lk], part.uk.double())
        k = torch.cat([k, rows[None, :, Lk:].expand(H, -1, -1)], -1)
        v = torch.einsum("jc,hdc->hjd", rows[:, :Lk], part.uv_nt.double())
        sc = torch.einsum("thd,hjd->htj", q[row:row + n], k) * part.scale
        far = torch.arange(start, start + n, device=DEV)[:, None] - torch.arange(start + n, device=DEV)
        sc.masked_fill_((far < 0) | (far >= (window or 1 << 30)), float("-inf"))
        if sink:
            sc = torch.cat([sc, part.sink.double()[:, None, None].expand(H, n, 1)], -1)
        p = torch.softmax(sc, -1)[..., :start + n]
        o = torch.einsum("htj,hjd->thd", p, v)
        if gate:
            o = o * torch.sigmoid(low[row:row + n, part.gate_at:part.gate_at + H])[..., None]
        want[row:row + n] = o.flatten(1)
        row += n
    want = want @ part.o.weight.double().T
    err, err_latent = ((t.double() - want).norm() / want.norm() for t in (got, other))
    # keys, values, weights, results and queries are rounded to 8 bits on the way: 2 ** -9 each at most, of which the sums keep less
    assert err < 2.0 ** -7 and err < 1.25 * err_latent + 1e-3, (float(err), float(err_latent))
    assert (got.double() - want).abs().max() < 2.0 ** -5 * want.abs().max()


def _attended(size, window, entries, n_singles, taken, monkeypatch):
    """The attention's result for entries (seed, cached tokens, tokens), the last ``n_singles`` single tokens: row by row the same inputs for
    the same seed, whatever stands beside it (the products in front, which may round by the step's size, are given)."""
    from tokenmill_amd.hip import ops

    H, Dn, Dr, Dv, Lq, Lk = SIZES[size]
    part, hidden = _part(size, False, True, False)
    part.window, page = window, 16
    part.rotary.max_positions = 10000
    g = torch.Generator().manual_seed(1)
    part.load({name: (torch.randn(spec.shape, generator=g) * 0.06 + (1.0 if spec.init == "ones" else 0.0)).to(BF).to(DEV)
               for name, spec in part.tensor_specs("m.").items()}, "m.")
    pages = [-(-(a + n) // page) for _, a, n in entries]
    tables = torch.zeros(len(entries), max(pages), dtype=torch.int32)
    for s, n in enumerate(pages):
        tables[s, :n] = torch.arange(sum(pages[:s]), sum(pages[:s + 1]))
    pool = torch.zeros(sum(pages), page, 1, Lk + Dr, dtype=BF, device=DEV)
    low, q = [], []
    for s, (seed, a, n) in enumerate(entries):
        g = torch.Generator().manual_seed(seed)
        pool.view(-1, Lk + Dr)[sum(pages[:s]) * page:][:a] = torch.randn(a, Lk + Dr, generator=g).to(BF).to(DEV)
        low.append(torch.randn(n, Lq + Lk + Dr + H, generator=g).to(DEV))
        q.append(torch.randn(n, H * (Dn + Dr), generator=g).to(BF).to(DEV))
    low, q = torch.cat(low), torch.cat(q)
    free = dict(cost=lambda rows, out_bytes=2: (0, 0), weight=part.uq.weight)
    part.down = types.SimpleNamespace(forward=lambda x, out_dtype: low, **free)
    part.uq = types.SimpleNamespace(forward=lambda cq: q, **free)
    part.o = types.SimpleNamespace(forward=lambda out: out, **free)
    split = len(entries) - n_singles
    step = _step([(a, n) for _, a, n in entries[:split]], [a + 1 for _, a, _ in entries[split:]], tables, page, window)
    real = ops.attn_heads
    with monkeypatch.context() as m:
        m.setattr(ops, "attn_heads", lambda *a, **k: taken.append(a[5].shape[0]) or real(*a, **k))
        out = part.forward(torch.zeros(step.num_tokens, hidden, dtype=BF, device=DEV), step, types.SimpleNamespace(k=pool, v=None, group=0, write=True))
    return list(out.split([n for _, _, n in entries]))


@pytest.mark.parametrize("size", list(SIZES))
@pytest.mark.parametrize("window", [None, 500])
def test_a_portions_bits_do_not_depend_on_its_neighbours(size, window, monkeypatch):
    """Portions of either form, several of each, between each other and beside single tokens, and more rows than pass at once: each alone
    gives what it gives in the step."""
    from tokenmill_amd.parts import attention_latent

    monkeypatch.setattr(attention_latent, "HEADS_MOST_ROWS", 1200)
    entries = [(11, 0, 100), (12, 0, 400), (14, 20, 33), (13, 700, 3), (15, 300, 200), (16, 0, 500), (17, 600, 1), (18, 40, 1), (19, 1300, 1)]
    taken: list[int] = []
    together = _attended(size, window, entries, 3, taken, monkeypatch)
    # blocks of 64 queries: of the 400 and the 3 tokens (448 and 704 rows, 512 in the window), then of the 200 and the 500 (512 rows each)
    assert taken == [7 + 1, 4 + 8]
    for i, (entry, got) in enumerate(zip(entries, together)):
        alone, = _attended(size, window, [entry], int(i >= 6), [], monkeypatch)
        assert torch.equal(got, alone), i


@pytest.mark.parametrize("cached,tokens,heads", [(0, 383, False), (0, 384, True), (382, 2, True), (381, 2, False), (4000, 2, True), (8190, 2, True),
                                                 (8191, 2, False)])
def test_a_portions_own_rows_choose_its_form(cached, tokens, heads, monkeypatch):
    taken: list[int] = []
    _attended("1k", None, [(5, cached, tokens)], 0, taken, monkeypatch)
    assert bool(taken) == heads


@pytest.mark.parametrize("entries,n_singles", [([(1, 0, 100)], 0), ([(1, 0, 100), (2, 0, 400), (3, 20, 30), (4, 500, 1)], 1)])
def test_a_profile_counts_a_layer_once(entries, n_singles, monkeypatch):
    from tokenmill_amd import profiling

    counted = []
    real = LatentAttention.cost
    monkeypatch.setattr(LatentAttention, "cost", lambda self, label, step, rows: counted.append((label, rows)) or real(self, label, step, rows))
    with profiling.collect(trace=False):
        _attended("1k", None, entries, n_singles, [], monkeypatch)
    T = sum(n for _, _, n in entries)
    assert sorted(counted) == [("attention", T), ("o_proj", T), ("qkv", T)]
