"""The 32-bit path's kernels for few rows (csrc/gemv_f32.hip, csrc/attention_decode_f32.hip) against 64-bit computations: rows and
columns that fill no tile, the shortest K, K in parts, contexts at the edges of chunks, windows, kept keys, caps, sinks, gates."""
from __future__ import annotations

import ctypes

import pytest
import torch

from tokenmill_amd.hip.library import library

pytestmark = pytest.mark.gpu
P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


def _ptr(t):
    return P(t.data_ptr() if t is not None else None)


def _stream():
    return P(torch.cuda.current_stream().cuda_stream)


def _operands(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda") * K ** -0.5
    return a, w, a.double() @ w.double().T


# 32-bit sums: a wavefront's chain of K / (4 x 8) additions or fewer and the wavefronts' sums, each rounding a sum of at most about 5
def _bound(K):
    return 2.0 ** -24 * 5 * (16 + K ** 0.5)


@pytest.mark.parametrize("N,K", [(4, 16), (20, 48), (896, 896), (1152, 4864), (8200, 896), (9000, 112)])
@pytest.mark.parametrize("M", [1, 7, 16])
def test_products_plain_and_in_parts(M, N, K):
    lib = library()
    a, w, ref = _operands(M, N, K, M + N + K)
    bias = torch.randn(N, device="cuda")
    out = torch.full((M, N), float("nan"), device="cuda")
    assert lib.tm_gemv_f32_mfma(_ptr(a), I(K), _ptr(w), _ptr(bias), _ptr(out), I(N), I(M), I(N), I(K), _stream()) == 0
    assert (out.double() - ref - bias.double()).abs().max() <= _bound(K)
    parts = lib.tm_gemv_f32_parts(N, K)
    sums = torch.full((parts, M, N), float("nan"), device="cuda")
    assert lib.tm_gemv_f32_mfma_split(_ptr(a), I(K), _ptr(w), _ptr(sums), I(M), I(N), I(K), _stream()) == 0
    assert (sums.double().sum(0) - ref).abs().max() <= _bound(K)


@pytest.mark.parametrize("N,K", [(20, 48), (36, 16 * 57), (896, 896), (40, 16 * 431), (2048, 5632), (8200, 912), (9000, 112)])
def test_a_row_is_the_same_whatever_rows_are_beside_it(N, K):
    """Odd numbers of steps, runs of one group and of several with a rest, one tile and two; up to four, up to eight and more rows."""
    lib = library()
    a, w, ref = _operands(16, N, K, N + K)

    def product(rows):
        out = torch.full((rows, N), float("nan"), device="cuda")
        assert lib.tm_gemv_f32_mfma(_ptr(a), I(K), _ptr(w), _ptr(None), _ptr(out), I(N), I(rows), I(N), I(K), _stream()) == 0
        return out

    most = product(16)
    assert (most.double() - ref).abs().max() <= _bound(K)
    for rows in (1, 2, 4, 5, 8, 9, 15):
        assert torch.equal(product(rows), most[:rows]), rows


@pytest.mark.parametrize("N,K", [(3580, 16 * 97), (3584, 16 * 105), (4092, 16 * 112), (3568, 16 * 97), (24000, 384), (2100, 16 * 49)])
def test_a_row_is_the_same_where_the_blocks_nearly_fill_the_chip(N, K):
    """From 224 blocks on two groups at a time for any rows, with a rest of every length; the shortest lines; a step of a pair that is not there."""
    test_a_row_is_the_same_whatever_rows_are_beside_it(N, K)


@pytest.mark.parametrize("N,K", [(3584, 16 * 98), (4092, 896), (4092, 1536), (4092, 1792), (6144, 768), (6144, 896), (6144, 960), (9728, 896), (32800, 896), (16384, 1040),
                                 (1536, 160), (1536, 272), (1536, 528), (8200, 272)])
def test_a_row_is_the_same_in_either_order_of_the_lanes(N, K):
    """Sizes at which the number of rows says whether neighbouring lanes load side by side, and sizes whose rows are half a line more than whole ones."""
    test_a_row_is_the_same_whatever_rows_are_beside_it(N, K)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("K,small,large", [(912, 1868, 1872), (1440, 1180, 1184), (6896, 244, 248), (448, 3800, 3808), (400, 4256, 4260)])
def test_whole_lines_and_a_load_a_step_have_the_same_bits(K, small, large, M):
    """Matrices of 6.5 MB and less: odd numbers of steps, one, two and three groups a wavefront, four and eight wavefronts, K in parts."""
    lib = library()
    a, w, ref = _operands(M, large, K, K)
    outs, parts, gates = [], [], []
    for N in (small, large):
        out = torch.full((M, N), float("nan"), device="cuda")
        assert lib.tm_gemv_f32_mfma(_ptr(a), I(K), _ptr(w), _ptr(None), _ptr(out), I(N), I(M), I(N), I(K), _stream()) == 0
        sums = torch.full((lib.tm_gemv_f32_parts(N, K), M, N), float("nan"), device="cuda")
        assert lib.tm_gemv_f32_mfma_split(_ptr(a), I(K), _ptr(w), _ptr(sums), I(M), I(N), I(K), _stream()) == 0
        n = N // 8 * 4
        both = torch.cat([w[:n], w[large - n:]])                # (up: the last rows, of which the smaller has the end)
        act = torch.full((M, n), float("nan"), device="cuda")
        assert lib.tm_gemv_f32_gate_up_silu(_ptr(a), I(K), _ptr(both), _ptr(act), I(M), I(n), I(K), _stream()) == 0
        want = torch.nn.functional.silu(ref[:, :n]) * ref[:, large - n:]
        assert ((act.double() - want).abs() <= _bound(K) * (1.1 * ref[:, large - n:].abs() + ref[:, :n].abs() + 1) + 2.0 ** -20 * want.abs()).all()
        assert (out.double() - ref[:, :N]).abs().max() <= _bound(K)
        outs.append(out[:, :small]), parts.append(sums[:, :, :small])
    assert torch.equal(*outs) and parts[0].shape == parts[1].shape and torch.equal(*parts)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("H,more,KVH,D,K", [(14, 28, 2, 64, 896), (5, 9, 1, 128, 1456)])
def test_qkv_by_whole_lines_has_the_bits_of_a_load_a_step(H, more, KVH, D, K, M):
    """The same query heads with so many beside them that the matrix is read by whole lines."""
    a, w, _ = _operands(M, (more + 2 * KVH) * D, K, H)
    bias = torch.randn((more + 2 * KVH) * D, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    angle = torch.rand(300, D // 2, generator=torch.Generator(device="cuda").manual_seed(2), device="cuda") * 6.28
    cos, sin, pos = angle.cos(), angle.sin(), torch.arange(M, device="cuda", dtype=torch.int32) * 7
    got = []
    for heads in (H, more):
        skip = (more - heads) * D
        rows = torch.cat([torch.arange(heads * D), torch.arange(heads * D + skip, w.shape[0])]).cuda()
        ww, bb = w[rows].contiguous(), bias[rows].contiguous()
        q, k, v = torch.empty(M, heads * D, device="cuda"), torch.zeros(2, 16, KVH, D, device="cuda"), torch.zeros(2, KVH, D, 16, device="cuda")
        slots = torch.arange(M, device="cuda", dtype=torch.int32)
        assert library().tm_gemv_f32_qkv_rope(_ptr(a), I(K), _ptr(ww), _ptr(bb), _ptr(q), I(M), I(K), I(heads), I(KVH), I(D), _ptr(cos), _ptr(sin), _ptr(pos),
                                              _ptr(slots), _ptr(k), _ptr(v), I(16), _stream()) == 0
        got.append((q[:, :H * D], k, v))
    assert 4 * K * (H + 2 * KVH) * D < 6656 * 1024 <= 4 * K * (more + 2 * KVH) * D
    assert all(torch.equal(x, y) for x, y in zip(*got))


def test_a_long_k_is_split():
    assert library().tm_gemv_f32_parts(896, 4864) == 4 and library().tm_gemv_f32_parts(896, 896) == 1


@pytest.mark.parametrize("n,K", [(4, 16), (36, 64), (4864, 896)])
@pytest.mark.parametrize("M", [1, 16])
def test_gate_up_silu(M, n, K):
    a, w, ref = _operands(M, 2 * n, K, M + n)
    out = torch.full((M, n), float("nan"), device="cuda")
    assert library().tm_gemv_f32_gate_up_silu(_ptr(a), I(K), _ptr(w), _ptr(out), I(M), I(n), I(K), _stream()) == 0
    gate, up = ref.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    assert ((out.double() - want).abs() <= _bound(K) * (1.1 * up.abs() + gate.abs() + 1) + 2.0 ** -20 * want.abs()).all()


@pytest.mark.parametrize("M,H,KVH,D,K", [(1, 14, 2, 64, 896), (16, 3, 1, 128, 64), (5, 4, 2, 32, 16)])
def test_qkv_with_rotation_and_cache_write(M, H, KVH, D, K):
    N, page = (H + 2 * KVH) * D, 16
    a, w, ref = _operands(M, N, K, M + H)
    g = torch.Generator(device="cuda").manual_seed(M)
    bias = torch.randn(N, generator=g, device="cuda")
    angle = torch.rand(300, D // 2, generator=g, device="cuda") * 6.28
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, 300, (M,), generator=g, device="cuda", dtype=torch.int32)
    slots = torch.randperm(3 * page, generator=g, device="cuda")[:M].int()
    slots[1::3] = -1
    q = torch.empty(M, H * D, device="cuda")
    k, v = torch.full((3, page, KVH, D), 7.0, device="cuda"), torch.full((3, KVH, D, page), 7.0, device="cuda")
    assert library().tm_gemv_f32_qkv_rope(_ptr(a), I(K), _ptr(w), _ptr(bias), _ptr(q), I(M), I(K), I(H), I(KVH), I(D), _ptr(cos), _ptr(sin),
                                          _ptr(pos), _ptr(slots), _ptr(k), _ptr(v), I(page), _stream()) == 0
    x = (ref + bias.double()).view(M, H + 2 * KVH, D)
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    c, s = (t.double()[pos.long()][:, None] for t in (cos, sin))
    turned = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    bound = 2 * _bound(K) + 2.0 ** -21
    assert (q.double().view(M, H, D) - turned[:, :H]).abs().max() <= bound
    kept = slots >= 0
    at = slots[kept].long()
    keys, values = k.view(-1, KVH, D), v.permute(0, 3, 1, 2).reshape(-1, KVH, D)
    assert (keys[at].double() - turned[kept, H:H + KVH]).abs().max() <= bound
    assert (values[at].double() - x[kept, H + KVH:]).abs().max() <= bound
    others = torch.ones(3 * page, dtype=torch.bool, device="cuda")
    others[at] = False
    assert (keys[others] == 7).all() and (values[others] == 7).all()


CONTEXTS = [1, 16, 17, 127, 128, 129, 700, 1024, 1500]


@pytest.mark.parametrize("extras", ["plain", "window", "window+keep", "cap+sink+gate"])
@pytest.mark.parametrize("H,KVH,D,page", [(14, 2, 64, 16), (5, 5, 32, 64), (16, 1, 128, 16)])
def test_attention_of_single_tokens(H, KVH, D, page, extras):
    g = torch.Generator(device="cuda").manual_seed(H + D)
    S, W = len(CONTEXTS), -(-max(CONTEXTS) // page)
    window, keep = (150 if "window" in extras else 0), (20 if "keep" in extras else 0)
    cap = 3.0 if "cap" in extras else 0.0
    sink = torch.randn(H, generator=g, device="cuda") if "sink" in extras else None
    gate = torch.randn(S, H * D, generator=g, device="cuda") if "gate" in extras else None
    q = torch.randn(S, H * D, generator=g, device="cuda") * 2
    pages = S * W + 1
    k, v = torch.randn(pages, page, KVH, D, generator=g, device="cuda"), torch.randn(pages, KVH, D, page, generator=g, device="cuda")
    k[0], v[0] = float("nan"), float("nan")                     # what released and padding entries of a table point at
    table = torch.zeros(S, W, dtype=torch.int32, device="cuda")
    out = torch.full((S, H * D), float("nan"), device="cuda")
    wants = []
    for s, ctx in enumerate(CONTEXTS):
        ids = torch.arange(1 + s * W, 1 + s * W + -(-ctx // page), device="cuda", dtype=torch.int32)
        seen = torch.arange(ctx, device="cuda")
        lo = max(0, ctx - window) if window else 0
        seen = seen[(seen >= lo) | (seen < keep)]
        for j in range(len(ids)):                               # pages that no seen key lies in have been given back
            if not ((seen // page) == j).any():
                ids[j] = 0
        table[s, :len(ids)] = ids
        at = ids[(seen // page).long()].long()
        kk, vv = k[at, seen % page].double(), v[at, :, :, seen % page].double()         # [keys, KVH, D]
        v[ids[-1].long(), :, :, (ctx - 1) % page + 1:] = float("nan")                   # places beyond the newest key
        k[ids[-1].long(), (ctx - 1) % page + 1:] = float("nan")
        for h in range(H):
            sc = kk[:, h // (H // KVH)] @ q[s, h * D:(h + 1) * D].double() * D ** -0.5
            if cap:
                sc = cap * torch.tanh(sc / cap)
            e = torch.exp(sc - sc.max())
            total = e.sum() + (torch.exp(sink[h].double() - sc.max()) if sink is not None else 0)
            o = (e / total) @ vv[:, h // (H // KVH)]
            wants.append(o * torch.sigmoid(gate[s, h * D:(h + 1) * D].double()) if gate is not None else o)
    ctxs = torch.tensor(CONTEXTS, dtype=torch.int32, device="cuda")
    chunks = -(-W * page // 128) + 1
    part_o, part_ml = (torch.full((S * H * chunks * n,), float("nan"), device="cuda") for n in (D, 2))
    assert library().tm_attn_decode_f32(_ptr(q), I(H * D), _ptr(out), I(H * D), _ptr(k), _ptr(v), _ptr(table), I(W), _ptr(ctxs), _ptr(part_o),
                                        _ptr(part_ml), I(chunks), I(S), I(H), I(KVH), I(D), I(page), F(D ** -0.5), I(window), I(keep), F(cap),
                                        _ptr(sink), _ptr(gate), I(H * D), _stream()) == 0
    want = torch.stack(wants).view(S, H * D)
    # scores of size up to about 10 with 32-bit dot products: 2^-20 absolute, which the exponential makes relative; values of size up to 5
    assert (out.double() - want).abs().max() <= 2.0 ** -17


def test_the_grid_of_the_attention_does_not_grow_with_the_longest_context_there_can_be():
    """A block for each of 256 chunks of 64 requests of two kv heads would be 32,768, next to all of which find no key."""
    blocks = library().tm_attn_decode_f32_blocks
    assert blocks(64, 2, 256) == 16 and blocks(1, 2, 256) == 256 and blocks(8, 2, 6) == 6 and blocks(5000, 8, 256) == 1


def test_attention_of_single_tokens_walks_the_chunks_of_long_contexts():
    """More chunks than the grid has blocks for a pair: the same bits as for each request alone, whose grid has one for each."""
    S, H, KVH, D, page, most = 32, 32, 16, 32, 16, 2000
    g = torch.Generator(device="cuda").manual_seed(3)
    W, chunks = -(-most // page), -(-most // 128)
    assert library().tm_attn_decode_f32_blocks(S, KVH, chunks) == 4 and library().tm_attn_decode_f32_blocks(1, KVH, chunks) == chunks
    q = torch.randn(S, H * D, generator=g, device="cuda")
    k, v = torch.randn(2, S * W * page * KVH * D, generator=g, device="cuda")
    table = torch.arange(S * W, device="cuda", dtype=torch.int32).view(S, W)
    ctxs = torch.randint(1, most + 1, (S,), generator=g, device="cuda", dtype=torch.int32)
    ctxs[:3] = torch.tensor([most, 1, 512])

    def run(rows, window, keep):
        n = len(rows)
        out = torch.full((n, H * D), float("nan"), device="cuda")
        part_o, part_ml = (torch.full((n * H * chunks * e,), float("nan"), device="cuda") for e in (D, 2))
        qs, ts, cs = q[rows].contiguous(), table[rows].contiguous(), ctxs[rows].contiguous()
        assert library().tm_attn_decode_f32(_ptr(qs), I(H * D), _ptr(out), I(H * D), _ptr(k), _ptr(v), _ptr(ts), I(W), _ptr(cs), _ptr(part_o),
                                            _ptr(part_ml), I(chunks), I(n), I(H), I(KVH), I(D), I(page), F(D ** -0.5), I(window), I(keep), F(0.0),
                                            _ptr(None), _ptr(None), I(H * D), _stream()) == 0
        return out

    for window, keep in ((0, 0), (300, 20)):
        together = run(list(range(S)), window, keep)
        assert together.isfinite().all()
        assert torch.equal(together, torch.cat([run([s], window, keep) for s in range(S)]))
