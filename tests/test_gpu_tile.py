"""The tiled products of prompt-sized steps (csrc/gemm_tile.hip) against 64-bit ones, at the edges of their tiles: rows and columns
that fill no tile, the shortest K, the last part of a split K shorter than the others, every tile shape the rule chooses with
every epilogue, rows of A that lie apart."""
from __future__ import annotations

import ctypes

import pytest
import torch

from tokenmill_amd.hip.library import library

pytestmark = pytest.mark.gpu
P, I = ctypes.c_void_p, ctypes.c_int

# (rows, result columns, K): every tile
SILU = [(65, 8, 256), (77, 4864, 320), (129, 1000, 256), (200, 4864, 256), (257, 4864, 448), (333, 4864, 256), (512, 4864, 896), (1000, 6000, 448),
        (700, 4864, 448), (1000, 4864, 896), (2048, 4864, 896), (4001, 4864, 896), (2000, 4096, 1792), (1025, 40, 256), (33, 2816, 1024),
        (700, 2816, 1024)]


def _operands(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    return a, w, a.double() @ w.double().T


def _stream():
    return P(torch.cuda.current_stream().cuda_stream)


def _product(what, size):
    """Rows, columns, K and parts of K of a case of one of the lists."""
    if what == "qkv":
        M, H, KVH, D, K, _ = size
        return M, (H + 2 * KVH) * D, K, 1
    M, n, K = size
    return M, 2 * n if what == "silu" else n, K, library().tm_tile_linear_parts(M, n, K) if what == "parts" else 1


def test_the_sizes_reach_every_tile_with_every_epilogue():
    lib = library()
    few = [size for size in PARTS if size[0] <= 64 and size[2] >= 320]          # these run one of two tiles of their own
    assert {K // 64 > 200 and N >= 3072 for M, N, K in few} == {True, False}
    for what, sizes in (("silu", SILU), ("qkv", QKV), ("parts", [size for size in PARTS if size not in few]), ("linear", [])):
        sizes = sizes + [size for of, size, _ in BETWEEN if of == what]
        runs = {lib.tm_gemm_tile_picked(*_product(what, size)) for size in sizes}
        assert runs >= (set(range(15)) if what != "linear" else set(range(11, 15))), what      # (plain products: test_gpu_tile_ends.py has the others)


@pytest.mark.parametrize("M,n,K", SILU)
def test_gate_up_silu(M, n, K):
    a, w, ref = _operands(M, 2 * n, K, M + n)
    out = torch.full((M, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    assert library().tm_tile_gate_up_silu(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(out.data_ptr()), I(n), _stream()) == 0
    gate, up = ref.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    # gate and up are rounded to bfloat16 (by at most 2^-8 of themselves; silu' <= 1.1), and the result is; 32-bit sums of K terms
    # of size 1 / sqrt(K) add less than 2^-18
    bound = 2.0 ** -8 * (1.1 * gate.abs() * up.abs() + 2 * want.abs()) * 1.02 + 2.0 ** -18 * (1.1 * up.abs() + gate.abs() + 1)
    assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("scale", [1.0, 2.0 ** 127])
def test_the_activation_is_the_one_of_the_other_products(scale):
    """Rows of A with one entry give gate and up without a rounding, so the activation alone is compared, bit for bit with the kernel
    behind a plain product: every bfloat16 gate there is, or, at the large scale, infinities too (and infinities times zero)."""
    M = n = K = 256
    g = torch.Generator(device="cuda").manual_seed(5)
    a = (torch.eye(K, device="cuda") * scale).bfloat16()
    w = (torch.randn(2 * n, K, generator=g, device="cuda") * 3).bfloat16()
    if scale == 1:
        every = torch.arange(65536, device="cuda").sub(32768).to(torch.int16).view(torch.bfloat16)
        w[:n] = torch.where(every.isfinite() & (every.float().abs() >= 2.0 ** -100), every, torch.zeros_like(every)).view(n, K)
    out, want = torch.empty(2, M, n, device="cuda", dtype=torch.bfloat16)
    lib = library()
    assert lib.tm_tile_gate_up_silu(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(out.data_ptr()), I(n), _stream()) == 0
    both = (w.float().T * scale).bfloat16().contiguous()
    assert lib.tm_silu_mul(P(both.data_ptr()), P(want.data_ptr()), I(1), I(M), I(n), _stream()) == 0
    assert both.isinf().any() == (scale > 1)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.nan_to_num(0.0), want.nan_to_num(0.0))


def test_the_activation_of_infinities_and_what_is_no_number():
    """One column of the matrix that is not zero: gates of every bfloat16 value down to 2^-100, both infinities and every NaN, times one; the bits of the kernel
    behind a plain product."""
    every = torch.arange(65536, device="cuda").sub(32768).to(torch.int16).view(torch.bfloat16)
    gates = torch.where(every.float().abs() < 2.0 ** -100, torch.zeros_like(every), every)
    M, n, K = 65, 65536, 256
    a, w = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16), torch.zeros(2 * n, K, device="cuda", dtype=torch.bfloat16)
    a[:, 0], w[:n, 0], w[n:, 0] = 1.0, gates, 1.0
    out = torch.empty(M, n, device="cuda", dtype=torch.bfloat16)
    assert library().tm_tile_gate_up_silu(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(out.data_ptr()), I(n), _stream()) == 0
    both, want = torch.cat([gates, torch.ones_like(gates)])[None].contiguous(), torch.empty(1, n, device="cuda", dtype=torch.bfloat16)
    assert library().tm_silu_mul(P(both.data_ptr()), P(want.data_ptr()), I(1), I(1), I(n), _stream()) == 0
    assert torch.equal(want.isnan()[0], gates.isnan() | (gates == float("-inf")))
    assert torch.equal(out.isnan(), want.isnan().expand(M, n)) and torch.equal(out.nan_to_num(0.0), want.nan_to_num(0.0).expand(M, n))


# (rows, heads, kv heads, head size, K, page): every tile
QKV = [(65, 14, 2, 64, 256, 16), (333, 14, 2, 64, 896, 16), (1000, 28, 4, 128, 256, 16), (2500, 14, 2, 64, 256, 16), (70, 3, 1, 192, 256, 16),
       (66, 28, 4, 128, 512, 4), (400, 28, 4, 128, 512, 64), (600, 28, 4, 128, 512, 128), (1001, 28, 4, 128, 512, 1), (1500, 28, 4, 128, 512, 32),
       (2000, 28, 4, 128, 512, 16), (2500, 28, 4, 128, 512, 16), (3001, 28, 4, 128, 512, 64), (3200, 28, 4, 128, 512, 16), (199, 28, 4, 128, 512, 16)]


@pytest.mark.parametrize("stored", [True, False])
@pytest.mark.parametrize("bias_dtype", [torch.float32, torch.bfloat16, None])
@pytest.mark.parametrize("M,H,KVH,D,K,page", QKV)
def test_qkv_with_rotation_and_cache_write(M, H, KVH, D, K, page, bias_dtype, stored):
    N = (H + 2 * KVH) * D
    a, w, ref = _operands(M, N, K, M + H)
    g = torch.Generator(device="cuda").manual_seed(M)
    bias = torch.randn(N, generator=g, device="cuda").to(bias_dtype) if bias_dtype else None
    angle = torch.rand(300, D // 2, generator=g, device="cuda") * 6.28
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, 300, (M,), generator=g, device="cuda", dtype=torch.int32)
    pages = -(-M // page) + 2
    slots = torch.randperm(pages * page, generator=g, device="cuda")[:M].int()
    slots[1::7] = -1
    q = torch.full((M, H * D), 7.0, device="cuda", dtype=torch.bfloat16)
    k = torch.full((pages, page, KVH, D), 7.0, device="cuda", dtype=torch.bfloat16)
    v = torch.full((pages, KVH, D, page), 7.0, device="cuda", dtype=torch.bfloat16)
    code = -1 if bias is None else (0 if bias_dtype == torch.float32 else 1)
    assert library().tm_tile_qkv_rope(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(bias.data_ptr() if bias is not None else None), I(code),
                                      P(q.data_ptr()), I(H), I(KVH), I(D), P(cos.data_ptr()), P(sin.data_ptr()), P(pos.data_ptr()),
                                      P(slots.data_ptr() if stored else None), P(k.data_ptr()), P(v.data_ptr()), I(page), _stream()) == 0
    x = (ref + (bias.double() if bias is not None else 0)).view(M, H + 2 * KVH, D)
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    c, s = (t.double()[pos.long()][:, None] for t in (cos, sin))
    turned = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    size = torch.cat([lo.abs() + hi.abs()] * 2, -1)             # each of the pair is rounded, then the result is
    bound = 2.0 ** -8 * (size + turned.abs()) * 1.02 + 2.0 ** -17
    assert ((q.double().view(M, H, D) - turned[:, :H]).abs() <= bound[:, :H]).all()
    kept = (slots >= 0) & stored
    at = slots[kept].long()
    keys, values = k.view(-1, KVH, D), v.permute(0, 3, 1, 2).reshape(-1, KVH, D)
    assert ((keys[at].double() - turned[kept, H:H + KVH]).abs() <= bound[kept, H:H + KVH]).all()
    assert ((values[at].double() - x[kept, H + KVH:]).abs() <= 2.0 ** -8 * x[kept, H + KVH:].abs() * 1.02 + 2.0 ** -17).all()
    others = torch.ones(pages * page, dtype=torch.bool, device="cuda")
    others[at] = False
    assert (keys[others] == 7).all() and (values[others] == 7).all()


PARTS = [(65, 896, 896), (77, 896, 4864), (130, 3584, 960), (333, 896, 4864), (1000, 1016, 4864), (2048, 896, 896), (2048, 896, 4864),
         (4000, 896, 4864), (1000, 3584, 3584), (500, 3584, 18944), (650, 3584, 18944), (520, 3584, 18944), (265, 3584, 18944),
         (200, 3584, 18944), (135, 3584, 18944), (135, 3584, 3584), (100, 3584, 3584),
         # few rows: the tile with a ring of five, its shortest parts, one part, K below the ring, the wide tile of long K
         (1, 896, 896), (8, 3584, 3584), (17, 1000, 320), (16, 896, 4864), (33, 40, 256), (64, 2048, 2048), (64, 520, 12800),
         (40, 264, 12864), (5, 8200, 640), (48, 3584, 18944), (3, 3072, 12864)]


@pytest.mark.parametrize("M,N,K", PARTS)
def test_partial_sums_of_a_split_k(M, N, K):
    lib = library()
    parts = lib.tm_tile_linear_parts(M, N, K)
    assert 1 <= parts <= 8
    a, w, ref = _operands(M, N, K, M + K)
    out = torch.full((parts, M, N), float("nan"), device="cuda")
    assert lib.tm_tile_linear_split(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), I(N), P(out.data_ptr()), _stream()) == 0
    # 32-bit sums of products of size 1 / sqrt(K): the rounding of each of K additions to a sum of at most about 5
    assert (out.double().sum(0) - ref).abs().max() <= 2.0 ** -24 * 5 * 4 * K ** 0.5


@pytest.mark.parametrize("M,K", [(40, 640), (77, 256), (300, 896)])
def test_rows_of_a_that_lie_apart(M, K):
    """The same bits as of rows side by side, from every epilogue and in both types."""
    lib, N, H, KVH, D = library(), 512, 2, 1, 128
    for dt in (torch.bfloat16, torch.float32):
        bf = dt is torch.bfloat16
        g = torch.Generator(device="cuda").manual_seed(M)
        wide = torch.randn(M, K + 24, generator=g, device="cuda").to(dt)
        w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(dt)
        cos, sin = torch.rand(2, M, D // 2, generator=g, device="cuda")
        pos = torch.arange(M, device="cuda", dtype=torch.int32)
        got = []
        for a in (wide[:, :K], wide[:, :K].contiguous()):
            lead = (P(a.data_ptr()), I(a.stride(0)), I(M), I(K), P(w.data_ptr()))
            act, q = torch.empty(M, N // 2, device="cuda", dtype=dt), torch.empty(M, H * D, device="cuda", dtype=dt)
            k, v = torch.zeros(2, M * KVH * D, device="cuda", dtype=dt)
            n = lib.tm_tile_linear_parts(M, N, K) if bf else 2
            sums = torch.empty(n, M, N, device="cuda")
            tail = (P(q.data_ptr()), I(H), I(KVH), I(D), P(cos.data_ptr()), P(sin.data_ptr()), P(pos.data_ptr()), P(pos.data_ptr()), P(k.data_ptr()),
                    P(v.data_ptr()), I(1), _stream())
            if bf:
                assert lib.tm_tile_gate_up_silu(*lead, P(act.data_ptr()), I(N // 2), _stream()) == 0
                assert lib.tm_tile_qkv_rope(*lead, P(None), I(-1), *tail) == 0
                assert lib.tm_tile_linear_split(*lead, I(N), P(sums.data_ptr()), _stream()) == 0
            else:
                assert lib.tm_tile_f32_gate_up_silu(*lead, P(act.data_ptr()), I(N // 2), _stream()) == 0
                assert lib.tm_tile_f32_qkv_rope(*lead, P(None), *tail) == 0
                assert lib.tm_tile_f32_linear_split(*lead, I(N), P(sums.data_ptr()), I(n), _stream()) == 0
            got.append((act, q, k, v, sums))
        assert all(torch.equal(x, y) for x, y in zip(*got)) and all(x.isfinite().all() for x in got[0])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_the_rows_do_not_change_a_row_of_gate_up_or_of_qkv(dt):
    """Whichever tile the number of rows chooses: K is not split, and a row's sums run over k in one order."""
    lib, most, K, n, H, KVH, D = library(), 3200, 896, 2048, 14, 2, 64
    g = torch.Generator(device="cuda").manual_seed(4)
    a = torch.randn(most, K, generator=g, device="cuda").to(dt)
    w = (torch.randn(2 * n, K, generator=g, device="cuda") * K ** -0.5).to(dt)
    cos, sin = torch.rand(2, most, D // 2, generator=g, device="cuda")
    pos = torch.arange(most, device="cuda", dtype=torch.int32)
    f32, tiles, got = dt is torch.float32, set(), []
    for M in (most, 17, 65, 130, 200, 333, 512, 700, 1000, 1500, 2048):
        act, q = torch.empty(M, n, device="cuda", dtype=dt), torch.empty(M, H * D, device="cuda", dtype=dt)
        k, v = torch.zeros(2, most, KVH * D, device="cuda", dtype=dt)
        lead = (P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()))
        tail = (P(q.data_ptr()), I(H), I(KVH), I(D), P(cos.data_ptr()), P(sin.data_ptr()), P(pos.data_ptr()), P(pos.data_ptr()), P(k.data_ptr()),
                P(v.data_ptr()), I(1), _stream())
        assert (lib.tm_tile_f32_gate_up_silu if f32 else lib.tm_tile_gate_up_silu)(*lead, P(act.data_ptr()), I(n), _stream()) == 0
        assert (lib.tm_tile_f32_qkv_rope(*lead, P(None), *tail) if f32 else lib.tm_tile_qkv_rope(*lead, P(None), I(-1), *tail)) == 0
        got.append((act, q, k[:M], v[:M]))
        tiles.add(lib.tm_gemm_tile_picked(M, 2 * n, K, 1))
    assert len(tiles) >= 6
    for few in got[1:]:
        assert all(torch.equal(x, y[:x.shape[0]]) for x, y in zip(few, got[0]))


# rows and matrices whose launch takes a tile between those of the table (11 to 14), and the table's where the sizes above have come to take another
BETWEEN = [("silu", (804, 2816, 320), 5), ("silu", (321, 4864, 320), 6), ("silu", (449, 2000, 320), 7), ("silu", (1409, 1000, 320), 11),
           ("silu", (417, 4864, 320), 12), ("silu", (804, 2816, 832), 13), ("silu", (579, 4864, 320), 14), ("qkv", (2242, 16, 16, 64, 320, 16), 4),
           ("qkv", (1601, 16, 16, 64, 320, 16), 5), ("qkv", (707, 28, 4, 128, 320, 16), 6), ("qkv", (611, 28, 4, 128, 320, 16), 11),
           ("qkv", (1345, 16, 16, 64, 320, 1), 12), ("qkv", (1605, 16, 16, 64, 832, 16), 13), ("qkv", (2017, 16, 16, 64, 320, 32), 14),
           ("parts", (1860, 1536, 320), 11), ("parts", (579, 3584, 1280), 12), ("parts", (648, 3584, 1600), 13), ("parts", (2311, 896, 2112), 14),
           ("linear", (929, 3072, 320), 11), ("linear", (1347, 3072, 320), 12), ("linear", (1606, 3072, 832), 13), ("linear", (2018, 3072, 320), 14)]


@pytest.mark.parametrize("what,size,tile", BETWEEN)
def test_tiles_between(what, size, tile):
    """Against 64 bits as above, and a row's bits are those of the calls of fewer rows, which take other tiles."""
    lib = library()
    M, N, K, parts = _product(what, size)
    assert lib.tm_gemm_tile_picked(M, N, K, parts) == tile
    if what == "qkv":
        test_qkv_with_rotation_and_cache_write(*size, torch.float32, True)
    if what == "parts":
        test_partial_sums_of_a_split_k(*size)
    if what == "silu":
        test_gate_up_silu(*size)
    a, w, ref = _operands(M, N, K, M)
    lead = lambda m: (P(a.data_ptr()), I(K), I(m), I(K), P(w.data_ptr()))

    def product(m, dt=torch.bfloat16):
        """A row a token of everything that the call gives."""
        if what == "qkv":
            _, H, KVH, D, _, page = size
            q, (k, v) = torch.full((m, H * D), float("nan"), device="cuda", dtype=dt), torch.zeros(2, -(-M // page), page * KVH * D, device="cuda", dtype=dt)
            cos, sin = torch.rand(2, M, D // 2, generator=torch.Generator(device="cuda").manual_seed(6), device="cuda")
            pos = torch.arange(m, device="cuda", dtype=torch.int32)
            assert lib.tm_tile_qkv_rope(*lead(m), P(None), I(-1), P(q.data_ptr()), I(H), I(KVH), I(D), P(cos.data_ptr()), P(sin.data_ptr()), P(pos.data_ptr()),
                                        P(pos.data_ptr()), P(k.data_ptr()), P(v.data_ptr()), I(page), _stream()) == 0
            return torch.cat([q, k.view(-1, KVH * D)[:m], v.view(-1, KVH * D, page).transpose(1, 2).reshape(-1, KVH * D)[:m]], 1)
        if what == "parts":
            sums = torch.full((parts, m, N), float("nan"), device="cuda")
            assert lib.tm_tile_linear_split(*lead(m), I(N), P(sums.data_ptr()), _stream()) == 0
            return sums.transpose(0, 1)
        out = torch.full((m, size[1]), float("nan"), device="cuda", dtype=dt)
        if what == "silu":
            assert lib.tm_tile_gate_up_silu(*lead(m), P(out.data_ptr()), I(N // 2), _stream()) == 0
        else:
            assert lib.tm_tile_linear(*lead(m), I(N), P(out.data_ptr()), I(N), I(1 if dt is torch.bfloat16 else 0), _stream()) == 0
        return out

    # fewer rows, which take other tiles (of the same number of parts of K)
    few = [77, 300] if what != "parts" else [m for m in range(M - 1, 64, -1) if lib.tm_tile_linear_parts(m, N, K) == parts and lib.tm_gemm_tile_picked(m, N, K, parts) != tile][:2]
    full = product(M)
    assert few and {lib.tm_gemm_tile_picked(m, N, K, parts) for m in few} != {tile} and not full.isnan().any()
    for m in few:
        assert torch.equal(product(m), full[:m])
    if what == "linear":
        sums = product(M, torch.float32)
        assert (sums.double() - ref).abs().max() <= 2.0 ** -24 * 5 * 4 * K ** 0.5 and torch.equal(sums.bfloat16(), full)


# an output and a down projection of the shipped shapes and what lies around the line between the two tiles of few rows
@pytest.mark.parametrize("N,K", [(896, 896), (896, 4864), (2048, 11008), (3584, 3584), (3584, 18944), (5120, 27648), (3072, 12864), (2944, 12864)])
def test_few_rows_do_not_change_a_row_of_a_split_product(N, K):
    lib = library()
    parts = lib.tm_tile_linear_parts(1, N, K)
    a, w, _ = _operands(64, N, K, N + K)
    sums = {}
    for M in (1, 5, 16, 17, 32, 33, 48, 64):
        assert lib.tm_tile_linear_parts(M, N, K) == parts
        out = torch.full((parts, M, N), float("nan"), device="cuda")
        assert lib.tm_tile_linear_split(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), I(N), P(out.data_ptr()), _stream()) == 0
        sums[M] = out
    assert all(torch.equal(out, sums[64][:, :M]) for M, out in sums.items())


# few experts; one wavefront, four, all; pairs that are held and that are not; experts without a pair, without matrices
@pytest.mark.parametrize("T,E,real,top,rows", [(1, 1, 1, 1, 32), (1024, 16, 15, 2, 64), (1025, 16, 16, 2, 64), (100, 17, 17, 2, 32), (128, 64, 64, 2, 64), (129, 64, 63, 2, 64), (5, 65, 65, 2, 32), (512, 256, 256, 2, 128), (513, 17, 16, 2, 64),
                                               (3, 257, 257, 5, 32), (64, 1024, 1000, 8, 32), (64, 1024, 1024, 8, 32), (2048, 3, 3, 2, 128), (4097, 1, 1, 1, 64),
                                               (3000, 70, 64, 4, 128), (5, 8, 0, 2, 32)])
def test_route(T, E, real, top, rows):
    lib = library()
    g = torch.Generator().manual_seed(T + E)
    table = torch.rand(T, E, generator=g).argsort(1)[:, :top].int().contiguous()
    n = T * top
    most = min(n, n // rows + E)
    slot_pair, pair_slot, tiles, n_tiles = (torch.full((k,), -7, dtype=torch.int32, device="cuda") for k in (n, n, 3 * most, 1))
    chosen = table.to("cuda")
    assert lib.tm_moe_route_chosen(None, P(chosen.data_ptr()), I(T), I(top), I(E), I(real), I(rows), P(slot_pair.data_ptr()), P(pair_slot.data_ptr()),
                                   P(tiles.data_ptr()), P(n_tiles.data_ptr()), _stream()) == 0
    e = table.flatten().long()
    count = torch.bincount(e[e < real], minlength=real)[:real].tolist()
    want, at = [], 0
    for x, c in enumerate(count):
        want += [(x, at + r, min(rows, c - r)) for r in range(0, c, rows)]
        at += c
    assert n_tiles.item() == len(want) and [tuple(t) for t in tiles.view(-1, 3)[:len(want)].tolist()] == want
    slots, pairs = pair_slot.cpu().long(), slot_pair.cpu().long()
    assert (slots[e >= real] == -1).all() and slots[e < real].sort().values.tolist() == list(range(at))
    assert torch.equal(pairs[slots[e < real]], torch.nonzero(e < real).flatten())
    assert (e[pairs[:at]].diff() >= 0).all() if at > 1 else True


# (tokens, experts, choices a token, K, width): experts without a token, with one, with tiles that are full and that are not
EXPERTS = [(40, 3, 1, 192, 16), (200, 5, 2, 256, 208), (700, 4, 2, 320, 576), (130, 16, 3, 192, 192)]


@pytest.mark.parametrize("tile_rows", [64, 128])
@pytest.mark.parametrize("kind", ["silu", "clamped", "relu2"])
@pytest.mark.parametrize("T,E,top,K,F", EXPERTS)
def test_experts(T, E, top, K, F, kind, tile_rows):
    from tokenmill_amd.hip import ops
    lib = library()
    g = torch.Generator(device="cuda").manual_seed(T + F)
    gated = kind != "relu2"
    x = torch.randn(T, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(E, F * (2 if gated else 1), K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    down = (torch.randn(E, K, F, generator=g, device="cuda") * F ** -0.5).bfloat16()
    table = torch.rand(50, E, generator=g, device="cuda").argsort(1)[:, :top].int().contiguous()
    if E == 16:
        table[:, 0] = 7                                         # most of the tokens in one expert
        table[:, 1:] = torch.tensor([2, 5], device="cuda", dtype=torch.int32)
    ids = torch.randint(0, 50, (T,), generator=g, device="cuda", dtype=torch.int32)
    slot_pair, _, tiles, n_tiles, _ = ops.moe_route(ids, table, E, tile_rows)
    weight = torch.rand(T * top, generator=g, device="cuda")
    limit, alpha = 1.5, 1.7
    act = torch.full((T * top, F), float("nan"), device="cuda", dtype=torch.bfloat16)
    part = torch.full((T * top, K), float("nan"), device="cuda")
    assert lib.tm_tile_experts_takes(P(x.data_ptr()), I(K), ctypes.c_longlong(T), P(w.data_ptr()), P(act.data_ptr()), I(tile_rows), I(K), I(w.shape[1]))
    common = (P(tiles.data_ptr()), P(n_tiles.data_ptr()), I(tiles.shape[0]), I(tile_rows))
    if kind == "clamped":
        rc = lib.tm_moe_clamped_mfma(P(x.data_ptr()), I(K), P(slot_pair.data_ptr()), I(top), P(weight.data_ptr()), P(w.data_ptr()), P(act.data_ptr()),
                                     *common, I(K), I(F), ctypes.c_float(limit), ctypes.c_float(alpha), _stream())
    else:
        first = lib.tm_moe_gate_up_mfma if gated else lib.tm_moe_up_act_mfma
        rc = first(P(x.data_ptr()), I(K), P(slot_pair.data_ptr()), I(top), P(w.data_ptr()), P(act.data_ptr()), *common, I(K), I(F), _stream())
    assert rc == 0
    takes_down = bool(lib.tm_tile_experts_takes(P(act.data_ptr()), I(F), ctypes.c_longlong(T * top), P(down.data_ptr()), P(part.data_ptr()), I(tile_rows), I(F), I(K)))
    assert takes_down == (F % 64 == 0 and F >= 192)
    assert lib.tm_moe_down_mfma(P(act.data_ptr()), P(down.data_ptr()), P(part.data_ptr()), *common, I(F), I(K), _stream()) == 0
    pairs = slot_pair.long()
    expert = table[ids.long()].flatten().long()[pairs]
    rows = x.double()[pairs // top]
    h = torch.empty(T * top, w.shape[1], dtype=torch.float64, device="cuda")
    for e in range(E):
        h[expert == e] = rows[expert == e] @ w[e].double().T
    if kind == "relu2":
        want, slope = h.clamp(min=0) ** 2, 2 * h.abs()
    else:
        a, b = h.chunk(2, 1)
        if kind == "silu":
            want, slope = torch.nn.functional.silu(a) * b, 1.1 * b.abs() + a.abs()
        else:
            a, b = a * weight.double()[pairs, None], b * weight.double()[pairs, None]
            a, b = a.clamp(max=limit), b.clamp(-limit, limit)
            want, slope = a * torch.sigmoid(alpha * a) * (b + 1), 1.5 * (b.abs() + 1) + a.abs()
    # the result is rounded to bfloat16 (by at most 2^-8 of itself); 32-bit sums of K terms of size 1 / sqrt(K) are off by less than 2^-18
    assert ((act.double() - want).abs() <= 2.0 ** -8 * want.abs() * 1.01 + 2.0 ** -18 * (slope + 1)).all()
    for e in range(E):
        ref = act[expert == e].double() @ down[e].double().T
        assert ((part[expert == e].double() - ref).abs() <= 2.0 ** -18 * (1 + act[expert == e].double().abs().amax(1, keepdim=True))).all()


def _operands32(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * K ** -0.5
    return a, w, a.double() @ w.double().T


# 32-bit sums in blocks of 128 k: a chain of 128 additions in a block, then K / 128 of sums of at most about 5
def _bound32(K):
    return 2.0 ** -24 * 5 * (6 + (K / 128) ** 0.5) * 2


@pytest.mark.parametrize("M,n,K", [(17, 8, 128), (65, 40, 160), (333, 1000, 896), (1000, 4864, 896)])
def test_gate_up_silu_in_32_bit(M, n, K):
    a, w, ref = _operands32(M, 2 * n, K, M + n)
    out = torch.full((M, n), float("nan"), device="cuda")
    assert library().tm_tile_f32_gate_up_silu(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(out.data_ptr()), I(n), _stream()) == 0
    gate, up = ref.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    assert ((out.double() - want).abs() <= _bound32(K) * (1.1 * up.abs() + gate.abs() + 1) + 2.0 ** -20 * want.abs()).all()


@pytest.mark.parametrize("M,H,KVH,D,K", [(17, 3, 1, 64, 128), (333, 14, 2, 64, 896), (130, 4, 2, 128, 224)])
def test_qkv_in_32_bit(M, H, KVH, D, K):
    N, page = (H + 2 * KVH) * D, 16
    a, w, ref = _operands32(M, N, K, M + H)
    g = torch.Generator(device="cuda").manual_seed(M)
    bias = torch.randn(N, generator=g, device="cuda")
    angle = torch.rand(300, D // 2, generator=g, device="cuda") * 6.28
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, 300, (M,), generator=g, device="cuda", dtype=torch.int32)
    pages = -(-M // page) + 2
    slots = torch.randperm(pages * page, generator=g, device="cuda")[:M].int()
    slots[1::7] = -1
    q = torch.empty(M, H * D, device="cuda")
    k, v = torch.full((pages, page, KVH, D), 7.0, device="cuda"), torch.full((pages, KVH, D, page), 7.0, device="cuda")
    assert library().tm_tile_f32_qkv_rope(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), P(bias.data_ptr()), P(q.data_ptr()), I(H), I(KVH), I(D),
                                          P(cos.data_ptr()), P(sin.data_ptr()), P(pos.data_ptr()), P(slots.data_ptr()), P(k.data_ptr()),
                                          P(v.data_ptr()), I(page), _stream()) == 0
    x = (ref + bias.double()).view(M, H + 2 * KVH, D)
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    c, s = (t.double()[pos.long()][:, None] for t in (cos, sin))
    turned = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    bound = 2 * _bound32(K) + 2.0 ** -20
    assert (q.double().view(M, H, D) - turned[:, :H]).abs().max() <= bound
    kept = slots >= 0
    at = slots[kept].long()
    keys, values = k.view(-1, KVH, D), v.permute(0, 3, 1, 2).reshape(-1, KVH, D)
    assert (keys[at].double() - turned[kept, H:H + KVH]).abs().max() <= bound
    assert (values[at].double() - x[kept, H + KVH:]).abs().max() <= bound
    others = torch.ones(pages * page, dtype=torch.bool, device="cuda")
    others[at] = False
    assert (keys[others] == 7).all() and (values[others] == 7).all()


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("M,N,K", [(17, 8, 384), (333, 896, 896), (1000, 896, 4864)])
def test_products_and_partial_sums_in_32_bit(M, N, K, splits):
    lib = library()
    splits = splits or lib.tm_tile_f32_parts(M, N, K)
    a, w, ref = _operands32(M, N, K, M + K)
    out = torch.full((splits, M, N), float("nan"), device="cuda")
    assert lib.tm_tile_f32_linear_split(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), I(N), P(out.data_ptr()), I(splits), _stream()) == 0
    assert (out.double().sum(0) - ref).abs().max() <= _bound32(K)


@pytest.mark.parametrize("N,K", [(896, 896), (896, 4864), (2048, 5504), (3584, 3584), (5120, 1120), (8, 96)])
def test_the_rows_do_not_change_a_row_of_a_split_product_in_32_bit(N, K):
    lib = library()
    parts = lib.tm_tile_f32_parts(1, N, K)
    a, w, _ = _operands32(700, N, K, N + K)
    sums = {}
    for M in (17, 64, 65, 200, 333, 700):
        assert lib.tm_tile_f32_parts(M, N, K) == parts
        out = torch.full((parts, M, N), float("nan"), device="cuda")
        assert lib.tm_tile_f32_linear_split(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), I(N), P(out.data_ptr()), I(parts), _stream()) == 0
        sums[M] = out
    assert all(torch.equal(out, sums[700][:, :M]) for M, out in sums.items())


@pytest.mark.parametrize("N,K", [(9728, 896), (896, 896), (896, 4864), (3584, 18944)])
def test_products_in_32_bit_lose_less_than_the_kernel_of_one_block_size(N, K):
    """rms error against 64 bits beside that of gemm_f32_mfma.hip, whose sums run in blocks of 128 k: in blocks of half that, or in
    parts, the chains are shorter. At K = 896 (one part) the roundings' variance goes with 128 / 4 + 7 and 64 / 4 + 14 additions, 39
    to 30, and what the matrix unit rounds inside an addition goes with the block: a tenth less at least."""
    lib = library()
    M, parts = 333, lib.tm_tile_f32_parts(333, N, K) if N < K or N == K else 1
    a, w, ref = _operands32(M, N, K, 9)
    out, before = torch.empty(parts, M, N, device="cuda"), torch.empty(M, N, device="cuda")
    assert lib.tm_tile_f32_linear_split(P(a.data_ptr()), I(K), I(M), I(K), P(w.data_ptr()), I(N), P(out.data_ptr()), I(parts), _stream()) == 0
    assert lib.tm_gemm_f32_mfma(P(a.data_ptr()), I(K), P(w.data_ptr()), None, P(before.data_ptr()), I(N), I(M), I(N), I(K), _stream()) == 0
    total = out[0]
    for part in out[1:]:
        total = total + part                                    # in 32-bit, in the order of the norm
    now, then = ((t.double() - ref).square().mean().sqrt() for t in (total, before))
    assert now <= 0.9 * then


def test_what_the_kernels_do_not_take_is_refused():
    lib = library()
    a, w, _ = _operands(65, 128, 320, 1)
    out = torch.zeros(65, 64, device="cuda", dtype=torch.bfloat16)

    def run(a_ptr, lda, K, n):
        return lib.tm_tile_gate_up_silu(P(a_ptr), I(lda), I(65), I(K), P(w.data_ptr()), P(out.data_ptr()), I(n), _stream())

    assert run(a.data_ptr(), 320, 320, 64) == 0
    assert run(a.data_ptr() + 2, 320, 320, 64) == 1             # rows off their 16-byte places
    assert run(a.data_ptr(), 324, 320, 64) == 1
    assert run(a.data_ptr(), 320, 300, 64) == 1                 # k that is not whole steps
    assert run(a.data_ptr(), 320, 192, 64) == 1                 # fewer steps than the ring has buffers
    assert run(a.data_ptr(), 320, 320, 60) == 1
