"""The decode attention that takes all of a (request, kv head)'s context in one block: the bits of the kernels that split it over blocks
and merge, at the edges of runs of 64 keys, chunks of 256 and rounds of wavefronts, with every option."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(H, KVH, D, page, lens, seed):
    g = torch.Generator().manual_seed(seed)
    S, width = len(lens), -(-max(lens) // page)
    pages = S * width
    k = torch.randn(pages, page, KVH, D, generator=g).bfloat16().to(DEV)
    v = torch.randn(pages, KVH, D, page, generator=g).bfloat16().to(DEV)
    tables = torch.randperm(pages, generator=g).int().view(S, width)
    for s, n in enumerate(lens):                        # what lies beyond a context is never used
        for i in range(-(-n // page), width):
            k[tables[s, i].item()], v[tables[s, i].item()] = float("nan"), float("nan")
        if n % page:
            v[tables[s, n // page].item(), :, :, n % page:] = float("nan")
    q = torch.randn(S, H * D, generator=g).bfloat16().to(DEV)
    return q, k, v, tables.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV), g


@pytest.mark.parametrize("H,KVH,D,page", [(14, 2, 64, 16), (8, 8, 32, 16), (28, 4, 128, 16), (16, 1, 64, 64), (6, 2, 96, 32), (16, 1, 128, 16)])
@pytest.mark.parametrize("lens", [[1, 63, 64, 65, 192, 255, 256], [257, 1, 448, 512], [513, 700, 768, 3], [769, 1024, 960], [1025, 1280, 257, 1]])
@pytest.mark.parametrize("window,keep,softcap,options", [(0, 0, 0.0, False), (100, 0, 0.0, True), (300, 70, 0.0, False), (0, 0, 20.0, True)])
def test_one_block_has_the_bits_of_the_split_contexts(H, KVH, D, page, lens, window, keep, softcap, options):
    from tokenmill_amd.hip import ops
    if D > 64 and H // KVH == 16 and max(lens) > 1024:
        pytest.skip("more than a block's LDS holds")
    q, k, v, tables, ctx, g = _case(H, KVH, D, page, lens, 7)
    S = len(lens)
    sink = torch.randn(H, generator=g).to(DEV) if options else None
    gate = torch.randn(S, H * D, generator=g).bfloat16().to(DEV) if options else None

    def run(max_context, table, **which):
        out = torch.full((S, H * D), 3.0, dtype=torch.bfloat16, device=DEV)
        return ops.attn_decode_mfma(q, out, k, v, table, ctx, H, KVH, D, D ** -0.5, window, max_context, softcap=softcap, sink=sink, keep=keep,
                                    channel_gate=gate, **which)

    got = run(max(lens), tables, whole=True)
    width = -(-(max(lens) + 256) // page)                # a chunk more than there is: the split kernels take even a context of one chunk
    wide = torch.zeros(S, width, dtype=torch.int32, device=DEV)
    wide[:, :tables.shape[1]] = tables
    want = run(max(lens) + 256, wide, split=True, whole=False)
    assert torch.isfinite(want.float()).all()
    assert torch.equal(got, want)
    sub = [S - 1, 0]                                     # the same requests in another step
    out = torch.empty(2, H * D, dtype=torch.bfloat16, device=DEV)
    ops.attn_decode_mfma(q[sub].contiguous(), out, k, v, tables[sub].contiguous(), ctx[sub].contiguous(), H, KVH, D, D ** -0.5, window, max(lens),
                         softcap=softcap, sink=sink, keep=keep, channel_gate=gate[sub].contiguous() if options else None, whole=True)
    assert torch.equal(out, got[sub])


def test_more_than_the_lds_holds_is_refused():
    from tokenmill_amd.hip import ops
    q, k, v, tables, ctx, _ = _case(16, 1, 128, 16, [1300], 3)
    with pytest.raises(Exception):
        ops.attn_decode_mfma(q, torch.empty_like(q), k, v, tables, ctx, 16, 1, 128, 0.1, 0, 1300, whole=True)
