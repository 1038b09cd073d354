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


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("keys", [256, 257])
def test_a_request_has_its_bits_in_either_order_of_the_key_loads(D, keys):
    """Up to 64 keys a wavefront and up to 64 channels, or beside 128 pairs and more, keys are loaded in the order of the product, else four lanes side by side."""
    from tokenmill_amd.hip import ops
    lens = [keys, 1, 64, 65, 200, keys - 1] + [100] * 58
    q, k, v, tables, ctx, _ = _case(6, 2, D, 16, lens, 11)

    def run(n):
        return ops.attn_decode_mfma(q[:n], torch.full_like(q[:n], 3.0), k, v, tables[:n], ctx[:n], 6, 2, D, D ** -0.5, 0, keys, whole=True)

    most = run(64)
    for n in (1, 6, 63):
        assert torch.equal(run(n), most[:n]), n


def test_more_than_the_lds_holds_is_refused():
    from tokenmill_amd.hip import ops
    q, k, v, tables, ctx, _ = _case(16, 1, 128, 16, [1300], 3)
    with pytest.raises(Exception):
        ops.attn_decode_mfma(q, torch.empty_like(q), k, v, tables, ctx, 16, 1, 128, 0.1, 0, 1300, whole=True)


@pytest.mark.parametrize("H,KVH,D", [(14, 2, 64), (8, 8, 32), (28, 4, 128), (16, 1, 64), (6, 2, 96), (16, 1, 128)])
@pytest.mark.parametrize("window,keep,softcap,options", [(0, 0, 0.0, False), (300, 70, 0.0, True), (0, 0, 20.0, False)])
def test_among_many_a_request_has_its_bits_whatever_the_lengths_beside_it(H, KVH, D, window, keep, softcap, options):
    """192 (request, kv head) pairs and more: by the kernel's rule one launch where all contexts are short, another beside a longer one."""
    from tokenmill_amd.hip import ops
    S = -(-192 // KVH) + 1
    edges = [1, 64, 65, 255, 256, 257, 512, 700, 768, 769, 1023, 1024, 1025, 1279, 1280, 1281, 1600]
    lens = [edges[i % len(edges)] for i in range(S - 1)] + [3000]
    q, k, v, tables, ctx, g = _case(H, KVH, D, 16, lens, 5)
    sink = torch.randn(H, generator=g).to(DEV) if options else None
    gate = torch.randn(S, H * D, generator=g).bfloat16().to(DEV) if options else None

    def run(longest):
        """The requests of at most so many keys, the others at one key; the rule's kernel for the longest."""
        cut = torch.where(ctx > longest, 1, ctx)
        out = torch.full((S, H * D), 3.0, dtype=torch.bfloat16, device=DEV)
        ops.attn_decode_mfma(q, out, k, v, tables, cut, H, KVH, D, D ** -0.5, window, longest, softcap=softcap, sink=sink, keep=keep, channel_gate=gate)
        assert torch.isfinite(out.float()).all()
        return out

    most = run(3000)
    for longest in (256, 512, 768, 1024, 1280, 1600):
        same = (ctx <= longest)
        assert torch.equal(run(longest)[same], most[same]), longest
    few = ops.attn_decode_mfma(q[:S - 1], torch.empty_like(q[:S - 1]), k, v, tables[:S - 1], ctx[:S - 1], H, KVH, D, D ** -0.5, window, 1600, softcap=softcap,
                               sink=sink, keep=keep, channel_gate=gate[:S - 1] if options else None)
    assert torch.equal(few, most[:S - 1])


def _many(portions, contexts, max_model_len, graphs):
    """The logits of a step of a small model (200 pairs and more of request and kv head)."""
    from conftest import qwen2_config
    from tokenmill_amd import EngineConfig, LLMEngine
    from tokenmill_amd.config.registry import architecture_name, get_architecture
    from tokenmill_amd.engine.runner import StepEntry
    shape = qwen2_config(num_hidden_layers=4, hidden_size=512, num_attention_heads=8, num_key_value_heads=2, intermediate_size=512, vocab_size=512,
                         rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True)
    arch = get_architecture(architecture_name(shape))
    model = arch.build_model(arch.config_from_dict(shape, None), None)
    g = torch.Generator(device="cuda").manual_seed(1)
    model.load({name: (torch.randn(spec.drawn_shape(), generator=g, device="cuda") * 0.1 + (spec.init == "ones")).bfloat16()
                for name, spec in sorted(model.tensor_specs().items())}, torch.bfloat16, torch.device(DEV))
    requests = [(0, n) for n in portions] + [(c - 1, 1) for c in contexts]
    engine = LLMEngine(EngineConfig(dtype="bfloat16", block_size=16, num_blocks=sum(-(-(a + b) // 16) for a, b in requests) + 4, watermark=0.0,
                                    max_model_len=max_model_len, max_num_seqs=128, max_num_batched_tokens=8192, hip_graphs=graphs), model=model)
    caches = [engine.cache.allocate(f"r{i}", a + b) for i, (a, b) in enumerate(requests)]
    ids = [torch.randint(0, 512, (a + b,), generator=torch.Generator().manual_seed(a + b)).tolist() for a, b in requests]
    for cache, prompt, (a, _) in zip(caches, ids, requests):
        if a:                                            # (without a graph of each prompt's shape)
            engine.runner.forward(engine.runner.prepare([StepEntry(cache, 0, prompt[:a])])[0])
    entries = [StepEntry(cache, a, prompt[a:], [b - 1]) for cache, prompt, (a, b) in zip(caches, ids, requests)]
    for _ in range(4 if graphs else 1):
        logits = engine.runner.step(entries).clone()
    assert not graphs or engine.runner.graphs.replays > 0 or engine.runner.step_graphs.replays > 0
    return logits


CONTEXTS = [(37 * i) % 1200 + 1 for i in range(99)]


@pytest.mark.parametrize("portions", [[], [40], [150, 90]])
def test_a_step_of_many_requests_beside_a_longer_one(portions):
    """The same through whole steps: 200 pairs, alone and beside prompt portions (whose launch attends them where contexts are short)."""
    got = [_many(portions, CONTEXTS + [longest], 3100, False)[:-1] for longest in (1000, 1400, 3000)]
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("portions", [[], [40]])
def test_a_replayed_step_of_many_requests_whatever_the_longest_there_may_be(portions):
    """A graph's kernels are chosen by the engine's limit, not by the contexts there are."""
    assert torch.equal(_many(portions, CONTEXTS, 1250, True), _many(portions, CONTEXTS, 3100, True))
