"""Which kernels a step takes (csrc/step_program.hip by the rules of csrc/choose.h): one layer at widths on both sides of each rule,
steps of row counts on both sides of it, told by the program's counters."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def runner_of():
    """A runner over one layer of the given width, the last one kept."""
    from tokenmill_amd import EngineConfig, LLMEngine
    from tokenmill_amd.config.registry import architecture_name, get_architecture
    from conftest import qwen2_config
    held = {}

    def get(width, heads, kv_heads, inside, dtype):
        key = (width, heads, kv_heads, inside, dtype)
        if key not in held:
            held.clear()
            torch.cuda.empty_cache()
            shape = qwen2_config(num_hidden_layers=1, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads,
                                 intermediate_size=inside, vocab_size=128, rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True)
            arch = get_architecture(architecture_name(shape))
            model = arch.build_model(arch.config_from_dict(shape, None), None)
            dt = getattr(torch, dtype)
            g = torch.Generator(device="cuda").manual_seed(1)
            tensors = {name: (torch.randn(spec.drawn_shape(), generator=g, device="cuda") * 0.02).to(dt)
                       for name, spec in sorted(model.tensor_specs().items())}
            model.load(tensors, dt, torch.device("cuda:0"))
            held[key] = LLMEngine(EngineConfig(dtype=dtype, block_size=16, num_blocks=128, watermark=0.0, max_model_len=512, max_num_seqs=128,
                                               max_num_batched_tokens=512, hip_graphs=False), model=model)
        return held[key]

    yield get
    held.clear()


def took(engine, requests):
    """The counters that one step of requests (cached tokens, tokens) moves."""
    from tokenmill_amd.engine.runner import StepEntry
    caches = [engine.cache.allocate(f"r{i}", a + b) for i, (a, b) in enumerate(requests)]
    if requests[0][0]:
        engine.runner.step([StepEntry(c, 0, [1] * a, [a - 1]) for c, (a, b) in zip(caches, requests)])
    before = engine.runner.program.counters()
    logits = engine.runner.step([StepEntry(c, a, [2] * b, [b - 1]) for c, (a, b) in zip(caches, requests)])
    assert logits.isfinite().all()
    for c in caches:
        engine.cache.free(c)
    return {k: n - before[k] for k, n in engine.runner.program.counters().items() if n != before[k] and not k.startswith(("prefill", "decode"))}


NORM = {"qkv_from_norm": 1, "gate_up_from_norm": 1}
TILED = {"qkv_plain": 1, "qkv_tiled": 1, "gate_up_plain": 1, "gate_up_tiled": 1, "project_tiled": 2}
GATE_UP = {"gate_up_plain": 1, "gate_up_tiled": 1}
BF16 = [
    # (width, heads, kv heads, inside), rows, what a prompt of so many tokens takes
    ((896, 14, 2, 4864), 8, NORM),
    ((896, 14, 2, 4864), 16, {"qkv_panel": 1, "gate_up_stream": 1}),
    ((896, 14, 2, 4864), 17, {"qkv_panel": 1, **GATE_UP, "project_tiled": 2}),
    ((896, 14, 2, 4864), 64, {"qkv_panel": 1, **GATE_UP, "project_tiled": 2}),
    ((896, 14, 2, 4864), 65, TILED),
    ((896, 14, 2, 4864), 300, TILED),
    ((2048, 16, 4, 8704), 16, {"qkv_stream": 1, "gate_up_stream": 1, "project_stream": 2}),
    ((2048, 16, 4, 8704), 17, {"qkv_stream": 1, "gate_up_stream": 1, "project_tiled": 2}),      # more columns than a tile a CU
    ((2048, 16, 4, 8704), 64, {"qkv_stream": 1, "gate_up_stream": 1, "project_tiled": 2}),
    ((2048, 16, 4, 8704), 65, TILED),
    ((2944, 23, 1, 2048), 16, {"qkv_stream": 1, "gate_up_stream": 1, "project_stream": 2}),
    ((3072, 24, 4, 2048), 4, NORM),
    ((3072, 24, 4, 2048), 5, {"qkv_stream": 1, "gate_up_stream": 1, "project_tiled": 2}),
    ((3072, 24, 4, 2048), 64, {"qkv_stream": 1, **GATE_UP, "project_tiled": 2}),
    ((4096, 32, 8, 2048), 4, {"qkv_stream": 1, "gate_up_stream": 1, "project_stream": 2}),
    ((4096, 32, 8, 2048), 5, {"qkv_stream": 1, "gate_up_stream": 1, "project_tiled": 2}),
    ((5120, 40, 8, 2048), 5, {"qkv_stream": 1, "gate_up_stream": 1, "project_stream": 2}),
    ((5120, 40, 8, 2048), 64, {"qkv_stream": 1, **GATE_UP, "project_stream": 2}),
    ((5120, 40, 8, 2048), 65, TILED),
]


@pytest.mark.parametrize("shape,rows,want", BF16)
def test_products_of_a_bfloat16_step(runner_of, shape, rows, want):
    assert took(runner_of(*shape, "bfloat16"), [(0, rows)]) == want


@pytest.mark.parametrize("rows,want", [(1, {"qkv_plain": 1, "qkv_few_f32": 1, "gate_up_plain": 1, "gate_up_few_f32": 1, "project_few_f32": 1}),
                                       (16, {"qkv_plain": 1, "qkv_few_f32": 1, "gate_up_plain": 1, "gate_up_few_f32": 1, "project_few_f32": 1}),
                                       (17, TILED), (300, TILED)])
def test_products_of_a_32_bit_step(runner_of, rows, want):
    assert took(runner_of(896, 14, 2, 4864, "float32"), [(0, rows)]) == want


@pytest.mark.parametrize("requests,split", [(1, 1), (95, 1), (96, 0)])
def test_attention_of_single_tokens_in_32_bit(runner_of, requests, split):
    """Below 192 pairs of request and kv head in chunks, beyond by the generic kernel."""
    engine = runner_of(896, 14, 2, 4864, "float32")
    before = engine.runner.program.counters()["decode_f32_split"]
    took(engine, [(4, 1)] * requests)
    assert engine.runner.program.counters()["decode_f32_split"] - before == split
