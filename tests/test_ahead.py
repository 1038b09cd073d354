"""Matrices brought ahead of the products that read them (csrc/ahead.h): every line once, by the die whose blocks read it (on the host), and
a step's bits with and without it."""
import ctypes

import pytest
import torch


def _runs(strip_bytes, units, two, blocks, first, last, head_units, rot_heads, die):
    from tokenmill_amd.hip.abi import bound
    room = 1 << 16
    strips, runs = (ctypes.c_int * room)(), (ctypes.c_int * room)()
    n = bound().tm_ahead_runs(*(ctypes.c_int(x) for x in (strip_bytes, units, two, blocks, first, last, head_units, rot_heads, die)), strips, runs, ctypes.c_int(room))
    assert n >= 0
    return list(zip(strips[:n], runs[:n]))


# (bytes of a strip, units, two strips a unit, blocks of the product, units of a head, heads of q and k)
@pytest.mark.parametrize("strip_bytes,units,two,blocks,head_units,rot_heads", [
    (28672, 304, 1, 152, 0, 0), (7168, 224, 0, 224, 0, 0), (38912, 224, 0, 224, 0, 0), (14336, 72, 1, 72, 4, 16), (8192, 1, 0, 1, 0, 0), (64, 9, 0, 9, 0, 0),
    (8256, 13, 1, 5, 0, 0), (16384, 257, 1, 129, 0, 0), (24576, 700, 1, 234, 0, 0), (1024, 30, 1, 30, 2, 11)])
def test_every_line_is_brought_once_by_the_die_that_reads_it(strip_bytes, units, two, blocks, head_units, rot_heads):
    rounds = -(-units // blocks)
    want = {}                                            # strip -> the die of the block that multiplies it
    for u in range(units):
        if head_units:
            head, jt = divmod(u, head_units)
            pair = (head * 2 * head_units + jt, head * 2 * head_units + head_units + jt) if head < rot_heads else (head * 2 * head_units + 2 * jt, head * 2 * head_units + 2 * jt + 1)
        else:
            pair = (u, units + u) if two else (u,)
        for strip in pair:
            want[strip] = u % blocks % 8
    seen = {}
    for first, last in {(0, 1), (1, rounds)} if rounds > 1 else {(0, rounds)}:
        for die in range(8):
            for strip, run in _runs(strip_bytes, units, two, blocks, first, last, head_units, rot_heads, die):
                assert (strip, run) not in seen and want[strip] == die
                seen[strip, run] = die
    assert len(seen) == len(want) * -(-strip_bytes // 8192)
    assert all(0 <= run and run * 8192 < strip_bytes for _, run in seen)


@pytest.mark.gpu
@pytest.mark.parametrize("width,heads,kv_heads,inside,layers", [(896, 14, 2, 4864, 3), (512, 8, 2, 1400, 3), (256, 4, 4, 5000, 2), (1024, 8, 1, 4096, 2)])
@pytest.mark.parametrize("contexts", [[1], [300, 17, 256], [40] * 8, [700, 5, 2100, 64, 513]])
def test_a_step_has_the_bits_of_its_operations_one_by_one(width, heads, kv_heads, inside, layers, contexts):
    """Operations run one by one know no operation behind them, so nothing is brought ahead."""
    from conftest import qwen2_config
    from tokenmill_amd import EngineConfig, LLMEngine
    from tokenmill_amd.config.registry import architecture_name, get_architecture
    from tokenmill_amd.engine.runner import StepEntry
    from tokenmill_amd.hip.program import Flow
    shape = qwen2_config(num_hidden_layers=layers, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads,
                         intermediate_size=inside, vocab_size=512, rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True)
    arch = get_architecture(architecture_name(shape))
    model = arch.build_model(arch.config_from_dict(shape, None), None)
    g = torch.Generator(device="cuda").manual_seed(1)
    tensors = {name: (torch.randn(spec.drawn_shape(), generator=g, device="cuda") * 0.02).bfloat16() for name, spec in sorted(model.tensor_specs().items())}
    model.load(tensors, torch.bfloat16, torch.device("cuda:0"))
    engine = LLMEngine(EngineConfig(dtype="bfloat16", block_size=16, num_blocks=sum(-(-c // 16) for c in contexts) + 4, watermark=0.0, max_model_len=2200,
                                    max_num_seqs=16, max_num_batched_tokens=4096, hip_graphs=False), model=model)
    caches = [engine.cache.allocate(f"r{i}", c) for i, c in enumerate(contexts)]
    ids = [torch.randint(0, 512, (c,), generator=torch.Generator().manual_seed(c)).tolist() for c in contexts]
    for cache, prompt in zip(caches, ids):
        if len(prompt) > 1:
            engine.runner.step([StepEntry(cache, 0, prompt[:-1], [len(prompt) - 2])])
    step = engine.runner.prepare([StepEntry(cache, len(prompt) - 1, prompt[-1:], [0]) for cache, prompt in zip(caches, ids)])[0]
    program = engine.runner.program
    before = program.counters()
    want = program.run(step).clone()
    assert program.counters()["gate_up_from_norm"] - before["gate_up_from_norm"] == layers
    T = step.num_tokens
    flow = Flow(resid=torch.empty((T, width), dtype=torch.float32, device="cuda"), accumulate=True)
    flow.logits = torch.empty((T, 512), dtype=torch.float32, device="cuda")
    (native,) = program.steps
    for op in range(native.first, native.first + native.count):
        program.run_ops(op, 1, step, flow)
    assert torch.equal(flow.logits, want)
