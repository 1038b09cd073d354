"""Matrices brought ahead of the products that read them (csrc/ahead.h): every line once, by the die whose blocks read it (on the host), and
a step's bits with and without it."""
import ctypes

import pytest
import torch


def _lines(name, *args):
    from tokenmill_amd.hip.abi import bound
    room = 1 << 20
    at = (ctypes.c_longlong * room)()
    n = getattr(bound(), name)(*(ctypes.c_int(x) for x in args), at, ctypes.c_int(room))
    assert n >= 0
    return at[:n]


# (bytes of a strip, units, two strips a unit, blocks of the product, neighbours to a block, units of a head, heads of q and k)
@pytest.mark.parametrize("strip_bytes,units,two,blocks,together,head_units,rot_heads", [
    (28672, 304, 1, 152, 0, 0, 0), (28672, 304, 1, 152, 1, 0, 0), (7168, 224, 0, 224, 0, 0, 0), (38912, 224, 0, 224, 0, 0, 0), (14336, 72, 1, 72, 0, 4, 16),
    (8192, 1, 0, 1, 0, 0, 0), (64, 9, 0, 9, 0, 0, 0), (8256, 13, 1, 5, 0, 0, 0), (8256, 13, 1, 5, 1, 0, 0), (16384, 257, 1, 129, 0, 0, 0),
    (24576, 700, 1, 234, 0, 0, 0), (1024, 30, 1, 30, 0, 2, 11)])
def test_every_line_of_a_packed_matrix_is_brought_once_by_the_die_that_reads_it(strip_bytes, units, two, blocks, together, head_units, rot_heads):
    rounds = -(-units // blocks)
    want = {}                                            # strip -> the die of the block that multiplies it
    for u in range(units):
        if head_units:
            head, jt = divmod(u, head_units)
            pair = (head * 2 * head_units + jt, head * 2 * head_units + head_units + jt) if head < rot_heads else (head * 2 * head_units + 2 * jt, head * 2 * head_units + 2 * jt + 1)
        else:
            pair = (u, units + u) if two else (u,)
        for strip in pair:
            want[strip] = (u // rounds if together else u % blocks) % 8
    seen = set()
    for first, last in {(0, 1), (1, rounds)} if rounds > 1 else {(0, rounds)}:
        for die in range(8):
            for at in _lines("tm_ahead_packed", strip_bytes, units, two, blocks, together, first, last, head_units, rot_heads, die):
                strip, off = divmod(at, strip_bytes)
                assert at not in seen and want[strip] == die and off % 128 == 0
                seen.add(at)
    assert len(seen) == len(want) * -(-strip_bytes // 128)


# (rows of a half, K, rows of a column tile, parts of K, 64 k a part, halves)
@pytest.mark.parametrize("row_end,K,rows,parts,lines,two", [(4864, 896, 32, 1, 14, 1), (896, 4864, 64, 4, 19, 0), (896, 4864, 64, 5, 16, 0), (896, 896, 64, 2, 7, 0),
                                                            (1152, 896, 64, 1, 14, 0), (1400, 512, 32, 1, 8, 1), (100, 256, 128, 1, 4, 0), (72, 320, 64, 1, 5, 1)])
def test_every_line_of_a_row_major_matrix_is_brought_once(row_end, K, rows, parts, lines, two):
    seen, all_lines, tiles = set(), K // 64, -(-row_end // rows)
    for die in range(8):
        for at in _lines("tm_ahead_row_major", row_end, K, rows, parts, lines, two, die):
            line, off = divmod(at, 128)
            assert off == 0 and 0 <= line < (1 + two) * row_end * all_lines and at not in seen
            row, k = divmod(line, all_lines)
            column = k // lines * tiles + row % row_end // rows             # in the order of the product's tiles, of which a die has a run
            assert die * tiles * parts // 8 <= column < (die + 1) * tiles * parts // 8
            seen.add(at)
    assert len(seen) == (1 + two) * row_end * all_lines


@pytest.mark.gpu
@pytest.mark.parametrize("width,heads,kv_heads,inside,layers", [(896, 14, 2, 4864, 3), (512, 8, 2, 1400, 3), (256, 4, 4, 5000, 2), (1024, 8, 1, 4096, 2)])
@pytest.mark.parametrize("contexts,portions", [([1], []), ([300, 17, 256], []), ([40] * 8, []), ([700, 5, 2100, 64, 513], []), ([90] * 12, []), ([300, 600] * 8, []),
                                               ([50] * 33, []), ([], [30]), ([], [77]), ([], [150, 90]), ([], [600]), ([20, 700], [100]), ([300] * 10, [241, 241])])
def test_a_step_has_the_bits_of_its_operations_one_by_one(width, heads, kv_heads, inside, layers, contexts, portions):
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
    requests = [(0, n) for n in portions] + [(c - 1, 1) for c in contexts]            # (cached tokens, tokens of the step)
    engine = LLMEngine(EngineConfig(dtype="bfloat16", block_size=16, num_blocks=sum(-(-(a + b) // 16) for a, b in requests) + 4, watermark=0.0,
                                    max_model_len=2200, max_num_seqs=64, max_num_batched_tokens=4096, hip_graphs=False), model=model)
    caches = [engine.cache.allocate(f"r{i}", a + b) for i, (a, b) in enumerate(requests)]
    ids = [torch.randint(0, 512, (a + b,), generator=torch.Generator().manual_seed(a + b)).tolist() for a, b in requests]
    for cache, prompt, (a, _) in zip(caches, ids, requests):
        if a:
            engine.runner.step([StepEntry(cache, 0, prompt[:a], [a - 1])])
    step = engine.runner.prepare([StepEntry(cache, a, prompt[a:], [b - 1]) for cache, prompt, (a, b) in zip(caches, ids, requests)])[0]
    program = engine.runner.program
    want = program.run(step).clone()
    T, R = step.num_tokens, step.num_logit_rows
    flow = Flow(resid=torch.empty((T, width), dtype=torch.float32, device="cuda"), accumulate=True)
    flow.logits = torch.empty((R, 512), dtype=torch.float32, device="cuda")
    (native,) = program.steps
    for op in range(native.first, native.first + native.count):
        program.run_ops(op, 1, step, flow)
    assert torch.equal(flow.logits, want)
