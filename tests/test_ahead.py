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


def _brought(width, heads, kv_heads, head_dim, inside, contexts, portions, graphs=False):
    """What a step of three layers is given to bring, and which kernels it takes (counters of the step program)."""
    from conftest import qwen2_config
    from tokenmill_amd import EngineConfig, LLMEngine
    from tokenmill_amd.config.registry import architecture_name, get_architecture
    from tokenmill_amd.engine.runner import StepEntry
    shape = qwen2_config(num_hidden_layers=3, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim,
                         intermediate_size=inside, vocab_size=16384, rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True)
    arch = get_architecture(architecture_name(shape))
    model = arch.build_model(arch.config_from_dict(shape, None), None)
    model.load({name: torch.full(spec.drawn_shape(), 0.01, dtype=torch.bfloat16, device="cuda") for name, spec in model.tensor_specs().items()},
               torch.bfloat16, torch.device("cuda:0"))
    requests = [(0, n) for n in portions] + [(c - 1, 1) for c in contexts]
    engine = LLMEngine(EngineConfig(dtype="bfloat16", block_size=16, num_blocks=sum(-(-(a + b) // 16) for a, b in requests) + 4, watermark=0.0,
                                    max_model_len=2200, max_num_seqs=128, max_num_batched_tokens=4096, hip_graphs=graphs), model=model)
    entries = [StepEntry(engine.cache.allocate(f"r{i}", a + b), a, [1] * b, [b - 1]) for i, (a, b) in enumerate(requests)]
    program = engine.runner.program
    before = program.brought(), program.counters()
    for _ in range(3 if graphs else 1):
        engine.runner.step(entries)
    after = program.brought(), program.counters()
    return [{k: n - b[k] for k, n in a.items() if n != b[k]} for a, b in zip(after, before)]


SMALL, WIDE_QKV, LARGE = (896, 14, 2, 64, 4864), (1024, 16, 8, 128, 3072), (1536, 12, 2, 128, 8960)
NORM = {"qkv_from_norm": 3, "gate_up_from_norm": 3, "head_few": 1}
TILED = {"qkv_plain": 3, "qkv_tiled": 3, "gate_up_plain": 3, "gate_up_tiled": 3, "project_tiled": 6, "head_few": 1}


@pytest.mark.gpu
@pytest.mark.parametrize("shape,contexts,portions,brought,kernels", [
    # q|k|v: half of gate|up; attention: o and the rest; gate|up: down and the next q|k|v
    (SMALL, [300], [], {"qkv": 3, "attention": 6, "gate_up": 5}, {**NORM, "decode_whole": 3}),
    (SMALL, [300] * 8, [], {"qkv": 3, "attention": 6, "gate_up": 5}, {**NORM, "decode_whole": 3}),
    (SMALL, [2100] * 4, [], {"qkv": 3, "attention": 6, "gate_up": 5}, NORM),
    # q|k|v has no CU to spare, gate|up room for down alone
    (WIDE_QKV, [300], [], {"attention": 3, "gate_up": 3}, {**NORM, "decode_whole": 3}),
    (LARGE, [300], [], {}, {**NORM, "decode_whole": 3}),
    # attention: o and down; gate|up too where it is one launch
    (SMALL, [90] * 12, [], {"attention": 9}, {"qkv_panel": 3, "gate_up_stream": 3, "head_few": 1, "decode_whole": 3}),
    (SMALL, [50] * 33, [], {"attention": 9, "row_major": 9}, {"qkv_panel": 3, "gate_up_plain": 3, "gate_up_tiled": 3, "project_tiled": 6, "decode_whole": 3}),
    (SMALL, [1500] * 24, [], {"attention": 6, "row_major": 6}, {"qkv_panel": 3, "gate_up_plain": 3, "gate_up_tiled": 3, "project_tiled": 6}),
    (SMALL, [], [30], {"attention": 6, "row_major": 6},
     {"qkv_panel": 3, "gate_up_plain": 3, "gate_up_tiled": 3, "project_tiled": 6, "prefill_split_keys": 3, "head_few": 1}),
    # q|k|v's tiles: o and gate|up; attention: down and the next q|k|v
    (SMALL, [], [77], {"qkv": 6, "attention": 5, "row_major": 11}, {**TILED, "prefill_split_keys": 3}),
    (SMALL, [300] * 10, [241, 241], {"qkv": 6, "attention": 5, "row_major": 11}, {**TILED, "prefill_split_keys": 3, "decode_beside": 3}),
    (SMALL, [1800] * 10, [241, 241], {"attention": 11, "row_major": 11}, {**TILED, "prefill_split_keys": 3}),
    (LARGE, [], [77], {}, {**TILED, "prefill_split_keys": 3}),
])
def test_which_matrices_a_step_brings_and_which_kernels_take_them(shape, contexts, portions, brought, kernels):
    """Each matrix is brought in the order of the kernel that takes it: row-major ones are the tiled products'."""
    got, took = _brought(*shape, contexts, portions)
    assert got == brought and took == kernels


@pytest.mark.gpu
def test_a_captured_step_brings_what_an_eager_one_does():
    got, took = _brought(*SMALL, [300] * 4, [], graphs=True)
    runs = took["qkv_from_norm"]                                             # (layers of the runs that a capture makes)
    assert runs >= 3 and got == {"qkv": runs, "attention": 2 * runs, "gate_up": 5 * runs // 3}


@pytest.mark.gpu
@pytest.mark.parametrize("width,heads,requests,few", [(896, 14, 16, 1), (896, 14, 17, 0), (3200, 25, 8, 1), (3200, 25, 9, 0)])
def test_which_heads_the_kernel_of_few_rows_takes(width, heads, requests, few):
    """Beyond eight rows a narrow head with a long K is the library's."""
    _, took = _brought(width, heads, 1, width // heads, 512, [20] * requests, [])
    assert took.get("head_few", 0) == few
