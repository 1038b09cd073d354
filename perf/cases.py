"""What this engine is timed on: steps of a server's life, through the engine's own step function.

A case is one step: requests that decode a token over a context they have, and portions of prompts. ``prepare`` has what a
server has before the step (a loaded model, an engine, requests whose earlier tokens are in the cache, graphs of the shape),
``run`` is the step and the sampling that follows it, as ``LLMEngine.step`` makes them: ``ModelRunner.step(entries)`` and
``Sampler.start(...)``, whose tokens stay on the device (the next step may be queued behind them). A step runs at the same
positions every time it is repeated: it writes the same keys and values to the same places of the cache.

    shape            a shipped configuration (tokenmill_amd/config/shapes)
    dtype            bfloat16, or float32 (the true 32-bit path)
    decodes          requests that decode one token each
    context          the longest of their contexts; with "ragged" they go down to half of it, as in a server's batch
    portions         prompt portions, of ``tokens`` tokens each, behind ``before`` tokens of their prompts that are cached
    temperature, top_k, top_p     how the step's tokens are drawn (temperature 0: greedy)
"""
from __future__ import annotations

import math

import torch

from tokenmill_amd import EngineConfig, LLMEngine, SamplingParams
from tokenmill_amd.config.registry import architecture_name, get_architecture
from tokenmill_amd.config.shapes import read_shape
from tokenmill_amd.engine.runner import StepEntry

PAGE = 16
FILL_TOKENS = 4096          # tokens a step that fills the cache may hold
GAIN = 0.6                  # of a product with a normed input: weights of 0.02 at the small model's width, less at larger ones
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


def _case(shape="qwen2.5-0.5b", dtype="bfloat16", decodes=0, context=0, ragged=False, portions=0, tokens=0, before=0,
          temperature=0.0, top_k=-1, top_p=1.0) -> dict:
    return dict(shape=shape, dtype=dtype, decodes=decodes, context=context, ragged=ragged, portions=portions, tokens=tokens,
                before=before, temperature=temperature, top_k=top_k, top_p=top_p)


def listed() -> list[dict]:
    return [
        # one user chatting with the small model: the smallest step, launches and latency
        dict(_case(decodes=1, context=300), name="decode-1"),
        # the headline of bench.py: eight requests that have read prompts of 2,048 tokens
        dict(_case(decodes=8, context=2048), name="decode-8"),
        # a full server: 64 requests of different lengths (an odd longest), sampled
        dict(_case(decodes=64, context=1021, ragged=True, temperature=0.8, top_k=50, top_p=0.95), name="decode-64-sampled"),
        # a few long documents being answered
        dict(_case(decodes=4, context=16000, ragged=True), name="decode-4-long"),
        # the large model at the headline's batch: its matrices dwarf everything else
        dict(_case("qwen2.5-7b", decodes=8, context=2048), name="decode-8-7b"),
        # a chat message arrives: time to the first token of a short prompt of an odd length
        dict(_case(portions=1, tokens=77), name="prompt-77"),
        # the headline prompt of bench.py
        dict(_case(portions=1, tokens=2048), name="prompt-2048"),
        # a document for the large model, no multiple of anything
        dict(_case("qwen2.5-7b", portions=1, tokens=3001), name="prompt-3001-7b"),
        # a chunked-prefill step: two portions behind what is cached of their prompts, beside decoding requests
        dict(_case(decodes=30, context=1000, ragged=True, portions=2, tokens=241, before=482), name="mixed-512"),
        # the true 32-bit path, both directions; decoding is sampled, and its tokens are compared too
        dict(_case(dtype="float32", decodes=8, context=700, temperature=0.7, top_p=0.9), name="decode-8-float32"),
        dict(_case(dtype="float32", portions=1, tokens=1000), name="prompt-1000-float32"),
        # another design: latent attention in a window, convolutions with state, layer norms, gates, experts by token id
        dict(_case("lusolix-2k", portions=1, tokens=1500), name="prompt-1500-lusolix"),
    ]


def draw(rng) -> dict:
    def log_uniform(lo, hi):
        return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    what = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "mixed", "float32", "lusolix"])
    sampling = rng.choice([{}, {}, dict(temperature=round(rng.uniform(0.3, 1.2), 2), top_k=rng.choice([-1, 20, 50]),
                                        top_p=rng.choice([1.0, 0.9, 0.95]))])
    ragged = rng.random() < 0.5
    if what == "decode":
        large = rng.random() < 0.3
        n = log_uniform(1, 32 if large else 64)
        context = log_uniform(50, min(16000, (20000 if large else 70000) // n))
        return _case("qwen2.5-7b" if large else "qwen2.5-0.5b", decodes=n, context=context, ragged=ragged, **sampling)
    if what == "prompt":
        large = rng.random() < 0.3
        return _case("qwen2.5-7b" if large else "qwen2.5-0.5b", portions=1, tokens=log_uniform(16, 2800 if large else 8000),
                     before=rng.choice([0, 0, rng.randint(1, 1500)]))
    if what == "mixed":
        return _case(decodes=log_uniform(2, 60), context=log_uniform(50, 1500), ragged=ragged, portions=rng.randint(1, 4),
                     tokens=log_uniform(16, 400), before=rng.choice([0, rng.randint(1, 1000)]), **sampling)
    if what == "float32":
        if rng.random() < 0.5:
            return _case(dtype="float32", decodes=log_uniform(1, 16), context=log_uniform(50, 1500), ragged=ragged, **sampling)
        return _case(dtype="float32", portions=1, tokens=log_uniform(16, 1500))
    return _case("lusolix-2k", portions=1, tokens=log_uniform(32, 1700))


# --- the model's numbers and a case's requests ---------------------------------------------------------

def _requests(case: dict) -> list[tuple[int, int]]:
    """(cached tokens, tokens of the step) of every request."""
    n, c = case["decodes"], case["context"]
    contexts = [c - (c // 2) * i // max(n - 1, 1) if case["ragged"] else c for i in range(n)]
    return [(case["before"], case["tokens"])] * case["portions"] + [(x, 1) for x in contexts]


def _prompts(case: dict, seed: int) -> list[list[int]]:
    g = torch.Generator().manual_seed(seed)
    shape = read_shape(case["shape"])
    vocab = shape.get("vocab_size", shape.get("vocab"))
    return [torch.randint(0, vocab, (a + b,), generator=g).tolist() for a, b in _requests(case)]


def _tensors(case: dict):
    """The model (nothing loaded) and its random weights: normal, norms about one, tables of experts. The width's root in the
    deviation keeps the larger model as well-conditioned as the small one, as training does."""
    shape, dtype = read_shape(case["shape"]), DTYPES[case["dtype"]]
    arch = get_architecture(architecture_name(shape))
    model = arch.build_model(arch.config_from_dict(shape, None), None)
    g = torch.Generator(device="cuda").manual_seed(1)
    tensors = {}
    for name, spec in sorted(model.tensor_specs().items()):
        size = spec.drawn_shape()
        if spec.kind == "int":          # rows of different expert numbers
            below = int(spec.init.split(":")[1])
            tensors[name] = torch.rand(size[0], below, generator=g, device="cuda").argsort(1)[:, :size[1]].int().contiguous()
            continue
        t = torch.empty(size, dtype=torch.float32, device="cuda").normal_(generator=g)
        if spec.init == "ones":
            t = 1 + 0.1 * t
        else:
            t *= GAIN / math.sqrt(shape.get("hidden_size", shape.get("width")))
        tensors[name] = t.to(dtype)
    return model, tensors


_loaded: dict = {}          # the model a server holds: one at a time, the same for every batch it is given


def _model(case: dict):
    key = (case["shape"], case["dtype"])
    if key not in _loaded:
        _loaded.clear()
        model, tensors = _tensors(case)
        model.load(tensors, DTYPES[case["dtype"]], torch.device("cuda:0"))
        _loaded[key] = model
    return _loaded[key]


# --- a step --------------------------------------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    requests, prompts = _requests(case), _prompts(case, seed)
    longest = max(a + b for a, b in requests)
    pages = sum(-(-(a + b) // PAGE) for a, b in requests)
    engine = LLMEngine(EngineConfig(dtype=case["dtype"], block_size=PAGE, num_blocks=pages, watermark=0.0,
                                    max_model_len=longest + 64, max_num_seqs=len(requests),
                                    max_num_batched_tokens=FILL_TOKENS, hip_graphs=True), model=_model(case))
    entries, fill, room = [], [], FILL_TOKENS
    caches = [engine.cache.allocate(f"r{i}", a + b) for i, (a, b) in enumerate(requests)]

    def filled():
        if fill:
            engine.runner.forward(engine.runner.prepare(fill)[0])
            fill.clear()

    for rc, ids, (a, b) in zip(caches, prompts, requests):
        for at in range(0, a, FILL_TOKENS):                 # what the request has read before this step
            part = ids[at:min(a, at + FILL_TOKENS)]
            if len(part) > room:
                filled()
                room = FILL_TOKENS
            fill.append(StepEntry(rc, at, part))
            room -= len(part)
            if at + FILL_TOKENS < a:                        # the next portion of this request needs this one's keys
                filled()
                room = FILL_TOKENS
        entries.append(StepEntry(rc, a, ids[a:], [b - 1]))
    filled()
    params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"])
    state = {"engine": engine, "entries": entries, "params": [params] * len(entries),
             "seeds": [seed + i for i in range(len(entries))], "counters": [0] * len(entries),
             "whole_prompts": bool(engine.pools.states), "tokens_too": case["dtype"] == "float32"}
    for _ in range(4):                                      # a server has run steps of this shape: its graph is there
        run(state)
    torch.cuda.synchronize()
    return state


@torch.inference_mode()
def run(state: dict) -> dict:
    """The step's logits and, as updated state, the cache (every page belongs to the case's requests). In bfloat16 the sampled tokens
    are left out: random weights give nearly equal logits, and a last bit decides which of them is the largest."""
    engine = state["engine"]
    if state["whole_prompts"]:                              # a request that comes in: its state starts from zero
        for e in state["entries"]:
            e.cache.fresh = True
    logits = engine.runner.step(state["entries"])
    drawn = engine.sampler.start(logits, state["params"], state["seeds"], state["counters"])
    out = {"logits": logits}
    if state["tokens_too"]:
        out["tokens"] = drawn.device
    if not state["whole_prompts"]:
        out["keys"], out["values"] = engine.pools.k[0], engine.pools.v[0]
    return out


# --- what a step cannot do without ------------------------------------------------------------------------

def work(case: dict) -> dict:
    c = read_shape(case["shape"])
    size = 4 if case["dtype"] == "float32" else 2
    requests = _requests(case)
    rows, wanted = sum(b for _, b in requests), len(requests)
    pairs = sum(b * a + b * (b + 1) // 2 for a, b in requests)          # (query, key) pairs
    if "width" in c:
        return _work_lusolix(c, size, rows, wanted, requests)
    hidden, layers, inter, vocab = c["hidden_size"], c["num_hidden_layers"], c["intermediate_size"], c["vocab_size"]
    heads, kv = c["num_attention_heads"], c["num_key_value_heads"]
    d = hidden // heads
    matrices = layers * (hidden * d * (2 * heads + 2 * kv) + 3 * hidden * inter)
    kv_row = layers * 2 * kv * d * size
    return {"bytes": size * (matrices + vocab * hidden + rows * hidden) + kv_row * sum(a + b for a, b in requests) + kv_row * rows
            + 4 * wanted * vocab,
            "flops": 2 * rows * matrices + 2 * wanted * vocab * hidden + 4 * layers * heads * d * pairs}


def _work_lusolix(c: dict, size: int, rows: int, wanted: int, requests) -> dict:
    W, vocab, nbytes, flops = c["width"], c["vocab"], 0, 0
    for layer in c["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        H, Dn, Dr, Dv, Lq, Lk = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["q_rank"], m["kv_rank"]
        window = m["mask"]["size"]
        pairs = sum(sum(min(a + t + 1, window) for t in range(b)) for a, b in requests)
        shared = W * (Lq + Lk + Dr + H) + Lq * H * (Dn + Dr) + H * Dv * W + 2 * W * W
        per_head = H * (Dn + Dv) * Lk
        if f["kind"] == "dense":
            every, used = 2 * W * f["ff"], 2 * W * f["ff"]
        else:
            e = 3 * W * f["expert"]["ff"]
            every, used = e * min(f["router"]["experts"], rows * f["router"]["top"]), e * f["router"]["top"]
        nbytes += size * (shared + per_head + every + 2 * rows * (Lk + Dr))
        # keys and values per head from the latents: once a row, the cheaper of the two orders for a prompt
        flops += 2 * rows * (shared + per_head + used) + 2 * pairs * H * (Dn + Dr + Dv)
    return {"bytes": nbytes + size * (vocab * W + 2 * rows * W) + 4 * wanted * vocab, "flops": flops + 2 * wanted * vocab * W}


def tolerance(case: dict) -> dict:
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    # the same step over other kernels (no packed matrices) differs by up to 0.010, 0.064 at most, with one token's path rounded otherwise
    return {"rel": 0.03, "max": 0.3}


# --- the same in 64 bits ------------------------------------------------------------------------------------

@torch.inference_mode()
def exact(case: dict, seed: int) -> dict | None:
    shape = read_shape(case["shape"])
    _, t = _tensors(case)
    if "width" in shape:
        return {"logits": torch.cat([_lusolix(shape, t, ids)[-1:] for ids in _prompts(case, seed)])}
    cost = work(case)["flops"] / max(1, sum(b for _, b in _requests(case))) * sum(a + b for a, b in _requests(case))
    if cost > 6e14:
        return None
    heads, kv = shape["num_attention_heads"], shape["num_key_value_heads"]
    d, layers = shape["hidden_size"] // heads, shape["num_hidden_layers"]
    requests = _requests(case)
    held = [-(-(a + b) // PAGE) for a, b in requests]
    keys = torch.zeros(layers, sum(held), PAGE, kv, d, dtype=torch.float32, device="cuda")
    values = torch.zeros(layers, sum(held), kv, d, PAGE, dtype=torch.float32, device="cuda")
    logits, page = [], 0
    for ids, n in zip(_prompts(case, seed), held):
        def stored(layer, k, v, page=page, n=n):
            """[tokens, kv, d] into the request's pages (an engine that is new gives them out in their order)."""
            pad = n * PAGE - k.shape[0]
            k, v = (torch.nn.functional.pad(x, (0, 0, 0, 0, 0, pad)).view(n, PAGE, kv, d) for x in (k, v))
            keys[layer, page:page + n], values[layer, page:page + n] = k, v.permute(0, 2, 3, 1)
        logits.append(_qwen2(shape, t, ids, stored))
        page += n
    out = {"logits": torch.cat(logits), "keys": keys, "values": values}
    if case["dtype"] == "float32":
        out["tokens"] = None
    return out


def _rms(x, w, eps):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _causal(q, k, v, scale, window=None):
    """q [T, H, D], k and v [T, H, *] of whole sequences, a head and a run of queries at a time."""
    T, H = q.shape[:2]
    out = torch.empty(T, H, v.shape[2], dtype=torch.float64, device=q.device)
    place = torch.arange(T, device=q.device)
    for h in range(H):
        for lo in range(0, T, 2048):
            hi = min(T, lo + 2048)
            s = (q[lo:hi, h] @ k[:hi, h].T) * scale
            far = place[lo:hi, None] - place[None, :hi]
            s.masked_fill_((far < 0) | (far >= (window or T)), float("-inf"))
            out[lo:hi, h] = torch.softmax(s, -1) @ v[:hi, h]
    return out.flatten(1)


def _qwen2(c: dict, t: dict, ids: list[int], stored) -> torch.Tensor:
    """Logits [1, vocab] of the last token; ``stored(layer, keys, values)`` is given what the layer caches."""
    heads, kv, eps = c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"]
    d = c["hidden_size"] // heads
    T = len(ids)
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * c["rope_theta"] ** (
        -torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turned(x):
        a, b = x.chunk(2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def linear(x, name):
        y = x @ t[name + ".weight"].double().T
        return y + t[name + ".bias"].double() if name + ".bias" in t else y

    x = t["model.embed_tokens.weight"][torch.tensor(ids, device="cuda")].double()
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        n = _rms(x, t[p + "input_layernorm.weight"], eps)
        q = turned(linear(n, p + "self_attn.q_proj").view(T, heads, d))
        k = turned(linear(n, p + "self_attn.k_proj").view(T, kv, d))
        v = linear(n, p + "self_attn.v_proj").view(T, kv, d)
        stored(i, k, v)
        k, v = (y.repeat_interleave(heads // kv, 1) for y in (k, v))
        x = x + linear(_causal(q, k, v, d ** -0.5), p + "self_attn.o_proj")
        n = _rms(x, t[p + "post_attention_layernorm.weight"], eps)
        g = torch.nn.functional.silu(linear(n, p + "mlp.gate_proj"))
        x = x + linear(g.mul_(linear(n, p + "mlp.up_proj")), p + "mlp.down_proj")
    head = t.get("lm_head.weight", t["model.embed_tokens.weight"])
    return _rms(x[-1:], t["model.norm.weight"], eps) @ head.double().T


def _lusolix(c: dict, t: dict, ids: list[int]) -> torch.Tensor:
    """Logits [1, vocab] of the last token of a whole prompt."""
    ids = torch.tensor(ids, device="cuda")
    T, eps = ids.numel(), c["norm"]["eps"]
    place = torch.arange(T, device="cuda", dtype=torch.float64)

    def linear(x, name):
        return x @ t[name].double().T

    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, t[name], eps) + t[name + ".b"].double()

    def gate(x, name):
        return c["residual_mult"] * torch.sigmoid(linear(x, name) + t[name + ".b"].double())

    def turned(x, rot):
        dims = rot["dims"]
        angle = place[:, None] * rot["base"] ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]
        out = x.clone()
        a, b = x[..., 0:dims:2], x[..., 1:dims:2]
        out[..., 0:dims:2], out[..., 1:dims:2] = a * cos - b * sin, b * cos + a * sin
        return out

    def mixed(u, m, p):
        H, Dn, Dr, Dv, Lk = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q = linear(_rms(linear(u, p + "dq"), t[p + "dq.norm"], eps), p + "uq").view(T, H, Dn + Dr)
        low = linear(u, p + "dkv")
        latent = _rms(low[:, :Lk], t[p + "dkv.norm"], eps)
        k = (latent @ t[p + "uk"].double().reshape(H * Dn, Lk).T).view(T, H, Dn)
        v = (latent @ t[p + "uv"].double().reshape(H * Dv, Lk).T).view(T, H, Dv)
        shared = turned(low[:, None, Lk:], m["rot"]).expand(T, H, Dr)
        q = torch.cat([q[..., :Dn], turned(q[..., Dn:], m["rot"])], -1)
        o = _causal(q, torch.cat([k, shared], -1), v, m["scale"], m["mask"]["size"])
        return linear((o.view(T, H, Dv) * torch.sigmoid(linear(u, p + "g"))[..., None]).flatten(1), p + "o")

    def fed(n, f, p):
        if f["kind"] == "dense":
            z, (a, b, e, const) = linear(n, p + "up"), t[p + "act"].double()
            return linear(a * _rms(z, None, eps) + b * _rms(z * z, None, eps) + e * _rms(z ** 3, None, eps) + const, p + "down")
        chosen = t[p + "table"].long()[ids]
        out = torch.zeros_like(n)
        for e in range(f["router"]["experts"]):
            rows = (chosen == e).any(1).nonzero()[:, 0]
            h = torch.nn.functional.silu(linear(n[rows], f"{p}e{e}.gate")) * linear(n[rows], f"{p}e{e}.up")
            out[rows] += linear(h, f"{p}e{e}.down") / chosen.shape[1]
        return out

    x = t["embed"].double()[ids] + t["pos"].double()[:T]
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        n = norm(x, p + "norm1")
        taps = t[p + "canon1"].double()
        before = torch.nn.functional.pad(n, (0, 0, taps.shape[1] - 1, 0))
        u = n + sum(before[j:j + T] * taps[:, j] for j in range(taps.shape[1]))
        x = x + mixed(u, layer["mixer"], p + "mix.") * gate(n, p + "rg1")
        n = norm(x, p + "norm2")
        x = x + fed(n, layer["mlp"], p + "mlp.") * gate(n, p + "rg2")
    return norm(x[-1:], "final.norm") @ t["embed"].double().T
