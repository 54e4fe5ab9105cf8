"""What the engine is timed on: steps of whole models through `ModelRunner.step`, and the sampler.

A case names a model (the layer sizes of a file under `configs/` and a dtype), what its steps look like, and sizes.  A program that serves keeps one runner and its captured graphs for as long as it lives, so the
runners here are kept by model; a state holds requests of its own in that runner's cache, and gives them back when it goes.
`run` feeds given tokens, as the trace-replay tool does, so every pass computes the same numbers: decoded tokens are taken
back out of the cache after the pass (`CacheManager.cancel`), prompts end with it.
"""

from __future__ import annotations

import itertools
import json
import math
import weakref
from pathlib import Path

import torch

from llmserve_amd import CacheConfig, GenerationConfig, ModelRunner, StepEntry, resolve_architecture
from llmserve_amd.cache.manager import Reservation
from llmserve_amd.kernels import HipKernels
from llmserve_amd.sampling import Sampler
from llmserve_amd.weights.loader import LoadedModel

DEVICE = "cuda:0"
PAGE = 16
SLOTS = 512
# file, dtype, cached tokens that all states together may hold
MODELS = {
    "qwen2.5-1.5b": ("qwen2.5-1.5b.json", "bfloat16", 1 << 19),
    "qwen2.5-1.5b float32": ("qwen2.5-1.5b.json", "float32", 1 << 17),
    "qwen2.5-7b": ("qwen2.5-7b.json", "bfloat16", 1 << 17),
    "dolezen-w1536": ("dolezen-w1536.json", "bfloat16", 1 << 17),
}
OUTSIDE = ("embed", "head", "model.embed_tokens.weight", "lm_head.weight")  # tensors outside the layers
STEPS = 4  # tokens that every request of a decode or mixed case brings, one a step


def listed():
    small, wide = "qwen2.5-1.5b", "qwen2.5-7b"
    return [
        # one user at a terminal, in the middle of an answer: the smallest step, where every launch counts
        {"name": "decode 1", "model": small, "kind": "decode", "requests": 1, "context": 640},
        # the benchmark's headline: eight requests of 512-token prompts half way through 256 outputs
        {"name": "decode 8", "model": small, "kind": "decode", "requests": 8, "context": 640},
        # a full batch of a busy server, contexts ragged around the same mean
        {"name": "decode 64", "model": small, "kind": "decode", "requests": 64, "context": 640},
        # eight requests over long documents: the cache is read more than the weights' products are
        {"name": "decode 8 long", "model": small, "kind": "decode", "requests": 8, "context": 8192},
        # the next larger layer sizes, untied head
        {"name": "decode 8 wide", "model": wide, "kind": "decode", "requests": 8, "context": 640},
        # the first token of a short question, an odd number of tokens
        {"name": "prompt 77", "model": small, "kind": "prompt", "length": 77, "portion": 2048},
        # the benchmark's prefill
        {"name": "prompt 2048", "model": small, "kind": "prompt", "length": 2048, "portion": 2048},
        # a long document in portions of the step's token budget
        {"name": "prompt 8191", "model": small, "kind": "prompt", "length": 8191, "portion": 2048},
        # continuous batching: a new prompt comes in portions beside 31 requests that decode
        {"name": "mixed 31+256", "model": small, "kind": "mixed", "requests": 31, "context": 500, "portion": 256},
        # the true 32-bit mode: a new prompt beside a few requests that decode
        {"name": "float32 mixed 3+126", "model": small + " float32", "kind": "mixed", "requests": 3, "context": 300, "portion": 126},
        # another architecture of the registry (latent attention, chunked attention with sinks, squared relu)
        {"name": "dolezen mixed 7+1024", "model": "dolezen-w1536", "kind": "mixed", "requests": 7, "context": 640, "portion": 1024},
        # temperature and top-p on the logits of a batch
        {"name": "sample 8", "model": small, "kind": "sample", "rows": 8, "temperature": 0.8, "top_p": 0.9},
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    model = rng.choices(list(MODELS), weights=(11, 3, 3, 3))[0]
    kind = rng.choices(("decode", "prompt", "mixed", "sample"), weights=(8, 5, 5, 2))[0]
    if kind == "sample":
        return {"model": "qwen2.5-1.5b", "kind": kind, "rows": _spread(rng, 1, 64), "temperature": round(rng.uniform(0.5, 1.5), 3),
                "top_p": rng.choice((1.0, round(rng.uniform(0.5, 0.99), 3)))}
    # what keeps a drawn case below the largest listed one: tokens a prompt, tokens cached beside it
    longest = {"qwen2.5-1.5b": 8192, "qwen2.5-1.5b float32": 512, "qwen2.5-7b": 2048, "dolezen-w1536": 3900}[model]
    cached = {"qwen2.5-1.5b": 65536, "qwen2.5-1.5b float32": 8192, "qwen2.5-7b": 16384, "dolezen-w1536": 16384}[model]
    if kind == "prompt":
        return {"model": model, "kind": kind, "length": _spread(rng, 3, longest), "portion": rng.choice((256, 512, 2048))}
    requests = _spread(rng, 1, 64 if kind == "decode" else 32)
    # (half as long again is the longest of the ragged contexts)
    context = _spread(rng, 24, min(cached // requests, 2 * longest // 3 if model == "dolezen-w1536" else 8192))
    case = {"model": model, "kind": kind, "requests": requests, "context": context}
    if kind == "mixed":
        case["portion"] = _spread(rng, 16, min(longest // STEPS, 1024))
    return case


# ---------------------------------------------------------------------------- models


def _read(model):
    file, dtype, held = MODELS[model]
    return json.loads((Path(__file__).resolve().parent.parent / "configs" / file).read_text()), getattr(torch, dtype), held


def _shapes(config):
    """Every tensor's shape by its name in a model folder; names end in what they are."""
    found = {}
    if config.get("architecture") == "Dolezen":
        width = config["width"]
        found["embed"], found["head"], found["final.norm"] = (config["vocab"], width), (config["vocab"], width), (width,)
        for index, layer in enumerate(config["layers"]):
            m, p = layer["mixer"], f"l{index}.mix."
            heads, values = m["heads"], m["heads"] * m["vdim"]
            if layer["type"] == "attention":
                parts = {"q": heads * m["dim"]}
                if "kv_from" not in m:
                    parts |= {"k": m["kv_heads"] * m["dim"], "v": m["kv_heads"] * m["vdim"]}
                found |= {p + name: (rows, width) for name, rows in parts.items()} | {p + name + ".b": (rows,) for name, rows in parts.items()}
                found |= {p + "sink": (heads,), p + "o": (width, values), p + "o.b": (width,)}
            else:
                found |= {p + "dq": (m["q_rank"], width), p + "dq.norm": (m["q_rank"],), p + "uq": (heads * (m["dim"] + m["rot_dim"]), m["q_rank"])}
                found |= {p + "dkv": (m["kv_rank"] + m["rot_dim"], width), p + "dkv.norm": (m["kv_rank"],)}
                found |= {p + "uk": (heads * m["dim"], m["kv_rank"]), p + "uv": (values, m["kv_rank"]), p + "o": (width, values)}
            found[f"l{index}.norm1"] = (width,)
            found |= {f"l{index}.mlp.up": (layer["mlp"]["ff"], width), f"l{index}.mlp.down": (width, layer["mlp"]["ff"])}
        return found
    width, inner, dim = config["hidden_size"], config["intermediate_size"], config["head_dim"]
    found["model.embed_tokens.weight"], found["model.norm.weight"] = (config["vocab_size"], width), (width,)
    if not config["tie_word_embeddings"]:
        found["lm_head.weight"] = (config["vocab_size"], width)
    for index in range(config["num_hidden_layers"]):
        p = f"model.layers.{index}."
        for name, heads in (("q", config["num_attention_heads"]), ("k", config["num_key_value_heads"]), ("v", config["num_key_value_heads"])):
            found |= {p + f"self_attn.{name}_proj.weight": (heads * dim, width), p + f"self_attn.{name}_proj.bias": (heads * dim,)}
        found[p + "self_attn.o_proj.weight"] = (width, config["num_attention_heads"] * dim)
        found |= {p + f"mlp.{name}_proj.weight": (inner, width) for name in ("gate", "up")}
        found[p + "mlp.down_proj.weight"] = (width, inner)
        found |= {p + name + "_layernorm.weight": (width,) for name in ("input", "post_attention")}
    return found


def _weights(config, dtype):
    """The model that a program has loaded: the same random weights always, as decoders are initialised: a matrix's by
    the root of its inputs, what writes to the residual stream smaller by the root of how often that happens (no layer
    drowns the others, and rounding does not grow from layer to layer), an embedding that gives logits a spread of two
    or three, norms around one."""
    generator = torch.Generator(device=DEVICE).manual_seed(20260)
    depth = config["num_hidden_layers"] if "num_hidden_layers" in config else len(config["layers"])
    found = {}
    for name, shape in _shapes(config).items():
        value = torch.randn(shape, generator=generator, device=DEVICE)
        if len(shape) == 1:
            value = value.mul_(0.1).add_(1.0) if "norm" in name else value.mul_(0.02)
        elif name in OUTSIDE:
            value.mul_(0.02 if "architecture" in config else 0.05)
        else:
            writes = name.endswith(("o_proj.weight", "down_proj.weight", "mix.o", "mlp.down"))
            value.mul_((0.8 / math.sqrt(2 * depth) if writes else 0.8) / math.sqrt(shape[1]))
        found[name] = value.to(dtype)
    return found


class _Engine:
    def __init__(self, model):
        values, self.dtype, held = _read(model)
        self.values, self.tensors = values, _weights(values, self.dtype)
        architecture = resolve_architecture(values)
        config = architecture.config_class.from_dict(values)
        loaded = LoadedModel(architecture, config, architecture.build_spec(config), self.tensors, self.dtype)
        self.kernels = HipKernels(self.dtype, DEVICE)
        self.runner = ModelRunner(loaded, self.kernels, CacheConfig(block_size=PAGE, num_blocks=held // PAGE, max_sequences=SLOTS))
        self.serial = itertools.count()


_engines: dict[str, _Engine] = {}


def _engine(model):
    if model not in _engines:
        _engines[model] = _Engine(model)
    return _engines[model]


# ---------------------------------------------------------------------------- inputs


def _vocab(config):
    return config["vocab"] if "vocab" in config else config["vocab_size"]


def _contexts(case):
    """Tokens that each request has cached: spread evenly from half the mean to half as much again."""
    count = case["requests"]
    return [max(1, round(case["context"] * (0.5 + (index * 0.6180339887 + 0.5) % 1.0))) for index in range(count)]


def _tokens(case, seed):
    """The tokens of a case: what is cached, what every request brings step by step, and the new prompt."""
    generator = torch.Generator().manual_seed(seed)
    values, _, _ = _read(case["model"])

    def some(count):
        return torch.randint(4, _vocab(values), (count,), generator=generator).tolist()

    if case["kind"] == "prompt":
        return [], [], some(case["length"])
    cached = [some(length) for length in _contexts(case)]
    brought = [some(STEPS) for _ in cached]
    return cached, brought, some(case["portion"] * STEPS) if case["kind"] == "mixed" else []


def _end(runner, names):
    for name in names:
        if runner.has_request(name):
            runner.end_request(name)


class _State:
    def __init__(self, case, seed):
        self.case = dict(case)
        self.engine = _engine(case["model"])
        runner, serial = self.engine.runner, next(self.engine.serial)
        self.name = f"new {serial}"
        cached, self.brought, self.prompt = _tokens(case, seed)
        self.names = [f"{serial}.{index}" for index in range(len(cached))]
        self.lengths = [len(tokens) for tokens in cached]
        weakref.finalize(self, _end, runner, [self.name, *self.names])
        # prompts of several requests share a step, up to its budget of tokens
        step, room = [], 2048
        for name, tokens in zip(self.names, cached):
            at = 0
            while at < len(tokens):
                piece = tokens[at : at + room]
                step.append(StepEntry(name, piece))
                at, room = at + len(piece), room - len(piece)
                if room == 0:
                    runner.step(step, create_missing=True)
                    step, room = [], 2048
        if step:
            runner.step(step, create_missing=True)


def prepare(case, seed):
    if case["kind"] == "sample":
        values, _, _ = _read(case["model"])
        generator = torch.Generator(device=DEVICE).manual_seed(seed)
        logits = 3.0 * torch.randn((case["rows"], _vocab(values)), generator=generator, device=DEVICE)
        configs = [GenerationConfig(temperature=case["temperature"], top_p=case["top_p"], seed=seed + row) for row in range(case["rows"])]
        return Sampler(_engine(case["model"]).kernels), logits, configs, list(range(case["rows"]))
    return _State(case, seed)


def run(state):
    if isinstance(state, tuple):
        sampler, logits, configs, steps = state
        return sampler.sample_on_device(logits, configs, steps)
    runner, case = state.engine.runner, state.case
    if case["kind"] == "prompt":
        portion, prompt = case["portion"], state.prompt
        for at in range(0, len(prompt), portion):
            piece = prompt[at : at + portion]
            logits = runner.step([StepEntry(state.name, piece, [len(piece) - 1] if at + portion >= len(prompt) else [])], create_missing=True)
        logits = logits.clone()  # (the next step may overwrite what a step returned)
        runner.end_request(state.name)
        return logits
    found = []
    for step in range(STEPS):
        entries = [StepEntry(name, (tokens[step],), (0,)) for name, tokens in zip(state.names, state.brought)]
        if case["kind"] == "mixed":
            portion = case["portion"]
            last = [portion - 1] if step == STEPS - 1 else []
            entries.append(StepEntry(state.name, state.prompt[step * portion : (step + 1) * portion], last))
        found.append(runner.step(entries, create_missing=case["kind"] == "mixed").clone())
    if case["kind"] == "mixed":
        runner.end_request(state.name)
    for name, length in zip(state.names, state.lengths):  # the brought tokens go again
        runner.cache.cancel(Reservation(name, 0, length, STEPS, ()))
    return found


# ---------------------------------------------------------------------------- what a pass cannot do without


def _queries(case):
    """(new tokens, keys before them) of every request in every step, and the rows of logits wanted, step by step."""
    if case["kind"] == "prompt":
        length, portion = case["length"], case["portion"]
        starts = range(0, length, portion)
        return [([(min(portion, length - at), at)], 1 if at + portion >= length else 0) for at in starts]
    steps = []
    for step in range(STEPS):
        queries = [(1, length + step) for length in _contexts(case)]
        if case["kind"] == "mixed":
            queries.append((case["portion"], step * case["portion"]))
        steps.append((queries, case["requests"] + (1 if case["kind"] == "mixed" and step == STEPS - 1 else 0)))
    return steps


def work(case):
    config, dtype, _ = _read(case["model"])
    vocab = _vocab(config)
    if case["kind"] == "sample":
        return {"bytes": 4.0 * case["rows"] * vocab, "flops": 4.0 * case["rows"] * vocab}
    shapes = _shapes(config)
    size = 2 if dtype == torch.bfloat16 else 4
    inside = sum(math.prod(shape) for name, shape in shapes.items() if name not in OUTSIDE)
    width = config.get("width", config.get("hidden_size"))
    if "layers" in config:  # a cached token's entries, and what its scores and weighted values multiply, layer by layer
        entries = pairs = 0
        for layer in config["layers"]:
            m = layer["mixer"]
            if layer["type"] == "attention":
                entries += 0 if "kv_from" in m else m["kv_heads"] * (m["dim"] + m["vdim"])
                pairs += m["heads"] * (m["dim"] + m["vdim"])
            else:
                entries += m["kv_rank"] + m["rot_dim"]
                pairs += m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
    else:
        entries = config["num_hidden_layers"] * 2 * config["num_key_value_heads"] * config["head_dim"]
        pairs = config["num_hidden_layers"] * 2 * config["num_attention_heads"] * config["head_dim"]
    moved = flops = 0.0
    for queries, wanted in _queries(case):
        tokens = sum(count for count, _ in queries)
        moved += size * (inside + tokens * width + (vocab * width if wanted else 0)) + 4.0 * wanted * vocab
        moved += size * entries * sum(count + before for count, before in queries)
        flops += 2.0 * inside * tokens + 2.0 * wanted * vocab * width
        flops += 2.0 * pairs * sum(count * before + count * (count + 1) / 2 for count, before in queries)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return {"differ": 0.01}  # whole numbers: a draw that falls on the edge between two tokens
    if "float32" in case["model"]:
        return {"rel": 1e-5, "max": 1e-4}  # 2e-6 off the same in 64 bits
    return {"rel": 0.022, "max": 0.2}  # 0.0055 off the same in 64 bits: bfloat16 activations through the layers


# ---------------------------------------------------------------------------- the same in 64 bits


def _norm(x, weight, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * weight


def _turn(x, positions, dims, base, neighbours):
    """x [n, heads, width]: the first `dims` dimensions turn in pairs, of neighbours or of i and i + dims / 2."""
    half = dims // 2
    angles = positions[:, None] * base ** (-torch.arange(half, device=x.device, dtype=x.dtype) / half)
    cos, sin = angles.cos()[:, None], angles.sin()[:, None]
    turned, rest = x[..., :dims], x[..., dims:]
    a, b = (turned[..., ::2], turned[..., 1::2]) if neighbours else (turned[..., :half], turned[..., half:])
    pair = [a * cos - b * sin, b * cos + a * sin]
    return torch.cat([torch.stack(pair, -1).flatten(-2) if neighbours else torch.cat(pair, -1), rest], -1)


def _attend(q, k, v, scale, lengths, seen, sinks=None):
    """Sequences side by side along the first axis, each over its own keys; `seen(i, j)`: whether query i sees key j."""
    out = q.new_empty(q.shape[0], q.shape[1], v.shape[2])
    at = 0
    for length in lengths:
        keys, values = (t[at : at + length].repeat_interleave(q.shape[1] // t.shape[1], 1).transpose(0, 1) for t in (k, v))
        place = torch.arange(length, device=q.device)
        for first in range(0, length, 1024):
            last = min(length, first + 1024)
            scores = q[at + first : at + last].transpose(0, 1) @ keys[:, :last].transpose(1, 2) * scale
            i, j = place[first:last, None], place[None, :last]
            scores.masked_fill_(~((j <= i) & seen(i, j)), -math.inf)
            if sinks is not None:
                scores = torch.cat([scores, sinks[:, None, None].expand(-1, last - first, 1)], -1)
            weights = scores.softmax(-1)[..., :last]
            out[at + first : at + last] = (weights @ values[:, :last]).transpose(0, 1)
        at += length
    return out.flatten(1)


def _qwen2(config, t, tokens, positions, lengths):
    eps, dim, base = config["rms_norm_eps"], config["head_dim"], config["rope_theta"]
    x = t("model.embed_tokens.weight", tokens)
    for index in range(config["num_hidden_layers"]):
        p = f"model.layers.{index}."
        h = _norm(x, t(p + "input_layernorm.weight"), eps)
        q, k, v = ((h @ t(p + f"self_attn.{n}_proj.weight").T + t(p + f"self_attn.{n}_proj.bias")).unflatten(1, (-1, dim)) for n in "qkv")
        q, k = _turn(q, positions, dim, base, True), _turn(k, positions, dim, base, True)
        x = x + _attend(q, k, v, dim ** -0.5, lengths, lambda i, j: j >= 0) @ t(p + "self_attn.o_proj.weight").T
        h = _norm(x, t(p + "post_attention_layernorm.weight"), eps)
        inner = torch.nn.functional.silu(h @ t(p + "mlp.gate_proj.weight").T) * (h @ t(p + "mlp.up_proj.weight").T)
        x = x + inner @ t(p + "mlp.down_proj.weight").T
    head = "model.embed_tokens.weight" if config["tie_word_embeddings"] else "lm_head.weight"
    return lambda rows: _norm(x[rows], t("model.norm.weight"), eps) @ t(head).T


def _dolezen(config, t, tokens, positions, lengths):
    eps = config["norm"]["eps"]
    x = t("embed", tokens) * config["embedding"]["scale"]
    kept = {}
    for index, layer in enumerate(config["layers"]):
        m, p = layer["mixer"], f"l{index}.mix."
        h = _norm(x, t(f"l{index}.norm1"), eps)
        size = m["mask"]["size"]
        if layer["type"] == "attention":
            if "kv_from" not in m:
                kept[index] = [(h @ t(p + n).T + t(p + n + ".b")).unflatten(1, (m["kv_heads"], -1)) for n in "kv"]
            q = (h @ t(p + "q").T + t(p + "q.b")).unflatten(1, (m["heads"], -1))
            mixed = _attend(q, *kept[m.get("kv_from", index)], m["scale"], lengths, lambda i, j: i // size == j // size, t(p + "sink"))
            update = mixed @ t(p + "o").T + t(p + "o.b")
        else:
            turn = (positions, m["rot"]["dims"], m["rot"]["base"], False)
            q = (_norm(h @ t(p + "dq").T, t(p + "dq.norm"), eps) @ t(p + "uq").T).unflatten(1, (m["heads"], -1))
            q = torch.cat([q[..., : m["dim"]], _turn(q[..., m["dim"] :], *turn)], -1)
            c, shared = (h @ t(p + "dkv").T).split([m["kv_rank"], m["rot_dim"]], 1)
            c = _norm(c, t(p + "dkv.norm"), eps)
            k, v = ((c @ t(p + n).T).unflatten(1, (m["heads"], -1)) for n in ("uk", "uv"))
            k = torch.cat([k, _turn(shared[:, None], *turn).expand(-1, m["heads"], -1)], -1)
            update = _attend(q, k, v, m["scale"], lengths, lambda i, j: i - j < size) @ t(p + "o").T
        x = x + update + (h @ t(f"l{index}.mlp.up").T).relu().square() @ t(f"l{index}.mlp.down").T
    return lambda rows: _norm(x[rows], t("final.norm"), eps) @ t("head").T


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "sample":
        return None
    config, dtype, _ = _read(case["model"])
    weights = _weights(config, dtype)
    cached, brought, prompt = _tokens(case, seed)
    sequences = [had + new for had, new in zip(cached, brought)] + ([prompt] if prompt else [])
    lengths = [len(tokens) for tokens in sequences]
    starts = list(itertools.accumulate(lengths, initial=0))
    positions = torch.cat([torch.arange(length) for length in lengths]).to(DEVICE, torch.float64)
    tokens = torch.tensor(list(itertools.chain(*sequences)), device=DEVICE)

    def tensor(name, rows=None):
        return (weights[name] if rows is None else weights[name][rows]).double()

    logits = (_dolezen if "layers" in config else _qwen2)(config, tensor, tokens, positions, lengths)
    last = starts[-1] - 1
    if case["kind"] == "prompt":
        return logits([last])
    found = []
    for step in range(STEPS):
        rows = [start + len(had) + step for start, had in zip(starts, cached)]
        found.append(logits(rows + [last] if case["kind"] == "mixed" and step == STEPS - 1 else rows))
    return found
