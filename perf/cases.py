"""Cases that stand for what this engine is used for: steps of a model through ``ModelRunner.step``,
the step function that generation, the scheduler and trace replay all go through.

Every case names a model (the three smallest dense sizes of ``bench.py``, or one of two other designs at the
sizes of its design comparison), a dtype, and a kind of pass:

* ``decode``  one step that brings one token for each of ``requests`` live requests, whose contexts lie
              between ``shortest`` and ``longest`` tokens: a step of running generation;
* ``prompts`` new requests, their whole prompts in one step, logits at the last token of each, ended again;
* ``mixed``   the step of continuous batching: ``requests`` live requests bring a token each and beside them
              a new request brings ``portion`` tokens of its prompt;
* ``turn``    a whole exchange: the prompts in one step, ``new`` tokens one by one, ended again.

Token ids are given, not sampled, as trace replay does it, so that two implementations whose logits differ in
the last bits still run on the same tokens.  Weights are drawn here, as models are initialised for training: a
sublayer's output is small beside the stream that it is added to, as it is in trained models too, so that a
rounding in one layer stays a rounding in the logits.  ``exact`` computes the same logits from the same weights with
plain torch in 64 bits, whole sequences at once.
"""

from __future__ import annotations

import math

import torch

from forge_engine_amd.config import load_model_config
from forge_engine_amd.engine import ModelRunner, StepEntry, build_model

DEVICE = "cuda:0"
BLOCK = 16              # tokens a cache page holds
FILL_TOKENS = 8192      # prompt tokens a step when a decode case's contexts are filled
GROWTH = 1024           # tokens a decoding request may grow by before it ends and its successor begins

# ------------------------------------------------------------------ models

_DENSE = {
    "qwen3-0.6b": {"hidden_size": 1024, "intermediate_size": 3072, "num_hidden_layers": 28, "num_attention_heads": 16,
                   "rope_theta": 1000000.0},
    "qwen3-1.7b": {"hidden_size": 2048, "intermediate_size": 6144, "num_hidden_layers": 28, "num_attention_heads": 16,
                   "rope_theta": 1000000.0},
    "qwen3-4b": {"hidden_size": 2560, "intermediate_size": 9728, "num_hidden_layers": 36, "num_attention_heads": 32,
                 "rope_theta": 5000000.0},
}


def _dense(name: str) -> dict:
    return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu", "vocab_size": 151936,
            "num_key_value_heads": 8, "head_dim": 128, "max_position_embeddings": 262144, "rms_norm_eps": 1e-6,
            "attention_bias": False, "eos_token_id": 151645, "tie_word_embeddings": True, **_DENSE[name]}


def _rekezen(width: int, layers: int = 6) -> dict:
    """Four residual streams, eight experts of which a token takes two beside a shared one, every second layer on
    the keys and values of the layer before it."""
    heads = max(4, width // 128)

    def mixer(index):
        sizes = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 30.0,
                 "rot": {"dims": 64, "base": 100000.0, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        if index % 2:
            sizes["kv_from"] = index - 1
        return sizes

    mlp = {"kind": "moe", "router": {"experts": 8, "top": 2}, "expert": {"ff": width, "limit": 7.0},
           "shared": {"ff": width, "limit": 7.0}}
    return {"architecture": "Rekezen", "vocab": 32000, "width": width, "norm": {"eps": 1e-6}, "streams": 4,
            "embedding": {"bigram": {"buckets": 65521, "mul_prev": 36313, "mul_cur": 27191}}, "logit_scale": 1.0,
            "layers": [{"type": "attention", "mixer": mixer(i), "mlp": mlp} for i in range(layers)]}


def _mazanex(width: int, layers: int = 6) -> dict:
    """Layers that cycle through attention beside RWKV time mixing, gated linear attention and mLSTM."""
    heads = max(4, width // 128)
    attention = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "conv": 4, "mask": {"size": 2048},
                 "rot": {"dims": 64, "base": 10000.0}, "scale": 128 ** -0.5}
    mixers = [("parallel", {"left": attention, "right": {"heads": width // 64, "dim": 64, "rank": 64}}),
              ("gla", {"heads": heads, "dim": 64, "vdim": 128, "tau": 16.0, "rank": 16}),
              ("mlstm", {"heads": max(2, heads // 2), "dim": 128, "vdim": 256, "gate_cap": 15.0})]
    return {"architecture": "Mazanex", "vocab": 32000, "width": width, "norm": {"eps": 1e-6},
            "layers": [{"type": mixers[i % 3][0], "mixer": mixers[i % 3][1], "mlp": {"kind": "dense", "ff": 3 * width}}
                       for i in range(layers)]}


def _raw(case: dict) -> dict:
    name = case["model"]
    if name.startswith("qwen3"):
        return _dense(name)
    return (_rekezen if name == "rekezen" else _mazanex)(case["width"])


def _vocab(case: dict) -> int:
    return 151936 if case["model"].startswith("qwen3") else 32000


# ------------------------------------------------------------------- cases

def listed() -> list[dict]:
    return [
        # one person talks to the smallest model: launches and latency are everything
        {"name": "decode 0.6b 1 request", "kind": "decode", "model": "qwen3-0.6b", "dtype": "bfloat16", "requests": 1,
         "longest": 217, "shortest": 217},
        # the headline: batch 8 behind 1,024-token prompts, weights streamed once a step
        {"name": "decode 4b 8 requests", "kind": "decode", "model": "qwen3-4b", "dtype": "bfloat16", "requests": 8,
         "longest": 1024, "shortest": 1024},
        # a busy server: as many requests as the headline's largest batch, contexts of all lengths
        {"name": "decode 4b 64 requests", "kind": "decode", "model": "qwen3-4b", "dtype": "bfloat16", "requests": 64,
         "longest": 2000, "shortest": 130},
        # few requests over long documents: the cache is most of what a step reads
        {"name": "decode 1.7b 4 long requests", "kind": "decode", "model": "qwen3-1.7b", "dtype": "bfloat16", "requests": 4,
         "longest": 16001, "shortest": 6000},
        # the headline's prompt
        {"name": "prompt 4b 2048 tokens", "kind": "prompts", "model": "qwen3-4b", "dtype": "bfloat16", "requests": 1,
         "longest": 2048, "shortest": 2048},
        # a document: the largest step, at a length that fills no tile
        {"name": "prompt 4b 6001 tokens", "kind": "prompts", "model": "qwen3-4b", "dtype": "bfloat16", "requests": 1,
         "longest": 6001, "shortest": 6001},
        # a few short chat prompts that arrive together
        {"name": "prompts 0.6b 3 short", "kind": "prompts", "model": "qwen3-0.6b", "dtype": "bfloat16", "requests": 3,
         "longest": 231, "shortest": 37},
        # the scheduler's default budget of 256 tokens a step: single tokens and a portion of a prompt
        {"name": "mixed 4b 7 and a portion", "kind": "mixed", "model": "qwen3-4b", "dtype": "bfloat16", "requests": 7,
         "longest": 900, "shortest": 100, "portion": 249},
        # the 32-bit mode, in which answers are checked: a prompt, and running generation
        {"name": "prompt 0.6b f32 700 tokens", "kind": "prompts", "model": "qwen3-0.6b", "dtype": "float32", "requests": 1,
         "longest": 700, "shortest": 700},
        {"name": "decode 1.7b f32 4 requests", "kind": "decode", "model": "qwen3-1.7b", "dtype": "float32", "requests": 4,
         "longest": 600, "shortest": 90},
        # the other designs, a whole exchange each: several streams and experts; recurrences over a matrix state
        {"name": "turn rekezen 8 requests", "kind": "turn", "model": "rekezen", "width": 2048, "dtype": "bfloat16",
         "requests": 8, "longest": 400, "shortest": 60, "new": 8},
        {"name": "turn mazanex 6 requests", "kind": "turn", "model": "mazanex", "width": 2048, "dtype": "bfloat16",
         "requests": 6, "longest": 500, "shortest": 70, "new": 8},
    ]


def _log(rng, low: int, high: int) -> int:
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    """Another case of the same ranges: batch sizes, prompt and context lengths spread over their logarithm."""
    kind = rng.choice(("decode", "decode", "prompts", "prompts", "mixed", "turn"))
    if kind == "turn":
        requests = _log(rng, 1, 8)
        longest = _log(rng, 24, 500)
        return {"kind": "turn", "model": rng.choice(("rekezen", "mazanex")), "width": rng.choice((1024, 2048)), "dtype": "bfloat16",
                "requests": requests, "longest": longest, "shortest": _log(rng, max(1, longest // 8), longest), "new": 8}
    dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float32"))
    model = rng.choice(("qwen3-0.6b", "qwen3-1.7b") if dtype == "float32" else tuple(_DENSE))
    case = {"kind": kind, "model": model, "dtype": dtype}
    if kind == "prompts":
        total = _log(rng, 16, 600 if dtype == "float32" else 6000)
        requests = min(_log(rng, 1, 12), max(1, total // 16))
        longest = max(2, total // requests)
        shortest = _log(rng, max(1, longest // 8), longest)
    else:
        requests = _log(rng, 1, 8 if dtype == "float32" else 64)
        longest = _log(rng, 60, max(61, min(12000, (8000 if dtype == "float32" else 40000) // requests)))
        shortest = _log(rng, max(1, longest // 8), longest)
    case.update(requests=requests, longest=longest, shortest=shortest)
    if kind == "mixed":
        case["portion"] = _log(rng, 16, 300 if dtype == "float32" else 1000)
    return case


def _lengths(case: dict) -> list[int]:
    """The requests' prompt lengths, from the longest to the shortest, evenly over the logarithm."""
    n, longest, shortest = case["requests"], case["longest"], case["shortest"]
    if n == 1:
        return [longest]
    return [int(round(longest * (shortest / longest) ** (i / (n - 1)))) for i in range(n)]


def _prompts(case: dict, seed: int) -> tuple[list[list[int]], list[list[int]], list[int]]:
    """(prompts, the single tokens of a few steps, the portion of a mixed case's new prompt)."""
    generator = torch.Generator().manual_seed(seed * 7919 + 17)

    def ids(count):
        return torch.randint(0, _vocab(case), (count,), generator=generator).tolist()

    prompts = [ids(n) for n in _lengths(case)]
    singles = [ids(case["requests"]) for _ in range(16)]
    return prompts, singles, ids(case.get("portion", 0))


def _fill(state: dict) -> None:
    """Begin the decoding requests anew: their prompts in steps of up to FILL_TOKENS tokens."""
    runner = state["runner"]
    step, room = [], FILL_TOKENS

    def flush():
        nonlocal step, room
        if step:
            runner.step(step)
        step, room = [], FILL_TOKENS

    for name, prompt in zip(state["names"], state["prompts"]):
        runner.begin(name)
        at = 0
        while at < len(prompt):
            count = min(room, len(prompt) - at)
            step.append(StepEntry(name, prompt[at:at + count], []))
            at, room = at + count, room - count
            if not room:
                flush()
    flush()
    state["grown"] = 0


def prepare(case: dict, seed: int) -> dict:
    """A model with its runner, as a serving program holds them; the requests of a decode or mixed case hold their
    contexts already."""
    model = build_model(load_model_config(_raw(case)), dtype=case["dtype"], device=torch.device(DEVICE))
    for name, tensor in _draw_weights(case, seed):
        model.set_param(name, tensor)
    model.finalize()
    prompts, singles, portion = _prompts(case, seed)
    lives = case["kind"] in ("decode", "mixed")
    extra = GROWTH if lives else case.get("new", 0)
    pages = sum(-(-(len(p) + extra) // BLOCK) for p in prompts) + -(-len(portion) // BLOCK) + 1
    runner = ModelRunner(model, block_size=BLOCK, block_capacity=pages, num_state_slots=case["requests"] + 1)
    state = {"kind": case["kind"], "runner": runner, "names": [f"r{i}" for i in range(case["requests"])], "prompts": prompts,
             "singles": singles, "portion": portion, "new": case.get("new", 0), "grown": 0}
    if lives:
        _fill(state)
    return state


def run(state: dict):
    kind, runner, names, prompts = state["kind"], state["runner"], state["names"], state["prompts"]
    if kind in ("decode", "mixed"):
        if state["grown"] == GROWTH:
            for name in names:
                runner.end(name)
            _fill(state)
        tokens = state["singles"][state["grown"] % len(state["singles"])]
        entries = [StepEntry(name, [token], [0]) for name, token in zip(names, tokens)]
        state["grown"] += 1
        if kind == "decode":
            return runner.step(entries)
        portion = state["portion"]
        runner.begin("new")
        logits = runner.step(entries + [StepEntry("new", portion, [len(portion) - 1])])
        runner.end("new")
        return logits
    for name in names:
        runner.begin(name)
    logits = runner.step([StepEntry(name, prompt, [len(prompt) - 1]) for name, prompt in zip(names, prompts)])
    if kind == "turn":
        logits = [logits.clone()]      # a step's logits are overwritten by the next step of its shape
        for tokens in state["singles"][:state["new"]]:
            logits.append(runner.step([StepEntry(name, [token], [0]) for name, token in zip(names, tokens)]).clone())
    for name in names:
        runner.end(name)
    return logits


# -------------------------------------------------------- what a pass needs

def _steps(case: dict) -> list[tuple[list[tuple[int, int]], int]]:
    """The steps of a pass: (tokens before and tokens brought of every request, rows of logits)."""
    lengths, n = _lengths(case), case["requests"]
    if case["kind"] == "decode":
        return [([(length, 1) for length in lengths], n)]
    if case["kind"] == "mixed":
        return [([(length, 1) for length in lengths] + [(0, case["portion"])], n + 1)]
    steps = [([(0, length) for length in lengths], n)]
    return steps + [([(length + i, 1) for length in lengths], n) for i in range(case.get("new", 0))]


def work(case: dict) -> dict:
    """Weights, the live cache and the stream's ends once a step; the products' and the attention's operations.  A
    token's recurrence over a matrix state is counted as its update and its read."""
    raw, size = _raw(case), 2 if case["dtype"] == "bfloat16" else 4
    matrices = {name: shape for name, shape, _, matrix in _tensors(case) if matrix}
    lookups = {"model.embed_tokens.weight", "embed", "bigram"}
    # what a token's products touch: two experts of eight
    dense = sum(math.prod(s) for n, s in matrices.items() if n not in lookups and n != "head" and ".mlp.e" not in n)
    experts = sum(math.prod(s) for n, s in matrices.items() if ".mlp.e" in n)
    vocab = _vocab(case)
    if case["model"].startswith("qwen3"):
        width, layers = raw["hidden_size"], raw["num_hidden_layers"]
        heads, reading, kv = raw["num_attention_heads"], layers, 2 * 8 * 128 * layers
        recurrent = state = 0
    else:
        width, layers = raw["width"], len(raw["layers"])
        heads = max(4, width // 128)
        rekezen = case["model"] == "rekezen"
        reading = layers if rekezen else layers // 3
        kv = 2 * (heads // 4) * 128 * (layers // 2 if rekezen else reading)
        # elements of the matrix states of the three mixers: RWKV, gated linear attention, mLSTM
        state = 0 if rekezen else (layers // 3) * (width * 64 + heads * 64 * 128 + max(2, heads // 2) * 128 * 256)
        recurrent = 4 * state
    total_bytes = total_flops = 0.0
    for requests, rows in _steps(case):
        tokens = sum(q for _, q in requests)
        touched = 0 if not experts else experts * min(1.0, tokens * 2 / 8)
        keys = sum(before * q + q * (q + 1) / 2 for before, q in requests)
        held = sum(before + q for before, q in requests)
        total_bytes += (dense + touched + vocab * width) * size + held * kv * size + tokens * (kv + width) * size \
            + 8 * state * len(requests) + rows * vocab * 4
        total_flops += 2.0 * tokens * (dense + experts / 4) + 4.0 * keys * heads * 128 * reading + recurrent * tokens \
            + 2.0 * rows * vocab * width
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case: dict) -> dict:
    """Measured on one 2,048-token prompt of the largest model fed whole, in two portions, in eight: the logits differ by
    1.1e-2 to 1.2e-2 in bfloat16 (and from the 64-bit ones by 0.7e-2 to 1.0e-2); in 32 bits they lie 1e-6 from the
    64-bit ones."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------ the same in 64 bits, plain

def _tensors(case: dict):
    """(name, shape, how it is drawn, whether it is kept in the compute dtype), in the order of the draw."""
    raw, kind = _raw(case), case["model"]
    if kind.startswith("qwen3"):
        width, ff, q, kv = raw["hidden_size"], raw["intermediate_size"], raw["num_attention_heads"] * 128, 1024
        yield "model.embed_tokens.weight", (raw["vocab_size"], width), "embed", True
        for i in range(raw["num_hidden_layers"]):
            p = f"model.layers.{i}"
            for name, shape in (("q", (q, width)), ("k", (kv, width)), ("v", (kv, width)), ("o", (width, q))):
                yield f"{p}.self_attn.{name}_proj.weight", shape, "out" if name == "o" else "normal", True
            yield f"{p}.self_attn.q_norm.weight", (128,), "norm", False
            yield f"{p}.self_attn.k_norm.weight", (128,), "norm", False
            for name, shape in (("gate", (ff, width)), ("up", (ff, width)), ("down", (width, ff))):
                yield f"{p}.mlp.{name}_proj.weight", shape, "out" if name == "down" else "normal", True
            yield f"{p}.input_layernorm.weight", (width,), "norm", False
            yield f"{p}.post_attention_layernorm.weight", (width,), "norm", False
        yield "model.norm.weight", (width,), "norm", False
        return
    width, vocab = raw["width"], raw["vocab"]
    heads = max(4, width // 128)
    kv = heads // 4 * 128
    yield "embed", (vocab, width), "embed", True
    if kind == "rekezen":
        yield "bigram", (raw["embedding"]["bigram"]["buckets"] + 1, width), "embed", True
    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}", layer["mixer"]
        if kind == "rekezen":
            for hc in ("hc1", "hc2"):
                yield f"{p}.{hc}.in", (4,), "uniform", False
                yield f"{p}.{hc}.out", (4,), "norm", False
                yield f"{p}.{hc}.mix", (4, 4), "identity", False
            own = "kv_from" not in m
            yield f"{p}.mix.q", (heads * 128, width), "normal", True
            if own:
                yield f"{p}.mix.k", (kv, width), "normal", True
                yield f"{p}.mix.v", (kv, width), "normal", True
            yield f"{p}.mix.o", (width, heads * 128), "out", True
            yield f"{p}.mix.q.norm", (heads * 128,), "norm", False
            if own:
                yield f"{p}.mix.k.norm", (kv,), "norm", False
            yield f"{p}.mix.g", (heads, width), "normal", True
            yield f"{p}.mlp.router", (8, width), "router", True
            yield f"{p}.mlp.router.b", (8,), "small", False
            for e in (*(f"e{j}" for j in range(8)), "shared"):
                yield f"{p}.mlp.{e}.gate", (width, width), "normal", True
                yield f"{p}.mlp.{e}.up", (width, width), "normal", True
                yield f"{p}.mlp.{e}.down", (width, width), "out", True
            for norm in ("norm1", "norm2"):
                yield f"{p}.{norm}", (width,), "norm", False
                yield f"{p}.{norm}.b", (width,), "small", False
            continue
        yield f"{p}.shift", (width,), "uniform", False
        if layer["type"] == "parallel":
            yield f"{p}.mix.left.out", (width,), "norm", False
            yield f"{p}.mix.right.out", (width,), "norm", False
            left = f"{p}.mix.left"
            sizes = (("q", heads * 128), ("k", kv), ("v", kv))
            for name, rows in sizes:
                yield f"{left}.{name}", (rows, width), "normal", True
            yield f"{left}.o", (width, heads * 128), "normal", True
            for name, rows in (*sizes, ("o", width)):
                yield f"{left}.{name}.b", (rows,), "zeros", False
            for name, rows in sizes:
                yield f"{left}.{name}.conv", (rows, 4), "taps", False
            yield f"{left}.sink", (heads,), "unit", False
            yield f"{left}.g", (heads * 128, width), "normal", True
            right = f"{p}.mix.right"
            for name in "rkvgw":
                yield f"{right}.mu.{name}", (width,), "uniform", False
            for name in "rkvg":
                yield f"{right}.{name}", (width, width), "normal", True
            yield f"{right}.w1", (64, width), "normal", True
            yield f"{right}.w2", (width, 64), "normal", True
            yield f"{right}.w0", (width,), "unit", False
            yield f"{right}.u", (width // 64, 64), "unit", False
            yield f"{right}.norm", (width,), "norm", False
            yield f"{right}.o", (width, width), "normal", True
        else:
            h, d, dv = m["heads"], m["dim"], m["vdim"]
            for name, shape in (("q", (h * d, width)), ("k", (h * d, width)), ("v", (h * dv, width)), ("g", (h * dv, width)),
                                ("o", (width, h * dv))):
                yield f"{p}.mix.{name}", shape, "normal", True
            if layer["type"] == "gla":
                yield f"{p}.mix.norm", (dv,), "norm", False
                yield f"{p}.mix.a1", (16, width), "normal", True
                yield f"{p}.mix.a2", (h * d, 16), "normal", True
                yield f"{p}.mix.a2.b", (h * d,), "unit", False
            else:
                yield f"{p}.mix.norm", (h * dv,), "norm", False
                yield f"{p}.mix.i", (h, width), "normal", True
                yield f"{p}.mix.f", (h, width), "normal", True
                yield f"{p}.mix.i.b", (h,), "unit", False
                yield f"{p}.mix.f.b", (h,), "unit", False
        yield f"{p}.mlp.up", (3 * width, width), "normal", True
        yield f"{p}.mlp.down", (width, 3 * width), "normal", True
        yield f"{p}.mlp.act", (4,), "unit", False
        yield f"{p}.norm1", (width,), "out_norm", False
        yield f"{p}.norm2", (width,), "out_norm", False
    yield "final.norm", (width,), "norm", False
    if kind == "rekezen":
        yield "final.norm.b", (width,), "small", False
    else:
        yield "head", (vocab, width), "normal", True


# how a tensor is drawn: (mean, standard deviation); an output projection of a sublayer the smaller, the deeper the
# model; an output norm leaves a sublayer's output a tenth of its size
_DRAWS = {"embed": (0.0, 0.3), "normal": (0.0, 0.02), "norm": (1.0, 0.05), "out_norm": (0.1, 0.005), "unit": (0.0, 0.5),
          "small": (0.0, 0.1), "router": (0.0, 0.5), "identity": (0.0, 0.1), "taps": (0.0, 0.2), "zeros": (0.0, 0.0)}


def _draw_weights(case: dict, seed: int):
    """(name, tensor) for every tensor of the model, in the dtype in which it is kept."""
    generator = torch.Generator(device=DEVICE).manual_seed(seed)
    stored = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    raw = _raw(case)
    depth = 2 * (raw.get("num_hidden_layers") or len(raw["layers"]))
    for name, shape, how, matrix in _tensors(case):
        if how == "uniform":
            value = torch.rand(shape, generator=generator, dtype=torch.float32, device=DEVICE)
        else:
            mean, deviation = _DRAWS["normal" if how == "out" else how]
            if how == "out":
                deviation /= math.sqrt(depth)
            value = torch.randn(shape, generator=generator, dtype=torch.float32, device=DEVICE).mul_(deviation).add_(mean)
        if how == "identity":
            value += torch.eye(shape[-1], dtype=torch.float32, device=DEVICE)
        elif how == "taps":
            value[..., -1] += 1.0      # most weight on the newest
        yield name, value.to(stored) if matrix else value


def _sequences(case: dict, seed: int) -> tuple[list[list[int]], list[list[int]]]:
    """(every request's tokens from its first to its last, the places whose logits a pass returns, step by step)."""
    prompts, singles, portion = _prompts(case, seed)
    if case["kind"] == "prompts":
        return prompts, [[len(p) - 1] for p in prompts]
    if case["kind"] == "turn":
        new = case["new"]
        return ([p + [singles[j][i] for j in range(new)] for i, p in enumerate(prompts)],
                [[len(p) - 1 + j for j in range(new + 1)] for p in prompts])
    sequences = [p + [singles[0][i]] for i, p in enumerate(prompts)] + ([portion] if portion else [])
    return sequences, [[len(s) - 1] for s in sequences]


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, weight, bias, eps):
    centred = x - x.mean(-1, keepdim=True)
    return _unit(centred, eps) * weight + bias


def _turned(x, frequencies, magnitude=1.0):
    """x [T, heads, D] at positions 0, 1, ...: dim i and dim i + half turn by position times the pair's frequency."""
    half = len(frequencies)
    angle = torch.arange(x.shape[0], dtype=x.dtype, device=x.device)[:, None] \
        * torch.tensor(frequencies, dtype=x.dtype, device=x.device)[None, :]
    cos, sin = (angle.cos() * magnitude)[:, None, :], (angle.sin() * magnitude)[:, None, :]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat((a * cos - b * sin, b * cos + a * sin, x[..., 2 * half:]), dim=-1)


def _frequencies(rot) -> tuple[list[float], float]:
    """Frequencies of the rotation's pairs and the factor on its cosines and sines (YaRN where the rotation is stretched)."""
    dims, base, scaling = rot["dims"], rot["base"], rot.get("scaling")
    plain = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not scaling:
        return plain, 1.0

    def turning(turns):
        return dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    low, high = max(math.floor(turning(scaling["fast"])), 0), min(math.ceil(turning(scaling["slow"])), dims - 1)
    ramps = [min(max((i - low) / max(high - low, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [f / scaling["factor"] * r + f * (1.0 - r) for f, r in zip(plain, ramps)], 0.1 * math.log(scaling["factor"]) + 1.0


def _attention(q, k, v, scale, cap=None, sink=None):
    """Causal attention of one sequence: q [T, H, D], k and v [T, G, D]; a few rows and one kv head at a time."""
    count, heads, dim = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    rows = max(1, min(count, (1 << 27) // (group * count)))
    for g in range(k.shape[1]):
        keys, values = k[:, g].t().contiguous(), v[:, g].contiguous()
        for at in range(0, count, rows):
            end = min(count, at + rows)
            mine = q[at:end, g * group:(g + 1) * group].transpose(0, 1).reshape(-1, dim)
            scores = (mine @ keys[:, :end]) * scale
            if cap:
                scores = cap * torch.tanh(scores / cap)
            scores = scores.view(group, end - at, end)
            hidden = torch.arange(end, device=q.device)[None, :] > torch.arange(at, end, device=q.device)[:, None]
            scores.masked_fill_(hidden[None], -math.inf)
            if sink is not None:       # a score without a value
                scores = torch.cat((scores, sink[g * group:(g + 1) * group, None, None].expand(-1, end - at, 1)), dim=-1)
            shares = torch.softmax(scores, dim=-1)[..., :end].reshape(-1, end)
            out[at:end, g * group:(g + 1) * group] = (shares @ values[:end]).view(group, end - at, dim).transpose(0, 1)
    return out


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_dense(case, w, sequences, wanted):
    raw = _raw(case)
    eps, heads, layers = raw["rms_norm_eps"], raw["num_attention_heads"], raw["num_hidden_layers"]
    frequencies = [raw["rope_theta"] ** (-2.0 * i / 128) for i in range(64)]
    ids = torch.tensor([t for s in sequences for t in s], device=DEVICE)
    embedding = w["model.embed_tokens.weight"]
    h = embedding[ids].double()
    for i in range(layers):
        p = f"model.layers.{i}"
        m = {name: w[f"{p}.self_attn.{name}.weight"].double() for name in ("q_proj", "k_proj", "v_proj", "o_proj", "q_norm", "k_norm")}
        x = _unit(h, eps) * w[f"{p}.input_layernorm.weight"].double()
        q = _unit((x @ m["q_proj"].t()).view(-1, heads, 128), eps) * m["q_norm"]
        k = _unit((x @ m["k_proj"].t()).view(-1, 8, 128), eps) * m["k_norm"]
        v = (x @ m["v_proj"].t()).view(-1, 8, 128)
        at, mixed = 0, []
        for s in sequences:
            part = slice(at, at + len(s))
            mixed.append(_attention(_turned(q[part], frequencies), _turned(k[part], frequencies), v[part], 128 ** -0.5))
            at += len(s)
        h = h + torch.cat(mixed).view(h.shape[0], -1) @ m["o_proj"].t()
        gate, up, down = (w[f"{p}.mlp.{name}_proj.weight"].double() for name in ("gate", "up", "down"))
        x = _unit(h, eps) * w[f"{p}.post_attention_layernorm.weight"].double()
        h = h + (_silu(x @ gate.t()) * (x @ up.t())) @ down.t()
    rows, at = [], 0
    for s, places in zip(sequences, wanted):
        rows.append(h[torch.tensor(places, device=DEVICE) + at])
        at += len(s)
    return (_unit(torch.cat(rows), eps) * w["model.norm.weight"].double()) @ embedding.double().t()


def _exact_rekezen(case, w, ids, places):
    raw = _raw(case)
    eps, width = raw["norm"]["eps"], raw["width"]
    heads, pair = max(4, width // 128), raw["embedding"]["bigram"]
    rows = [pair["buckets"]] + [(a * pair["mul_prev"] + b * pair["mul_cur"]) % pair["buckets"] for a, b in zip(ids, ids[1:])]
    x = w["embed"][torch.tensor(ids, device=DEVICE)] + w["bigram"][torch.tensor(rows, device=DEVICE)]
    streams = x[None].repeat(raw["streams"], 1, 1)
    held = {}
    for i, layer in enumerate(raw["layers"]):
        m, p = layer["mixer"], f"l{i}"
        frequencies, magnitude = _frequencies(m["rot"])

        def mixer(u):
            x = _layer_norm(u, w[f"{p}.norm1"], w[f"{p}.norm1.b"], eps)
            q = (_unit(x @ w[f"{p}.mix.q"].t(), eps) * w[f"{p}.mix.q.norm"]).view(len(ids), heads, 128)
            if "kv_from" not in m:
                k = (_unit(x @ w[f"{p}.mix.k"].t(), eps) * w[f"{p}.mix.k.norm"]).view(len(ids), -1, 128)
                held[i] = _turned(k, frequencies, magnitude), (x @ w[f"{p}.mix.v"].t()).view(len(ids), -1, 128)
            o = _attention(_turned(q, frequencies, magnitude), *held[m.get("kv_from", i)], m["scale"], cap=m["softcap"])
            o = o * torch.sigmoid(x @ w[f"{p}.mix.g"].t())[:, :, None]
            return o.reshape(len(ids), -1) @ w[f"{p}.mix.o"].t()

        def expert(x, name):
            limit = layer["mlp"]["expert"]["limit"]
            g = (x @ w[f"{p}.mlp.{name}.gate"].t()).clamp(max=limit)
            u = (x @ w[f"{p}.mlp.{name}.up"].t()).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[f"{p}.mlp.{name}.down"].t()

        def feed_forward(u):
            x = _layer_norm(u, w[f"{p}.norm2"], w[f"{p}.norm2.b"], eps)
            z = x @ w[f"{p}.mlp.router"].t() + w[f"{p}.mlp.router.b"]
            best = z.topk(2, dim=-1)
            shares = torch.zeros_like(z).scatter(1, best.indices, torch.softmax(best.values, dim=-1))
            return expert(x, "shared") + sum(shares[:, e, None] * expert(x, f"e{e}") for e in range(8))

        for hc, sublayer in (("hc1", mixer), ("hc2", feed_forward)):
            y = sublayer((w[f"{p}.{hc}.in"][:, None, None] * streams).sum(0))
            flat = w[f"{p}.{hc}.mix"].t() @ streams.reshape(streams.shape[0], -1)
            streams = flat.view_as(streams) + w[f"{p}.{hc}.out"][:, None, None] * y[None]
    z = _layer_norm(streams.sum(0)[places], w["final.norm"], w["final.norm.b"], eps)
    return z @ w["embed"].t() * raw["logit_scale"]


def _before(h):
    return torch.cat((torch.zeros_like(h[:1]), h[:-1]))


def _conv(u, taps):
    padded = torch.cat((torch.zeros_like(u[:taps.shape[1] - 1]), u))
    return sum(padded[j:j + len(u)] * taps[:, j] for j in range(taps.shape[1]))


def _exact_mazanex(case, w, ids, places):
    raw = _raw(case)
    eps, width, count = raw["norm"]["eps"], raw["width"], len(ids)
    x = w["embed"][torch.tensor(ids, device=DEVICE)]

    def left(h, p, m):
        heads, kv = m["heads"], m["kv_heads"]
        frequencies, _ = _frequencies(m["rot"])
        q, k, v = (_conv(h @ w[f"{p}.{n}"].t() + w[f"{p}.{n}.b"], w[f"{p}.{n}.conv"]) for n in "qkv")
        q = _unit(_turned(q.view(count, heads, 128), frequencies), eps)
        k = _unit(_turned(k.view(count, kv, 128), frequencies), eps)
        assert count <= m["mask"]["size"]       # one run of keys
        o = _attention(q, k, v.view(count, kv, 128), m["scale"], sink=w[f"{p}.sink"])
        return (o.reshape(count, -1) * torch.sigmoid(h @ w[f"{p}.g"].t())) @ w[f"{p}.o"].t() + w[f"{p}.o.b"]

    def right(h, p, m):
        heads, dim = m["heads"], m["dim"]
        mixed = {n: h + (_before(h) - h) * w[f"{p}.mu.{n}"] for n in "rkvgw"}
        r, k, v = ((mixed[n] @ w[f"{p}.{n}"].t()).view(count, heads, dim) for n in "rkv")
        decay = torch.exp(-torch.exp(torch.tanh(mixed["w"] @ w[f"{p}.w1"].t()) @ w[f"{p}.w2"].t() + w[f"{p}.w0"])).view(count, heads, dim)
        held, out = torch.zeros(heads, dim, dim, dtype=h.dtype, device=DEVICE), []
        for t in range(count):
            kv = k[t][:, :, None] * v[t][:, None, :]
            out.append(((held + w[f"{p}.u"][:, :, None] * kv) * r[t][:, :, None]).sum(1))
            held = decay[t][:, :, None] * held + kv
        o = _unit(torch.stack(out), eps).reshape(count, -1) * w[f"{p}.norm"] * _silu(mixed["g"] @ w[f"{p}.g"].t())
        return o @ w[f"{p}.o"].t()

    def recurrent(h, p, m, kind):
        heads, dim, wide = m["heads"], m["dim"], m["vdim"]
        q = (h @ w[f"{p}.q"].t()).view(count, heads, dim) * dim ** -0.5
        k = (h @ w[f"{p}.k"].t()).view(count, heads, dim)
        v = (h @ w[f"{p}.v"].t()).view(count, heads, wide)
        held, out = torch.zeros(heads, dim, wide, dtype=h.dtype, device=DEVICE), []
        if kind == "gla":
            z = (h @ w[f"{p}.a1"].t()) @ w[f"{p}.a2"].t() + w[f"{p}.a2.b"]
            keep = (torch.sigmoid(z) ** (1.0 / m["tau"])).view(count, heads, dim)
            for t in range(count):
                held = keep[t][:, :, None] * held + k[t][:, :, None] * v[t][:, None, :]
                out.append((held * q[t][:, :, None]).sum(1))
            o = (_unit(torch.stack(out), eps) * w[f"{p}.norm"]).reshape(count, -1) * _silu(h @ w[f"{p}.g"].t())
            return o @ w[f"{p}.o"].t()
        cap = m["gate_cap"]
        take = cap * torch.tanh((h @ w[f"{p}.i"].t() + w[f"{p}.i.b"]) / cap)
        keep = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w[f"{p}.f"].t() + w[f"{p}.f.b"]) / cap))
        total = torch.zeros(heads, dim, dtype=h.dtype, device=DEVICE)
        top = torch.zeros(heads, dtype=h.dtype, device=DEVICE)
        for t in range(count):
            higher = torch.maximum(keep[t] + top, take[t])
            a, b = torch.exp(keep[t] + top - higher), torch.exp(take[t] - higher)
            held = a[:, None, None] * held + b[:, None, None] * k[t][:, :, None] * v[t][:, None, :]
            total = a[:, None] * total + b[:, None] * k[t]
            top = higher
            below = torch.maximum((total * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            out.append((held * q[t][:, :, None]).sum(1) / below[:, None])
        o = _unit(torch.stack(out), eps).reshape(count, -1) * w[f"{p}.norm"] * torch.sigmoid(h @ w[f"{p}.g"].t())
        return o @ w[f"{p}.o"].t()

    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}", layer["mixer"]
        h = x + (_before(x) - x) * w[f"{p}.shift"]
        if layer["type"] == "parallel":
            mixed = 0.5 * (_unit(left(h, f"{p}.mix.left", m["left"]), eps) * w[f"{p}.mix.left.out"]
                           + _unit(right(h, f"{p}.mix.right", m["right"]), eps) * w[f"{p}.mix.right.out"])
        else:
            mixed = recurrent(h, f"{p}.mix", m, layer["type"])
        x = x + _unit(mixed, eps) * w[f"{p}.norm1"]
        z = x @ w[f"{p}.mlp.up"].t()
        a, b, c, e = w[f"{p}.mlp.act"]
        z = a * _unit(z, eps) + b * _unit(z ** 2, eps) + c * _unit(z ** 3, eps) + e
        x = x + _unit(z @ w[f"{p}.mlp.down"].t(), eps) * w[f"{p}.norm2"]
    return (_unit(x[places], eps) * w["final.norm"]) @ w["head"].t()


@torch.inference_mode()
def exact(case: dict, seed: int):
    weights = dict(_draw_weights(case, seed))
    sequences, wanted = _sequences(case, seed)
    if case["model"].startswith("qwen3"):
        return _exact_dense(case, weights, sequences, wanted)
    forward = _exact_rekezen if case["model"] == "rekezen" else _exact_mazanex
    weights = {name: tensor.double() for name, tensor in weights.items()}
    logits = [forward(case, weights, ids, torch.tensor(places, device=DEVICE)) for ids, places in zip(sequences, wanted)]
    return [torch.stack([rows[step] for rows in logits]) for step in range(case["new"] + 1)]
