"""The cases that this framework's speed is judged by: steps of its step function, from one token to a full token budget.

A case is one step: some requests bring a single token each (they decode), one more may bring a whole prompt or the next
portion of one.  ``prepare`` makes what a serving program holds when such a step is due (the model, the cache with what the
requests' earlier tokens left in it, the step's entries), ``run`` is ``ModelRunner.step``, which generation, replay and
measurement all go through, and its result is the 32-bit logits at the wanted places.  ``exact`` computes the same logits
in 64 bits from the same weights, cached keys and values and tokens, in plain torch.

Layer sizes are those of the benchmark (``bench.py``): the Qwen2.5-7B and 14B shapes, a Qwen2 model 2,048 wide, four layers
of the 7B shape in 32-bit, and the Lukelix design 2,048 wide (attention and selective state spaces).
"""

from __future__ import annotations

import functools
import math
import zlib

import torch

DEVICE = "cuda:0"
PAGE = 16

QWEN2_7B = {
    "architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": 3584, "num_hidden_layers": 28,
    "num_attention_heads": 28, "num_key_value_heads": 4, "head_dim": 128, "intermediate_size": 18944, "vocab_size": 152064,
    "rope_theta": 1000000.0, "rms_norm_eps": 1e-6, "tie_word_embeddings": False, "use_sliding_window": False,
    "max_position_embeddings": 32768,
}
ATTENTION = {
    "heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "conv": 4,
    "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 1024}},
}
SELECTIVE = {"heads": 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}


def _lukelix_layers() -> list[dict]:
    layers = []
    for index in range(12):
        if index % 4:
            layers.append({"type": "mamba2", "mixer": SELECTIVE, "mlp": None})
        else:  # the last attention layer reads the first one's keys and values
            mixer = dict(ATTENTION, kv_from=0) if index == 8 else ATTENTION
            layers.append({"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": 8192}})
    return layers


SHAPES = {
    "7b": QWEN2_7B,
    "14b": dict(QWEN2_7B, hidden_size=5120, num_hidden_layers=48, num_attention_heads=40, num_key_value_heads=8,
                intermediate_size=13824, rms_norm_eps=1e-5),
    "7b-4layers": dict(QWEN2_7B, num_hidden_layers=4),
    "2k": dict(QWEN2_7B, hidden_size=2048, num_hidden_layers=8, num_attention_heads=16, num_key_value_heads=4,
               intermediate_size=8192, vocab_size=32000),
    "lukelix-2k": {
        "architecture": "Lukelix", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-6}, "layers": _lukelix_layers(),
        "embedding": {"bigram": {"buckets": 32749, "mul_prev": 31, "mul_cur": 17}},
    },
}


def _case(model: str, dtype: str = "bfloat16", *, singles: int = 0, least: int = 0, most: int = 0, tokens: int = 0, held: int = 0) -> dict:
    """``singles`` requests bring one token each and hold between ``least`` and ``most`` tokens before it; one more
    brings ``tokens`` tokens behind the ``held`` it has in the cache."""
    return {"model": model, "dtype": dtype, "singles": singles, "least": least, "most": most, "tokens": tokens, "held": held}


def listed() -> list[dict]:
    return [
        # One user of a small model: some sixty short kernels, where launches and their gaps count.
        {"name": "decode_1_small", **_case("2k", singles=1, least=300, most=300)},
        # One user of the 7B model a few hundred tokens into an answer: the weights' bytes, one row.
        {"name": "decode_1", **_case("7b", singles=1, least=640, most=640)},
        # The benchmark's default: 8 requests with long contexts, weights and cache.
        {"name": "decode_8_long", **_case("7b", singles=8, least=8191, most=8191)},
        # A busy server: 64 requests of the serving profile's lengths, ragged.
        {"name": "decode_64", **_case("7b", singles=64, least=128, most=1535)},
        # A short prompt alone: the time to a chat's first token.
        {"name": "prompt_299", **_case("7b", tokens=299)},
        # A prompt that fills the token budget: the benchmark's prefill.
        {"name": "prompt_2048", **_case("7b", tokens=2048)},
        # The last portion of a long prompt: attention over what the earlier portions left in the cache.
        {"name": "portion_509", **_case("7b", tokens=509, held=7680)},
        # Continuous batching: decoding requests beside a new prompt in one step, the 14B shape.
        {"name": "mixed_14b", **_case("14b", singles=32, least=512, most=2047, tokens=2016)},
        # The true 32-bit path (``--dtype float32``): decode and a prompt.
        {"name": "decode_8_fp32", **_case("7b-4layers", "float32", singles=8, least=1023, most=1023)},
        {"name": "prompt_500_fp32", **_case("7b-4layers", "float32", tokens=500)},
        # A design of attention and state-space layers: a prompt and decoding behind prompts.
        {"name": "lukelix_prompt", **_case("lukelix-2k", tokens=1999)},
        {"name": "lukelix_decode_8", **_case("lukelix-2k", singles=8, least=1024, most=2047)},
    ]


def draw(rng) -> dict:
    def between(low: int, high: int) -> int:  # spread over the logarithm
        return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))

    def singles_of(count: int, longest: int, total: int) -> dict:
        most = between(64, max(64, min(longest, total // count)))
        return {"singles": count, "least": rng.randint(max(1, most // 4), most), "most": most}

    kind = rng.choice(["decode", "decode", "prompt", "prompt", "portion", "mixed", "decode32", "prompt32", "design"])
    if kind == "decode":
        return _case(rng.choice(["2k", "7b", "7b"]), **singles_of(between(1, 64), 16384, 131072))
    if kind == "prompt":
        return _case(rng.choice(["2k", "7b", "7b"]), tokens=between(16, 2048))
    if kind == "portion":
        return _case("7b", tokens=between(64, 1536), held=between(256, 16384))
    if kind == "mixed":
        return _case(rng.choice(["7b", "14b"]), tokens=between(64, 2016), **singles_of(between(2, 32), 2047, 65536))
    if kind == "decode32":
        return _case("7b-4layers", "float32", **singles_of(between(1, 32), 2048, 32768))
    if kind == "prompt32":
        return _case("7b-4layers", "float32", tokens=between(16, 500))
    if rng.random() < 0.5:
        return _case("lukelix-2k", tokens=between(32, 2048))
    return _case("lukelix-2k", **singles_of(between(1, 32), 2048, 16384))


# -- inputs ------------------------------------------------------------------------------------------------


def _dtype(case: dict) -> torch.dtype:
    return {"bfloat16": torch.bfloat16, "float32": torch.float32}[case["dtype"]]


def _generator(*key) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(zlib.crc32(repr(key).encode()))


def _weight(name: str, shape: tuple[int, ...], dtype: torch.dtype) -> torch.Tensor:
    """A checkpoint's tensor: matrices N(0, 0.02), those that end a residual branch smaller by the root of twice the
    7B shape's layers, token tables N(0, 1) (so that a layer adds to the stream what it adds in a trained model and
    rounding does not grow from layer to layer), norm gains around 1, a selective state's constants as such layers are
    initialised (rates 1 to 16, steps 0.001 to 0.1)."""
    generator = _generator("weight", name, tuple(shape))
    leaf = name.rsplit(".", 1)[-1]
    if leaf in ("A_log", "dt_bias"):
        u = torch.rand(shape, generator=generator, device=DEVICE)
        if leaf == "A_log":
            return torch.log(1.0 + 15.0 * u)
        step = torch.exp(u * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
        return step + torch.log(-torch.expm1(-step))
    if leaf == "D":
        return torch.ones(shape, device=DEVICE)
    if leaf == "conv":  # taps whose sum keeps the input's size
        return (torch.randn(shape, generator=generator, device=DEVICE) * 0.5).to(dtype)
    std = 0.02
    if "embed" in name or name == "bigram":
        std = 1.0
    elif "o_proj" in name or "down_proj" in name:
        std /= math.sqrt(2 * 28)
    values = torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, std, generator=generator)
    is_gain = "norm" in name and not name.endswith(".b")
    return values + 1.0 if is_gain else values


@functools.lru_cache(maxsize=None)
def _model(shape: str, dtype: torch.dtype):
    from turboserve_amd.engine.loading import build_model, make_runtime
    from turboserve_amd.weights.loader import TensorSupply

    _, model = build_model(SHAPES[shape], make_runtime(dtype, DEVICE))
    specs = model.tensor_specs()
    model.load(TensorSupply(specs, lambda name: _weight(name, tuple(specs[name].shape), dtype)))
    return model


def _contexts(case: dict) -> list[int]:
    """What the single-token requests hold: spread between the case's bounds, the same for every seed."""
    return [case["least"] + round((case["most"] - case["least"]) * ((i * 0.6180339887498949) % 1.0)) for i in range(case["singles"])]


def _tokens(case: dict, seed: int, request: int, count: int) -> list[int]:
    shape = SHAPES[case["model"]]
    vocab = shape.get("vocab_size") or shape["vocab"]
    generator = torch.Generator().manual_seed(zlib.crc32(repr(("tokens", seed, request)).encode()))
    return torch.randint(0, vocab, (count,), generator=generator).tolist()


def _cached(case: dict, seed: int, layer: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Keys and values of a layer that the requests' earlier tokens left: ``[tokens, KV heads, head size]``, the requests
    one behind the other, spread as random weights of this width spread them."""
    shape = SHAPES[case["model"]]
    size = (sum(_contexts(case)) + case["held"], shape["num_key_value_heads"], shape["head_dim"])
    spread = 0.02 * math.sqrt(shape["hidden_size"])
    generator = _generator("cache", seed, layer)
    return tuple(torch.empty(size, dtype=_dtype(case), device=DEVICE).normal_(0.0, spread, generator=generator) for _ in range(2))


def prepare(case: dict, seed: int) -> dict:
    from turboserve_amd.cache.manager import CacheManager
    from turboserve_amd.engine.batch import StepEntry
    from turboserve_amd.engine.loading import build_storage
    from turboserve_amd.engine.runner import ModelRunner

    model = _model(case["model"], _dtype(case))
    contexts = _contexts(case)
    requests = [(held, 1) for held in contexts]
    if case["tokens"]:
        requests.append((case["held"], case["tokens"]))
    pages = sum(-(-(held + new) // PAGE) for held, new in requests)
    storage = build_storage(model, pages, PAGE, len(requests))
    manager = CacheManager(storage.layout.windows(), pages, PAGE, len(requests), chunks=storage.layout.chunks(), kept=storage.layout.kept())
    runner = ModelRunner(model, storage)
    stateful = bool(storage.states)

    entries, fresh, earlier, where = [], [], [], []
    for index, (held, new) in enumerate(requests):
        cache = manager.admit(index)
        slots = manager.append(index, held) if held else []
        tokens = _tokens(case, seed, index, (held if stateful else 0) + new)
        for first in range(0, held if stateful else 0, 2048):  # the earlier tokens run through the engine
            count = min(2048, held - first)
            earlier.append((StepEntry(index, tokens[first:first + count], first, cache.tables, [s[first:first + count] for s in slots],
                                      cache.state_slot), [cache.state_slot] if first == 0 else []))
        if held:
            where += list(slots[0])
        last = manager.append(index, new)
        entries.append(StepEntry(index, tokens[-new:], held, cache.tables, last, cache.state_slot, [new - 1]))
        if held == 0:
            fresh.append(cache.state_slot)
    state = {"runner": runner, "entries": entries, "fresh": fresh, "manager": manager}
    if not case["tokens"]:
        run(state)  # a serving program has recorded its steps of single tokens long before
    if stateful:
        for entry, slots in earlier:
            entry.tables = manager.get(entry.request).tables
            runner.step([entry], fresh_state_slots=slots)
    elif where:
        at = torch.tensor(where, device=DEVICE)
        page, offset = at // PAGE, at % PAGE
        for layer, view in enumerate(runner.views):
            keys, values = _cached(case, seed, layer)
            view.k[page, :, offset, :] = keys
            view.v[page, :, :, offset] = values
    return state


def run(state: dict) -> torch.Tensor:
    return state["runner"].step(state["entries"], fresh_state_slots=state["fresh"])


# -- what a step cannot do without ---------------------------------------------------------------------------


def work(case: dict) -> dict:
    shape, itemsize = SHAPES[case["model"]], 4 if case["dtype"] == "float32" else 2
    contexts = _contexts(case)
    rows, wanted = case["singles"] + case["tokens"], case["singles"] + (1 if case["tokens"] else 0)
    # (query, key) pairs: a token sees what its request held and the new tokens up to itself
    pairs = sum(c + 1 for c in contexts) + case["tokens"] * case["held"] + case["tokens"] * (case["tokens"] + 1) / 2
    cached, written = sum(contexts) + case["held"], rows
    if case["model"] == "lukelix-2k":
        width, vocab, attention, state = shape["width"], shape["vocab"], ATTENTION, SELECTIVE
        heads, kv, dim = attention["heads"] * attention["dim"], attention["kv_heads"] * attention["dim"], attention["dim"]
        inner, both = state["heads"] * state["vdim"], 2 * state["groups"] * state["state"]
        weights = 3 * (2 * width * heads + 2 * width * 8192) + 2 * 2 * width * kv + 9 * (width * (2 * inner + both + state["heads"]) + inner * width)
        selective = state["heads"] * state["state"] * state["vdim"]
        states = 9 * wanted * 2 * 4 * selective  # 32-bit states read and written
        moved = states + itemsize * (2 * 2 * kv * (cached + written) + 2 * kv * cached)  # two layers keep keys and values, three read
        flops = 2.0 * rows * weights + 4.0 * pairs * heads * 3 + 9 * rows * 4.0 * selective
    else:
        width, vocab, layers = shape["hidden_size"], shape["vocab_size"], shape["num_hidden_layers"]
        heads, kv = shape["num_attention_heads"] * shape["head_dim"], shape["num_key_value_heads"] * shape["head_dim"]
        weights = layers * (2 * width * heads + 2 * width * kv + 3 * width * shape["intermediate_size"])
        moved = itemsize * layers * 2 * kv * (cached + written)
        flops = 2.0 * rows * weights + 4.0 * layers * pairs * heads
    moved += itemsize * (weights + vocab * width + rows * width) + 4.0 * wanted * vocab
    return {"bytes": float(moved), "flops": flops + 2.0 * wanted * vocab * width}


def tolerance(case: dict) -> dict:
    """About four times what the path's logits were from 64 bits when the cases were written: 2.2e-6 in 32-bit, 0.003 to
    0.009 with bfloat16 weights and activations (28 layers), twice that with 48 layers and in the other design."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 0.025 if case["model"] in ("2k", "7b") else 0.03}


# -- the same logits in 64 bits ------------------------------------------------------------------------------


def exact(case: dict, seed: int):
    return _exact_lukelix(case, seed) if case["model"] == "lukelix-2k" else _exact_qwen2(case, seed)


def _product(x: torch.Tensor, name: str, shape: tuple[int, int], dtype: torch.dtype, bias: str | None = None) -> torch.Tensor:
    y = x @ _weight(name, shape, dtype).double().T
    return y if bias is None else y + _weight(bias, shape[:1], dtype).double()


def _rms_norm(x: torch.Tensor, name: str, eps: float, dtype: torch.dtype) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * _weight(name, (x.shape[-1],), dtype).double()


def _turn_halves(x: torch.Tensor, positions: torch.Tensor, base: float) -> torch.Tensor:
    """``x [T, heads, D]`` rotated, element ``i`` paired with ``i + D / 2``."""
    half = x.shape[-1] // 2
    angle = positions.double()[:, None] * base ** (-torch.arange(half, device=x.device).double() / half)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> torch.Tensor:
    """The last ``len(q)`` positions of a request over its keys: ``[T, H, D]``, ``[S, G, D]`` twice -> ``[T, H D]``."""
    count, total, per = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    seen = torch.arange(total, device=q.device)[None] <= torch.arange(total - count, total, device=q.device)[:, None]
    out = torch.empty_like(q)
    for g in range(k.shape[1]):
        for h in range(g * per, (g + 1) * per):
            scores = (q[:, h] @ k[:, g].T * scale).masked_fill(~seen, -math.inf)
            out[:, h] = torch.softmax(scores, -1) @ v[:, g]
    return out.reshape(count, -1)


def _exact_qwen2(case: dict, seed: int) -> torch.Tensor:
    shape, dtype = SHAPES[case["model"]], _dtype(case)
    width, ff, vocab, eps = shape["hidden_size"], shape["intermediate_size"], shape["vocab_size"], shape["rms_norm_eps"]
    heads, kv_heads, dim = shape["num_attention_heads"], shape["num_key_value_heads"], shape["head_dim"]
    requests = [(c, 1) for c in _contexts(case)] + ([(case["held"], case["tokens"])] if case["tokens"] else [])
    ids = [t for i, (_, new) in enumerate(requests) for t in _tokens(case, seed, i, new)]
    positions = torch.tensor([held + t for held, new in requests for t in range(new)], device=DEVICE)
    x = _weight("model.embed_tokens.weight", (vocab, width), dtype)[torch.tensor(ids, device=DEVICE)].double()
    for layer in range(shape["num_hidden_layers"]):
        at = f"model.layers.{layer}."
        h = _rms_norm(x, at + "input_layernorm.weight", eps, dtype)
        q, k, v = (
            _product(h, f"{at}self_attn.{p}_proj.weight", (n * dim, width), dtype, f"{at}self_attn.{p}_proj.bias").view(len(ids), n, dim)
            for p, n in (("q", heads), ("k", kv_heads), ("v", kv_heads)))
        q, k = (_turn_halves(t, positions, shape["rope_theta"]) for t in (q, k))
        old_k, old_v = _cached(case, seed, layer)
        mixed, row, old = [], 0, 0
        for held, new in requests:
            keys = torch.cat([old_k[old:old + held].double(), k[row:row + new]])
            values = torch.cat([old_v[old:old + held].double(), v[row:row + new]])
            mixed.append(_attend(q[row:row + new], keys, values, dim ** -0.5))
            row, old = row + new, old + held
        x = x + _product(torch.cat(mixed), at + "self_attn.o_proj.weight", (width, heads * dim), dtype)
        h = _rms_norm(x, at + "post_attention_layernorm.weight", eps, dtype)
        gate = torch.nn.functional.silu(_product(h, at + "mlp.gate_proj.weight", (ff, width), dtype))
        x = x + _product(gate * _product(h, at + "mlp.up_proj.weight", (ff, width), dtype), at + "mlp.down_proj.weight", (width, ff), dtype)
    ends = torch.tensor([new for _, new in requests]).cumsum(0).to(DEVICE) - 1
    return _product(_rms_norm(x[ends], "model.norm.weight", eps, dtype), "lm_head.weight", (vocab, width), dtype)


def _layer_norm(x: torch.Tensor, name: str, eps: float, dtype: torch.dtype) -> torch.Tensor:
    centred = x - x.mean(-1, keepdim=True)
    size = (x.shape[-1],)
    return centred / torch.sqrt((centred * centred).mean(-1, keepdim=True) + eps) * _weight(name, size, dtype).double() + _weight(name + ".b", size, dtype).double()


def _turn_pairs(x: torch.Tensor, rot: dict) -> torch.Tensor:
    """``x [T, heads, D]`` rotated at positions ``0 ..``, neighbours paired, long wavelengths stretched."""
    f = rot["base"] ** (-2.0 * torch.arange(rot["dims"] // 2, device=x.device).double() / rot["dims"])
    s = rot["scaling"]
    wave = 2 * math.pi / f
    blend = ((s["original"] / wave - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    f = (1 - blend) * f / s["factor"] + blend * f
    angle = torch.arange(x.shape[0], device=x.device).double()[:, None] * f
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _convolved(u: torch.Tensor, name: str, dtype: torch.dtype) -> torch.Tensor:
    """Every channel of ``u [T, C]`` with its taps, over the tokens up to each."""
    taps = _weight(name, (u.shape[1], 4), dtype).double()
    padded = torch.cat([u.new_zeros(3, u.shape[1]), u])
    return sum(taps[:, j] * padded[j:j + u.shape[0]] for j in range(4))


def _exact_lukelix(case: dict, seed: int) -> torch.Tensor:
    shape, dtype, eps = SHAPES["lukelix-2k"], _dtype(case), SHAPES["lukelix-2k"]["norm"]["eps"]
    width, rule = shape["width"], shape["embedding"]["bigram"]
    requests = [(c, 1) for c in _contexts(case)] + ([(case["held"], case["tokens"])] if case["tokens"] else [])
    lengths = [held + new for held, new in requests]
    ids = [_tokens(case, seed, i, n) for i, n in enumerate(lengths)]
    rows = [t for one in ids for t in [rule["buckets"]] + [(a * rule["mul_prev"] + b * rule["mul_cur"]) % rule["buckets"] for a, b in zip(one, one[1:])]]
    x = _weight("embed", (shape["vocab"], width), dtype)[torch.tensor([t for one in ids for t in one], device=DEVICE)].double()
    x = x + _weight("bigram", (rule["buckets"] + 1, width), dtype)[torch.tensor(rows, device=DEVICE)].double()

    def each(call, *tensors):  # request by request
        return torch.cat([call(*parts) for parts in zip(*(t.split(lengths) for t in tensors))])

    kept: dict = {}
    for index, layer in enumerate(shape["layers"]):
        at, m = f"l{index}.mix", layer["mixer"]
        if layer["type"] == "attention":
            def projected(which: str, heads: int, turned: bool) -> torch.Tensor:
                u = _product(x, f"{at}.{which}", (heads * m["dim"], width), dtype, f"{at}.{which}.b")
                u = each(lambda t: _convolved(t, f"{at}.{which}.conv", dtype), u).view(-1, heads, m["dim"])
                return each(lambda t: _turn_pairs(t, m["rot"]), _rms_norm(u, f"{at}.{which}.norm", eps, dtype)) if turned else u

            if "kv_from" not in m:
                kept[index] = projected("k", m["kv_heads"], True), projected("v", m["kv_heads"], False)
            mixed = each(lambda q, k, v: _attend(q, k, v, m["scale"]), projected("q", m["heads"], True), *kept[m.get("kv_from", index)])
            mixed = _product(mixed, at + ".o", (width, m["heads"] * m["dim"]), dtype)
        else:
            mixed = _exact_selective(x, at, m, lengths, eps, dtype, each)
        x = x + _layer_norm(mixed, f"l{index}.norm1", eps, dtype)
        if layer["mlp"]:
            ff = layer["mlp"]["ff"]
            h = torch.relu(_product(x, f"l{index}.mlp.up", (ff, width), dtype)) ** 2
            x = x + _layer_norm(_product(h, f"l{index}.mlp.down", (width, ff), dtype), f"l{index}.norm2", eps, dtype)
    ends = torch.tensor(lengths).cumsum(0).to(DEVICE) - 1
    return _product(_layer_norm(x[ends], "final.norm", eps, dtype), "head", (shape["vocab"], width), dtype)


def _exact_selective(x: torch.Tensor, at: str, m: dict, lengths: list[int], eps: float, dtype: torch.dtype, each) -> torch.Tensor:
    width, H, P, N, G = x.shape[1], m["heads"], m["vdim"], m["state"], m["groups"]
    inner = H * P
    z, u, dt = _product(x, at + ".in", (2 * inner + 2 * G * N + H, width), dtype).split([inner, inner + 2 * G * N, H], 1)
    u = torch.nn.functional.silu(each(lambda t: _convolved(t, at + ".conv", dtype), u) + _weight(at + ".conv.b", (inner + 2 * G * N,), dtype).double())
    dt = torch.nn.functional.softplus(dt + _weight(at + ".dt_bias", (H,), dtype).double())
    decay = torch.exp(-dt * torch.exp(_weight(at + ".A_log", (H,), dtype).double()))
    value, b, c = u.split([inner, G * N, G * N], 1)
    value = value.reshape(-1, H, P)
    b, c = (t.reshape(-1, G, N).repeat_interleave(H // G, 1) for t in (b, c))

    def padded(t: torch.Tensor) -> torch.Tensor:  # [requests, tokens of the longest, ...], then token by token
        return torch.nn.utils.rnn.pad_sequence(list(t.split(lengths)), batch_first=True).transpose(0, 1).contiguous()

    walk = [padded(t) for t in (decay, dt[:, :, None] * value, b, c)]
    state = x.new_zeros(len(lengths), H, N, P)
    out = []
    for a, v, key, query in zip(*walk):
        state = torch.addcmul(key[..., None] * v[..., None, :], a[..., None, None], state)
        out.append((query[..., None, :] @ state)[..., 0, :])
    y = torch.stack(out, 1)
    y = torch.cat([y[i, :n] for i, n in enumerate(lengths)]) + _weight(at + ".D", (H,), dtype).double()[:, None] * value
    y = (y.reshape(-1, inner) * torch.nn.functional.silu(z)).view(-1, m["norm_groups"], inner // m["norm_groups"])
    y = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps)).reshape(-1, inner) * _weight(at + ".norm", (inner,), dtype).double()
    return _product(y, at + ".o", (width, inner), dtype)
