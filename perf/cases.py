"""The work whose speed this repository answers for, as cases with inputs, one pass, and a tolerance.

Each case is a plain dict; ``kind`` says which public entry points it goes through:

``linear``   one call of a linear: the module a rollout's policy holds (``Int4Linear``, prepacked or not), or the
             torch operators over the canonical tensors (``vrl_hip::int4_gemv``, ``vrl_hip::int4_gate_up_silu``)
``grouped``  the weight set of a decoder as one grouped launch (``GroupedGemv``)
``decode``   one decode step of a Llama trunk (``NativeDecodeTrunk``) and its image-token head
``sample``   the head and the guided draw of a decode step (``head_sample``)
``prompt``   the linears of a prompt pass through the modules, without gradients
``replay``   the same modules in a training replay: forward, and backward to their inputs

Shapes are those of the benchmark's workloads: a 24 x (2048, 5632) trunk with 16 heads and a 30 x (4096, 11008)
trunk with 32, a head of 16384 image tokens, prompts of 256 tokens padded on the left, images of 576 tokens.
"""

from __future__ import annotations

import math
import types

import torch

from visionrl_amd import ops
from visionrl_amd.decode_step import NativeDecodeTrunk
from visionrl_amd.linear import Int4Linear, Int4LlamaMLP

HEAD = 16384
PROMPT, IMAGE = 256, 576
LARGE = {"layers": 30, "hidden": 4096, "inter": 11008, "heads": 32}
SMALL = {"layers": 24, "hidden": 2048, "inter": 5632, "heads": 16}


def listed() -> list[dict]:
    return [
        # the smallest thing a rollout does: one projection of one token (launch latency, host time)
        {"name": "linear_2048_m1", "kind": "linear", "form": "module", "prepacked": True,
         "M": 1, "K": 2048, "N": 2048, "G": 128},
        # the operator over canonical tensors at a ragged width, small groups and an odd row count
        {"name": "op_5632x2050_g32_m7", "kind": "linear", "form": "op", "prepacked": False,
         "M": 7, "K": 5632, "N": 2050, "G": 32},
        # decoder weights once each, nothing waiting for anything: the streaming rate (nine layers are 241 MB)
        {"name": "grouped_9x2048_m1", "kind": "grouped", "M": 1, "head": False, "layers": 9, "hidden": 2048,
         "inter": 5632},
        # the same at the rollout batch of 16 samples with guidance, plus the head
        {"name": "grouped_8x2048_head_m32", "kind": "grouped", "M": 32, "head": True, "layers": 8, "hidden": 2048,
         "inter": 5632},
        # a decode step for one image (two rows: conditional and unconditional), early in the image
        {"name": "decode_24x2048_b1", "kind": "decode", "B": 1, "slots": 330, "lora": 0, **SMALL, "kv_heads": 16},
        # a decode step of the default rollout: 8 samples, rank-32 adapters on q, k, v, o; middle of the image
        {"name": "decode_24x2048_b8_lora", "kind": "decode", "B": 8, "slots": 544, "lora": 32, **SMALL,
         "kv_heads": 16},
        # the largest rollout batch of the benchmark, late in the image (the caches are what is read)
        {"name": "decode_24x2048_b16", "kind": "decode", "B": 16, "slots": 700, "lora": 0, **SMALL, "kv_heads": 16},
        # the larger trunk at 4 samples
        {"name": "decode_30x4096_b4", "kind": "decode", "B": 4, "slots": 400, "lora": 0, **LARGE, "kv_heads": 32},
        # what follows every decode step: head, guidance, draw, log-probability
        {"name": "sample_2048_b16", "kind": "sample", "B": 16, "K": 2048, "V": HEAD},
        # the prompt pass of one image (2 x 256 rows), four layers of it
        {"name": "prompt_4x2048_rows512", "kind": "prompt", "rows": 512, "layers": 4, "hidden": 2048, "inter": 5632},
        # the prompt pass of 16 images (32 x 256 rows)
        {"name": "prompt_4x2048_rows8192", "kind": "prompt", "rows": 8192, "layers": 4, "hidden": 2048, "inter": 5632},
        # a training micro-batch: two samples of prompt and image tokens, forward and backward through two layers
        {"name": "replay_2x2048_rows1664", "kind": "replay", "rows": 2 * (PROMPT + IMAGE), "layers": 2,
         "hidden": 2048, "inter": 5632},
    ]


def _log(rng, low: int, high: int) -> int:
    """A whole number between ``low`` and ``high``, even over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "grouped", "decode", "decode", "decode", "sample", "prompt", "prompt",
                       "replay"])
    if kind == "linear":
        G = rng.choice([32, 64, 128, 128])
        form = rng.choice(["module", "module", "op", "gate_up"])
        N = _log(rng, 512, 11008)
        return {"kind": kind, "form": form, "prepacked": form == "module" and rng.random() < 0.75,
                "M": _log(rng, 1, 32), "K": 128 * _log(rng, 4, 44), "N": N + N % 2 if form == "gate_up" else N, "G": G}
    if kind == "grouped":
        return {"kind": kind, "M": _log(rng, 1, 32), "head": rng.random() < 0.5, "layers": rng.randint(3, 8),
                "hidden": 2048, "inter": 5632}
    if kind == "decode":
        large = rng.random() < 0.25
        shape = dict(LARGE if large else SMALL)
        shape["layers"] = rng.randint(6, shape["layers"])
        return {"kind": kind, "B": _log(rng, 1, 4 if large else 16), "slots": rng.randint(60, PROMPT + IMAGE - 1),
                "lora": rng.choice([0, 0, 16, 32]), **shape, "kv_heads": shape["heads"] // rng.choice([1, 1, 4])}
    if kind == "sample":
        return {"kind": kind, "B": _log(rng, 1, 16), "K": 2048 * rng.choice([1, 1, 2]), "V": 16 * _log(rng, 256, 1024)}
    if kind == "prompt":
        return {"kind": kind, "rows": 2 * _log(rng, 1, 16) * rng.randint(20, PROMPT), "layers": rng.randint(1, 4),
                "hidden": 2048, "inter": 5632}
    return {"kind": kind, "rows": _log(rng, 40, 3 * (PROMPT + IMAGE)), "layers": rng.randint(1, 2), "hidden": 2048,
            "inter": 5632}


# ------------------------------------------------------------------------------------------------ inputs
class _Inputs:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.made = None    # a list: the operand triples, in the order they are made (for ``exact``)

    def normal(self, *shape, scale: float = 1.0, dtype=torch.bfloat16) -> torch.Tensor:
        return torch.randn(shape, generator=self.gen, device=self.dev, dtype=dtype).mul_(scale)

    def words(self, *shape) -> torch.Tensor:
        return torch.randint(-2 ** 31, 2 ** 31, shape, generator=self.gen, device=self.dev,
                             dtype=torch.int64).to(torch.int32)

    def packed(self, K: int, N: int, G: int, scale: float = 0.02):
        """Uniform nibbles, scales of ``|N(0, scale)|``, uniform zero-points: the operand triple of a linear."""
        groups = K // G
        scales = self.normal(N, groups, scale=scale, dtype=torch.float32).abs_().clamp_(min=scale / 20)
        qzeros = self.words(N, (groups + 7) // 8)
        if groups % 8:
            qzeros[:, -1] &= (1 << (4 * (groups % 8))) - 1
        triple = self.words(N, K // 8), scales.to(torch.bfloat16), qzeros
        if self.made is not None:
            self.made.append((*triple, G))
        return triple

    def linear(self, K: int, N: int, G: int = 128, scale: float = 0.02, prepack: bool = True) -> Int4Linear:
        module = Int4Linear.from_packed(*self.packed(K, N, G, scale), G)
        return module.prepack_() if prepack else module

    def norm(self, hidden: int):
        return types.SimpleNamespace(weight=self.normal(hidden, scale=0.1).add_(1.0), variance_epsilon=1e-6)


class _Adapted(torch.nn.Module):
    """A projection under one low-rank adapter, with the attributes of peft's wrapper."""

    def __init__(self, inp: _Inputs, base: Int4Linear, rank: int):
        super().__init__()
        self.base_layer = base
        holder = lambda w: types.SimpleNamespace(weight=torch.nn.Parameter(w, requires_grad=False), bias=None)
        self.lora_A = {"default": holder(inp.normal(rank, base.in_features, scale=base.in_features ** -0.5,
                                                    dtype=torch.float32))}
        self.lora_B = {"default": holder(inp.normal(base.out_features, rank, scale=0.02, dtype=torch.float32))}
        self.scaling, self.active_adapters = {"default": 2.0}, ["default"]
        self.merged = self.disable_adapters = False


# weights of the scale trained layers have (0.02 root mean square): hidden states stay of order one
_TRUNK_SCALE = 0.003


def _decoder_layer(inp: _Inputs, case: dict):
    hidden, inter = case["hidden"], case["inter"]
    dim = hidden // case["heads"]
    wide = case["kv_heads"] * dim
    attn = types.SimpleNamespace(scaling=dim ** -0.5)
    linears = {name: inp.linear(hidden, n, scale=_TRUNK_SCALE)
               for name, n in (("q_proj", hidden), ("k_proj", wide), ("v_proj", wide), ("o_proj", hidden))}
    for name, module in linears.items():
        setattr(attn, name, _Adapted(inp, module, case["lora"]) if case["lora"] else module)
    mlp = Int4LlamaMLP(types.SimpleNamespace(
        gate_proj=inp.linear(hidden, inter, scale=_TRUNK_SCALE, prepack=False),
        up_proj=inp.linear(hidden, inter, scale=_TRUNK_SCALE, prepack=False),
        down_proj=inp.linear(inter, hidden, scale=_TRUNK_SCALE, prepack=False)), 128).prepack_()
    return types.SimpleNamespace(self_attn=attn, mlp=mlp, input_layernorm=inp.norm(hidden),
                                 post_attention_layernorm=inp.norm(hidden))


def _rotary(dim: int, device):
    """The rotary tables of a Llama trunk: ``(x, position_ids) -> (cos, sin)``."""
    inv = 10000.0 ** (-torch.arange(0, dim, 2, device=device, dtype=torch.float32) / dim)

    def tables(x, position_ids):
        angle = position_ids[..., None].float() * inv
        angle = torch.cat([angle, angle], dim=-1)
        return angle.cos().to(x.dtype), angle.sin().to(x.dtype)

    return tables


def _prepare_decode(case: dict, inp: _Inputs):
    rows, slots, length = 2 * case["B"], case["slots"], PROMPT + IMAGE
    dim = case["hidden"] // case["heads"]
    layers = [_decoder_layer(inp, case) for _ in range(case["layers"])]
    trunk = types.SimpleNamespace(
        config=types.SimpleNamespace(hidden_size=case["hidden"], num_attention_heads=case["heads"],
                                     num_key_value_heads=case["kv_heads"], head_dim=dim),
        layers=layers, norm=inp.norm(case["hidden"]), rotary_emb=_rotary(dim, inp.dev))
    cached = lambda: inp.normal(rows, case["kv_heads"], length, dim)
    cache = types.SimpleNamespace(layers=[types.SimpleNamespace(keys=cached(), values=cached(), is_initialized=True)
                                          for _ in layers])
    mask = torch.ones((rows, length), dtype=torch.uint8, device=inp.dev)
    pad = torch.randint(0, min(slots, PROMPT) // 2, (rows, 1), generator=inp.gen, device=inp.dev)
    mask[torch.arange(length, device=inp.dev)[None] < pad] = 0          # prompts are padded on the left
    embedded = inp.normal(rows, 1, case["hidden"])
    step = NativeDecodeTrunk(trunk, cache, embedded, mask,
                             torch.full((1,), slots, dtype=torch.int64, device=inp.dev))
    head = inp.linear(case["hidden"], HEAD, scale=_TRUNK_SCALE)
    appended = [t[:, :, slots] for layer in cache.layers for t in (layer.keys, layer.values)]
    return {"trunk": trunk, "cache": cache, "mask": mask, "embedded": embedded, "step": step, "short": step.short_form(slots), "head": head, "appended": appended}


def _prepare_modules(case: dict, inp: _Inputs):
    """Decoder layers' int4 modules as a quantised policy holds them, and the inputs that reach them."""
    hidden, inter, rows = case["hidden"], case["inter"], case["rows"]
    layers = []
    for _ in range(case["layers"]):
        q, k, v, o = (inp.linear(hidden, hidden) for _ in range(4))
        q.group_with(k, v)
        mlp = Int4LlamaMLP(types.SimpleNamespace(
            gate_proj=inp.linear(hidden, inter, prepack=False), up_proj=inp.linear(hidden, inter, prepack=False),
            down_proj=inp.linear(inter, hidden, prepack=False)), 128).prepack_()
        layers.append((q, k, v, o, mlp))
    state = {"layers": layers,
             "x": [tuple(inp.normal(rows, hidden) for _ in range(3)) for _ in layers]}
    if case["kind"] == "replay":
        state["grads"] = [tuple(inp.normal(rows, hidden) for _ in range(5)) for _ in layers]
    return state


def prepare(case: dict, seed: int):
    return _prepare(case, _Inputs(seed))


def _prepare(case: dict, inp: _Inputs):
    kind = case["kind"]
    if kind == "linear":
        M, K, N, G = case["M"], case["K"], case["N"], case["G"]
        x = inp.normal(M, K)
        if case["form"] == "module":
            return {"x": x, "module": inp.linear(K, N, G, prepack=case["prepacked"])}
        return {"x": x, "packed": inp.packed(K, N, G), "op": case["form"], "G": G}
    if kind == "grouped":
        hidden, inter, M = case["hidden"], case["inter"], case["M"]
        problems = []
        weight = lambda K, N: ops.int4_prepack(*inp.packed(K, N, 128), 128)
        for _ in range(case["layers"]):
            a, b, c, d = (inp.normal(M, K) for K in (hidden, hidden, hidden, inter))
            problems += [(a, weight(hidden, hidden), False) for _ in range(3)]
            problems += [(b, weight(hidden, hidden), False)]
            problems += [(c, weight(hidden, inter), False) for _ in range(2)]
            problems += [(d, weight(inter, hidden), False)]
        if case["head"]:
            problems.append((inp.normal(M, hidden), weight(hidden, HEAD), False))
        return {"rows": [x for x, _, _ in problems], "plan": ops.GroupedGemv(problems)}
    if kind == "decode":
        return _prepare_decode(case, inp)
    if kind == "sample":
        B, K, V = case["B"], case["K"], case["V"]
        return {"x": inp.normal(2 * B, K), "head": ops.int4_prepack(*inp.packed(K, V, 128, _TRUNK_SCALE), 128),
                "noise": torch.empty((B, V), dtype=torch.bfloat16, device=inp.dev).exponential_(generator=inp.gen),
                "workspace": ops.head_sample_workspace(B, V, inp.dev),
                "logits": torch.empty((2 * B, V), dtype=torch.bfloat16, device=inp.dev)}
    return _prepare_modules(case, inp)


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    with torch.no_grad():
        if "module" in state:
            return state["module"](state["x"])
        if "op" in state:
            op = ops.int4_gate_up_silu if state["op"] == "gate_up" else ops.int4_gemv
            return op(state["x"], *state["packed"], state["G"])
        if "plan" in state:
            return state["plan"].launch()
        if "step" in state:
            hidden = state["step"].run(state["short"])
            return {"hidden": hidden, "logits": state["head"](hidden), "appended": state["appended"]}
        if "noise" in state:
            token, logprob = ops.head_sample(state["x"], state["head"], 5.0, 1.0, noise=state["noise"],
                                             workspace=state["workspace"], logits_out=state["logits"])
            return {"token": token, "logprob": logprob, "logits": state["logits"]}
        if "grads" not in state:
            return [(q(x), k(x), v(x), o(a), mlp(h))
                    for (q, k, v, o, mlp), (x, a, h) in zip(state["layers"], state["x"])]
    out = []
    for (q, k, v, o, mlp), inputs, grads in zip(state["layers"], state["x"], state["grads"]):
        x, a, h = (t.detach().requires_grad_() for t in inputs)
        ys = (q(x), k(x), v(x), o(a), mlp(h))
        out.append((*(y.detach() for y in ys), *torch.autograd.grad(ys, (x, a, h), grads)))
    return out


# ------------------------------------------------------------------------------------------------ what it takes
def _weight_bytes(K: int, N: int, G: int = 128) -> float:
    return K * N / 2 + (K // G) * N * 2.5


def _layer_shapes(case: dict):
    hidden, inter = case["hidden"], case["inter"]
    kv = hidden if "heads" not in case else hidden * case.get("kv_heads", case["heads"]) // case["heads"]
    return [(hidden, hidden), (hidden, kv), (hidden, kv), (hidden, hidden), (hidden, inter), (hidden, inter),
            (inter, hidden)]


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("linear", "sample"):
        M, K = (case["M"], case["K"]) if kind == "linear" else (2 * case["B"], case["K"])
        N = case["N"] if kind == "linear" else case["V"]
        columns = N // 2 if case.get("form") == "gate_up" else N
        extra = case["B"] * N * 2 if kind == "sample" else 0            # the draws
        return {"bytes": _weight_bytes(K, N, case.get("G", 128)) + 2 * M * (K + columns) + extra,
                "flops": 2 * M * K * N}
    shapes = _layer_shapes(case) * case["layers"]
    if case.get("head") or kind == "decode":
        shapes.append((case["hidden"], HEAD))
    weights, products = sum(_weight_bytes(K, N) for K, N in shapes), sum(K * N for K, N in shapes)
    if kind == "grouped":
        M = case["M"]
        return {"bytes": weights + 2 * M * sum(K + N for K, N in shapes), "flops": 2 * M * products}
    if kind == "decode":
        rows, dim = 2 * case["B"], case["hidden"] // case["heads"]
        slot = 2 * 2 * rows * case["kv_heads"] * dim * case["layers"]     # keys and values of one slot, bf16
        adapters = sum(case["lora"] * (K + N) * 4 for K, N in _layer_shapes(case)[:4]) * case["layers"]
        return {"bytes": weights + slot * (case["slots"] + 1) + adapters + 2 * rows * (case["hidden"] * 2 + HEAD),
                "flops": rows * (2 * products + adapters / 2 +
                                 4 * case["heads"] * dim * (case["slots"] + 1) * case["layers"])}
    # modules: three inputs and five outputs of [rows, hidden] per layer, and the gradients of both in a replay
    rows, per_layer = case["rows"], 8 * case["rows"] * case["hidden"] * 2 * case["layers"]
    if kind == "prompt":
        return {"bytes": weights + per_layer, "flops": 2 * rows * products}
    return {"bytes": 2 * weights + 2 * per_layer, "flops": 4 * rows * products}


def tolerance(case: dict):
    """Relative errors that sums in another order show, times four."""
    if case["kind"] == "decode":
        return {"rel": 0.02, "max": 0.3}
    if case["kind"] == "sample":
        return {"rel": 0.004, "max": 0.05, "differ": 0.01}
    if case["kind"] in ("prompt", "replay"):
        return {"rel": 0.01, "max": 0.1}
    return {"rel": 0.004, "max": 0.05}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _dense(qweight, scales, qzeros, G: int) -> torch.Tensor:
    """The weight an operand triple stands for: ``(q - z) * s`` rounded to bf16 once, as float64 ``[N, K]``."""
    shifts = torch.arange(0, 32, 4, device=qweight.device, dtype=torch.int32)
    nibbles = lambda t: ((t[..., None] >> shifts) & 15).flatten(1)
    q, z = nibbles(qweight), nibbles(qzeros)[:, :scales.shape[1]]
    q = q.unflatten(1, (-1, G)) - z[..., None]
    return (q.float() * scales.float()[..., None]).to(torch.bfloat16).flatten(1).double()


def _rms(x, norm):
    return norm.weight.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + norm.variance_epsilon)


def _adapted(x, weight, module):
    y = x @ weight.T
    if isinstance(module, _Adapted):
        a, b = (p["default"].weight.data.double() for p in (module.lora_A, module.lora_B))
        y = y + module.scaling["default"] * (x @ a.T @ b.T)
    return y


def _exact_decode(case: dict, state, made) -> dict:
    slot, heads, kv_heads = case["slots"], case["heads"], case["kv_heads"]
    dim = case["hidden"] // heads
    trunk, hidden = state["trunk"], state["embedded"][:, 0].double()
    cos, sin = (t[0].double() for t in trunk.rotary_emb(state["embedded"], torch.full((1, 1), slot,
                                                                                     device=hidden.device)))
    turn = lambda t: t * cos + torch.cat([-t[..., dim // 2:], t[..., :dim // 2]], -1) * sin
    seen, appended = state["mask"][:, None, :slot + 1] != 0, []
    for layer, cached in zip(trunk.layers, state["cache"].layers):
        at, x = layer.self_attn, _rms(hidden, layer.input_layernorm)
        q, k, v = (_adapted(x, _dense(*next(made)), m).unflatten(1, (-1, dim)) for m in (at.q_proj, at.k_proj, at.v_proj))
        q, k = turn(q), turn(k)
        appended += [k, v]
        keys, values = (torch.cat([c[:, :, :slot].double(), new[:, :, None]], 2).repeat_interleave(heads // kv_heads, 1)
                        for c, new in ((cached.keys, k), (cached.values, v)))
        scores = (keys * q[:, :, None]).sum(-1) * at.scaling
        probs = scores.masked_fill(~seen, -math.inf).softmax(-1)
        mixed = (probs[..., None] * values).sum(2).flatten(1)
        hidden = hidden + _adapted(mixed, _dense(*next(made)), at.o_proj)
        x = _rms(hidden, layer.post_attention_layernorm)
        gate, up, down = (_dense(*next(made)) for _ in range(3))
        hidden = hidden + (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T
    hidden = _rms(hidden, trunk.norm)
    return {"hidden": hidden, "logits": hidden @ _dense(*next(made)).T, "appended": appended}


def exact(case: dict, seed: int):
    """What ``run`` returns for these inputs, in 64 bits (the dequantised weights are bf16 by definition)."""
    inp = _Inputs(seed)
    inp.made = []
    state, kind = _prepare(case, inp), case["kind"]
    made = iter(inp.made)
    if kind == "decode":
        return _exact_decode(case, state, made)
    if kind == "linear":
        y = state["x"].double() @ _dense(*next(made)).T
        if case["form"] == "gate_up":
            gate, up = y.chunk(2, dim=1)
            y = torch.nn.functional.silu(gate) * up
        return y
    if kind == "grouped":
        return [x.double() @ _dense(*m).T for x, m in zip(state["rows"], made)]
    if kind == "sample":
        return {"token": None, "logprob": None, "logits": state["x"].double() @ _dense(*next(made)).T}
    out = []
    for n, inputs in enumerate(state["x"]):
        x, a, h = (t.double().requires_grad_(kind == "replay") for t in inputs)
        q, k, v, o, gate, up, down = (_dense(*next(made)) for _ in range(7))
        ys = (x @ q.T, x @ k.T, x @ v.T, a @ o.T, (torch.nn.functional.silu(h @ gate.T) * (h @ up.T)) @ down.T)
        grads = torch.autograd.grad(ys, (x, a, h), [g.double() for g in state["grads"][n]]) if kind == "replay" else ()
        out.append((*(y.detach() for y in ys), *grads))
    return out
