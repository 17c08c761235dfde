"""The workloads this framework's performance is judged on, through its public entry points.

Every case compiles a ``torch.export`` graph once (``chroma_amd.compile``) and then calls the loaded ``Program``
or ``Decoder`` as a user's program does. Two kinds of calls are covered:

* host calls: ``program(x)`` and ``Decoder.append(tokens)``, host arrays in and host arrays out (``mlp``,
  ``forward``, ``decode``, ``prefill``);
* device-resident calls: the inputs lie in the program's input staging (``chroma_hip_input_pointer``) and
  ``chroma_hip_execute`` leaves the results in its output staging (``chain``, ``attention``, ``experts``), as the
  layers of a larger pipeline on the GPU are called.

``exact`` evaluates the same formulas in 64 bits with plain torch; nothing of the framework computes there.
"""

from __future__ import annotations

import math
import os
import shutil
import tempfile
from pathlib import Path

import numpy as np
import torch
from torch import nn

import chroma_amd
from chroma_amd.models.cached import export_cached
from chroma_amd.models.gpt_oss import AttentionBlock, Transformer
from chroma_amd.models.variants import dev, gpt_oss_20b

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
WEIGHTS_SEED = 7  # a user's program has one set of weights; the inputs change from call to call


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: an MLP block over a few rows, where launches and the host link count
        {"name": "mlp_f32_8", "kind": "mlp", "rows": 8, "hidden": 1024, "inner": 4096, "dtype": "f32"},
        # the same block in bfloat16 over an ordinary, ragged batch of rows: mid-sized dense products
        {"name": "mlp_bf16_300", "kind": "mlp", "rows": 300, "hidden": 1024, "inner": 4096, "dtype": "bf16"},
        # the bandwidth workload of bench.py: a fused elementwise chain and a row softmax over 0.5 GB operands
        {"name": "chain_f32_16384x8192", "kind": "chain", "rows": 16384, "columns": 8192, "dtype": "f32"},
        # a GPT-OSS-20B attention layer: a long prompt into an empty cache, ...
        {"name": "attention_prefill_2048", "kind": "attention", "tokens": 2048, "context": 4096, "past": 0, "window": 0},
        # ... a short follow-up prompt behind a conversation, on a windowed layer and with ragged sizes, ...
        {"name": "attention_chunk_100", "kind": "attention", "tokens": 100, "context": 1000, "past": 777, "window": 128},
        # ... and one decode step against a full cache
        {"name": "attention_decode_4096", "kind": "attention", "tokens": 1, "context": 4096, "past": 4096, "window": 0},
        # a GPT-OSS-20B mixture-of-experts layer behind its router: a long prompt, a short ragged one, a decode step
        {"name": "experts_prefill_2048", "kind": "experts", "tokens": 2048},
        {"name": "experts_chunk_100", "kind": "experts", "tokens": 100},
        {"name": "experts_decode_1", "kind": "experts", "tokens": 1},
        # whole models (the 12-layer fp32 dev model): a short uncached forward, a cached decode step whose cache is
        # full, and a prompt through the cached prefill graph
        {"name": "dev_forward_8", "kind": "forward", "tokens": 8},
        {"name": "dev_decode_256", "kind": "decode", "context": 256},
        {"name": "dev_prefill_250", "kind": "prefill", "context": 256, "tokens": 250},
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))


def draw(rng):
    kind = rng.choice(["mlp", "chain", "attention", "attention", "experts", "experts", "forward", "decode", "prefill"])
    if kind == "mlp":
        hidden = rng.choice([512, 1000, 1024, 2048, 2880])
        return {"kind": kind, "rows": _log_uniform(rng, 1, 1024), "hidden": hidden, "inner": 4 * hidden, "dtype": rng.choice(["f32", "bf16"])}
    if kind == "chain":
        columns = _log_uniform(rng, 64, 201088)
        return {"kind": kind, "rows": _log_uniform(rng, 1, min(16384, 16384 * 8192 // columns)), "columns": columns,
                "dtype": rng.choice(["f32", "bf16"])}
    if kind == "attention":
        context = _log_uniform(rng, 128, 4096)
        return {"kind": kind, "tokens": _log_uniform(rng, 1, min(2048, context)), "context": context, "past": rng.randint(0, context),
                "window": rng.choice([0, 128])}
    if kind == "experts":
        return {"kind": kind, "tokens": _log_uniform(rng, 1, 2048)}
    if kind == "forward":
        return {"kind": kind, "tokens": _log_uniform(rng, 1, 64)}
    if kind == "decode":
        return {"kind": kind, "context": _log_uniform(rng, 32, 512)}
    context = _log_uniform(rng, 16, 512)
    return {"kind": kind, "context": context, "tokens": rng.randint(max(2, context // 2), context)}


# -------------------------------------------------------------------------------------- weights and the modules
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(generator, dtype, *shape, std):
    return (torch.randn(*shape, generator=generator, device="cuda") * std).to(dtype)


def _mlp_weights(case):
    g, dtype, h, f = _generator(WEIGHTS_SEED), DTYPES[case["dtype"]], case["hidden"], case["inner"]
    return {
        "norm": torch.ones(h, device="cuda") + 0.1 * torch.randn(h, generator=g, device="cuda"),
        "gate": _weight(g, dtype, f, h, std=h**-0.5),
        "up": _weight(g, dtype, f, h, std=h**-0.5),
        "down": _weight(g, dtype, h, f, std=f**-0.5),
    }


class MLP(nn.Module):
    """RMSNorm, SiLU(gate) * up, down projection, residual."""

    def __init__(self, weights):
        super().__init__()
        for name, value in weights.items():
            setattr(self, name, nn.Parameter(value.cpu(), requires_grad=False))

    def forward(self, x):
        h = x.float()
        h = (h * torch.rsqrt(torch.mean(h**2, dim=-1, keepdim=True) + 1e-5) * self.norm).to(x.dtype)
        inner = nn.functional.silu(nn.functional.linear(h, self.gate)) * nn.functional.linear(h, self.up)
        return nn.functional.linear(inner, self.down) + x


class Chain(nn.Module):
    """A fused elementwise chain and a softmax over its rows."""

    def forward(self, x, y):
        z = torch.tanh(x * 0.5 + y) * torch.sigmoid(y) - torch.exp(torch.clamp(x, -8, 8)) * 1e-3
        return torch.softmax(z, -1)


def _attention_weights():
    c, g, dtype = gpt_oss_20b, _generator(WEIGHTS_SEED), torch.bfloat16
    width = c.head_dim * (c.num_attention_heads + 2 * c.num_key_value_heads)
    heads = c.head_dim * c.num_attention_heads
    return {
        "sinks": _weight(g, dtype, c.num_attention_heads, std=1.0),
        "norm.scale": torch.ones(c.hidden_size, device="cuda") + 0.1 * torch.randn(c.hidden_size, generator=g, device="cuda"),
        "qkv.weight": _weight(g, dtype, width, c.hidden_size, std=c.hidden_size**-0.5),
        "qkv.bias": _weight(g, dtype, width, std=0.1),
        "out.weight": _weight(g, dtype, c.hidden_size, heads, std=heads**-0.5),
        "out.bias": _weight(g, dtype, c.hidden_size, std=0.1),
    }


class Attention(nn.Module):
    """One cached attention layer of the GPT-OSS-20B shape with its norm, projections and residual, as
    ``export_cached`` writes it: x, positions, the cache's keys and values and the mask in; x, new keys, new values out."""

    def __init__(self, weights):
        super().__init__()
        self.block = AttentionBlock(gpt_oss_20b, 1)
        self.block.load_state_dict({name: value.cpu() for name, value in weights.items()})
        self.requires_grad_(False)

    def forward(self, x, positions, keys, values, mask):
        block = self.block
        q, k, v = block.project(x, positions)
        all_k, all_v = torch.cat((keys, k), dim=0), torch.cat((values, v), dim=0)
        steps, kv_heads, group, _ = q.shape
        all_k = all_k[:, :, None, :].expand(-1, -1, group, -1)
        all_v = all_v[:, :, None, :].expand(-1, -1, group, -1)
        scores = torch.einsum("qhmd,khmd->hmqk", q, all_k) * block.sm_scale
        scores = scores + mask[None, None, :, :]
        sinks = block.sinks.reshape(kv_heads, group, 1, 1).expand(-1, -1, steps, -1)
        weights = torch.cat((scores, sinks), dim=-1).softmax(-1)[..., :-1]
        attended = torch.einsum("hmqk,khmd->qhmd", weights, all_v).reshape(steps, -1)
        return x + block.out(attended), k, v


def _expert_weights():
    c, g, dtype = gpt_oss_20b, _generator(WEIGHTS_SEED), torch.bfloat16
    return {
        "norm": torch.ones(c.hidden_size, device="cuda") + 0.1 * torch.randn(c.hidden_size, generator=g, device="cuda"),
        "mlp1_weight": _weight(g, dtype, c.num_experts, 2 * c.intermediate_size, c.hidden_size, std=c.hidden_size**-0.5),
        "mlp1_bias": _weight(g, dtype, c.num_experts, 2 * c.intermediate_size, std=0.1),
        "mlp2_weight": _weight(g, dtype, c.num_experts, c.hidden_size, c.intermediate_size, std=c.intermediate_size**-0.5),
        "mlp2_bias": _weight(g, dtype, c.num_experts, c.hidden_size, std=0.1),
    }


class Experts(nn.Module):
    """One GPT-OSS-20B mixture-of-experts layer behind its router (the chosen expert ids and their weights are
    inputs, so that no tie between two experts makes two correct results differ): norm, up product, clamped
    SwiGLU, down product, weighted sum, residual."""

    def __init__(self, weights):
        super().__init__()
        for name, value in weights.items():
            setattr(self, name, nn.Parameter(value.cpu(), requires_grad=False))

    def forward(self, x, experts, expert_weights):
        h = x.float()
        t = (h * torch.rsqrt(torch.mean(h**2, dim=-1, keepdim=True) + 1e-5) * self.norm).to(x.dtype)
        t = torch.einsum("beck,bk->bec", self.mlp1_weight[experts, ...], t) + self.mlp1_bias[experts, ...]
        glu, linear = t[..., ::2], t[..., 1::2]
        glu = glu.clamp(min=None, max=gpt_oss_20b.swiglu_limit)
        linear = linear.clamp(min=-gpt_oss_20b.swiglu_limit, max=gpt_oss_20b.swiglu_limit)
        t = glu * torch.sigmoid(1.702 * glu) * (linear + 1)
        t = torch.einsum("beck,bek->bec", self.mlp2_weight[experts, ...], t)
        t = t + self.mlp2_bias[experts, ...]
        return x + torch.einsum("bec,be->bc", t, expert_weights)


def _dev_weights():
    """The dev model's parameters by name: norm scales 1, biases and sinks 0, everything else N(0, 0.02)."""
    with torch.device("meta"):
        model = Transformer(dev)
    g = _generator(WEIGHTS_SEED)
    weights = {}
    for name, parameter in model.named_parameters():
        if name.endswith(".scale"):
            weights[name] = torch.ones(parameter.shape, device="cuda")
        elif name.endswith(("bias", ".sinks")):
            weights[name] = torch.zeros(parameter.shape, device="cuda")
        else:
            weights[name] = _weight(g, torch.float32, *parameter.shape, std=0.02)
    return weights


def _dev_model():
    model = Transformer(dev).float()
    model.load_state_dict({name: value.cpu() for name, value in _dev_weights().items()})
    return model.eval().requires_grad_(False)


# ---------------------------------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """The inputs of one call, on the GPU (token ids of the host calls: host arrays)."""
    g, kind = _generator(seed), case["kind"]
    if kind == "mlp":
        return (torch.randn(case["rows"], case["hidden"], generator=g, device="cuda").to(DTYPES[case["dtype"]]).cpu(),)
    if kind == "chain":
        shape, dtype = (case["rows"], case["columns"]), DTYPES[case["dtype"]]
        return tuple((torch.rand(shape, generator=g, device="cuda") * 8 - 4).to(dtype) for _ in range(2))
    if kind == "attention":
        c, bf16 = gpt_oss_20b, torch.bfloat16
        tokens, context, past = case["tokens"], case["context"], case["past"]
        x = torch.randn(tokens, c.hidden_size, generator=g, device="cuda").to(bf16)
        positions = past + torch.arange(tokens, device="cuda", dtype=torch.float32)
        cache = [torch.randn(context, c.num_key_value_heads, c.head_dim, generator=g, device="cuda").to(bf16) for _ in range(2)]
        for part in cache:
            part[past:] = 0  # rows of the cache that hold no key yet
        return (x, positions, *cache, torch.where(_live(case, "cuda"), 0.0, -math.inf).to(bf16))
    if kind == "experts":
        c, tokens = gpt_oss_20b, case["tokens"]
        x = torch.randn(tokens, c.hidden_size, generator=g, device="cuda").to(torch.bfloat16)
        # experts are not equally popular: a bias per expert beside the token's own logits
        logits = torch.randn(tokens, c.num_experts, generator=g, device="cuda") + 0.5 * torch.randn(c.num_experts, generator=g, device="cuda")
        chosen = torch.topk(logits, c.experts_per_token, dim=-1)
        return x, chosen.indices, torch.softmax(chosen.values, -1).to(torch.bfloat16)
    count = {"forward": case.get("tokens"), "prefill": case.get("tokens"), "decode": case.get("context", 0) + 1}[kind]
    return (np.random.default_rng(seed).integers(0, dev.vocab_size, count, dtype=np.int64),)


def _live(case, device):
    """Which of the context + tokens keys each query of an attention call sees."""
    tokens, context, past = case["tokens"], case["context"], case["past"]
    window = case["window"] or context
    key = torch.cat((torch.arange(context, device=device), past + torch.arange(tokens, device=device)))
    valid = torch.cat((torch.arange(context, device=device) < past, torch.ones(tokens, dtype=torch.bool, device=device)))
    query = (past + torch.arange(tokens, device=device))[:, None]
    return valid & (key <= query) & (key > query - window)


# ------------------------------------------------------------------------------------- compiled artifacts, calls
class _Artifacts:
    """The compiled artifacts of the last case that was prepared, in a folder of this process."""

    def __init__(self):
        self.key, self.folder = None, None

    def get(self, case, modules):
        key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
        if key != self.key:
            self.drop()
            self.folder = Path(tempfile.mkdtemp(prefix=f"chroma-perf-{os.getpid()}-"))
            for name, exported in modules().items():
                chroma_amd.compile(exported, self.folder / name).close()
            self.key = key
        return self.folder

    def drop(self):
        for folder in Path(tempfile.gettempdir()).glob("chroma-perf-*"):
            owner = folder.name.split("-")[2]
            if folder == self.folder or (owner.isdigit() and not Path(f"/proc/{owner}").exists()):
                shutil.rmtree(folder, ignore_errors=True)
        self.key = self.folder = None


_artifacts = _Artifacts()


def _modules(case):
    """The graphs of a case, exported on examples of its shapes."""
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("decode", "prefill"):
            model, context = _dev_model(), case["context"]
            return {"prefill": export_cached(model, context, context), "decode": export_cached(model, context, 1)}
        if kind == "forward":
            return {"program": torch.export.export(_dev_model(), (torch.zeros(case["tokens"], dtype=torch.int64),))}
        module = {"mlp": lambda: MLP(_mlp_weights(case)), "chain": Chain, "attention": lambda: Attention(_attention_weights()),
                  "experts": lambda: Experts(_expert_weights())}[kind]().eval()
        return {"program": torch.export.export(module, tuple(value.cpu() for value in _inputs(case, 0)))}


class _DeviceArray:
    """A staging region of a loaded program as an array on the GPU (it keeps the program alive)."""

    def __init__(self, program, address, spec):
        self.program = program
        kind = {"float32": "<f4", "bfloat16": "<i2", "int64": "<i8"}[spec["dtype"]]
        self.__cuda_array_interface__ = {"shape": tuple(spec["shape"]), "typestr": kind, "data": (address, False), "version": 2}


def _staging(program, address, spec):
    array = torch.as_tensor(_DeviceArray(program, address, spec), device="cuda")
    return array.view(torch.bfloat16) if spec["dtype"] == "bfloat16" else array


def prepare(case, seed):
    folder = _artifacts.get(case, lambda: _modules(case))
    inputs = _inputs(case, seed)
    if case["kind"] in ("decode", "prefill"):
        decoder = chroma_amd.Decoder(chroma_amd.Program(folder / "prefill"), chroma_amd.Program(folder / "decode"))
        tokens = inputs[0]
        if case["kind"] == "decode":
            decoder.append(tokens[:-1])  # the cache is full; every further step is a decode step
            tokens = tokens[-1:]
        return {"kind": case["kind"], "decoder": decoder, "tokens": tokens}
    program = chroma_amd.Program(folder / "program")
    if case["kind"] in ("mlp", "forward"):
        return {"kind": case["kind"], "program": program, "inputs": inputs if case["kind"] == "mlp" else [inputs[0]]}
    native = program.native
    for index, (spec, value) in enumerate(zip(program.inputs, inputs)):
        _staging(program, native.input_pointer(index), spec).copy_(value)
    torch.cuda.synchronize()  # the program runs on a stream of its own
    outputs = [_staging(program, native.output_pointer(index), spec) for index, spec in enumerate(program.outputs)]
    return {"kind": case["kind"], "program": program, "outputs": outputs}


def run(state):
    kind = state["kind"]
    if kind in ("mlp", "forward"):
        return _host_tensor(state["program"](*state["inputs"]))
    if kind == "decode":
        return _host_tensor(state["decoder"].append(state["tokens"]))
    if kind == "prefill":
        state["decoder"].reset()
        return _host_tensor(state["decoder"].append(state["tokens"]))
    state["program"].native.execute()
    return state["outputs"]


def _host_tensor(array):
    if array.dtype.kind == "f" and array.dtype.itemsize == 4:
        return torch.from_numpy(array)
    return torch.from_numpy(array.view(np.int16)).view(torch.bfloat16)


# ---------------------------------------------------------------------------------------- work and tolerances
def work(case):
    """Bytes and operations of one pass: each input and weight that the result depends on read once, each output
    written once; attention over the live query-key pairs."""
    kind = case["kind"]
    if kind == "mlp":
        rows, h, f, size = case["rows"], case["hidden"], case["inner"], DTYPES[case["dtype"]].itemsize
        return {"bytes": size * (3 * h * f + 2 * rows * h), "flops": 6 * rows * h * f}
    if kind == "chain":
        n = case["rows"] * case["columns"]
        return {"bytes": 3 * n * DTYPES[case["dtype"]].itemsize, "flops": 0}
    if kind == "attention":
        c = gpt_oss_20b
        live = _live(case, "cpu")
        tokens, context, pairs = case["tokens"], case["context"], int(live.sum())
        seen = int(live[:, :context].any(0).sum())
        heads, kv = c.num_attention_heads * c.head_dim, c.num_key_value_heads * c.head_dim
        weights = c.hidden_size * (2 * heads + 2 * kv)
        moved = weights + 2 * tokens * c.hidden_size + 2 * seen * kv + 2 * tokens * kv + tokens * (context + tokens)
        return {"bytes": 2 * moved, "flops": 2 * tokens * weights + 4 * pairs * heads}
    if kind == "experts":
        c, tokens = gpt_oss_20b, case["tokens"]
        slots = tokens * c.experts_per_token
        used = c.num_experts * (1 - (1 - 1 / c.num_experts) ** slots)  # experts that a call of this size meets
        used = max(used, min(c.experts_per_token, c.num_experts))
        per_expert = 3 * c.hidden_size * c.intermediate_size
        return {"bytes": 2 * (used * per_expert + 2 * tokens * c.hidden_size), "flops": 2 * slots * per_expert}
    c = dev
    tokens = {"forward": case.get("tokens"), "prefill": case.get("tokens"), "decode": 1}[kind]
    logits_rows = tokens if kind == "forward" else 1
    heads, kv = c.num_attention_heads * c.head_dim, c.num_key_value_heads * c.head_dim
    dense = c.hidden_size * (2 * heads + 2 * kv + c.num_experts)
    per_expert = 3 * c.hidden_size * c.intermediate_size
    slots = tokens * c.experts_per_token
    used = max(c.experts_per_token, c.num_experts * (1 - (1 - 1 / c.num_experts) ** slots))
    context = case["context"] if kind == "decode" else 0
    pairs = context if kind == "decode" else tokens * (tokens + 1) // 2
    layer = dense + used * per_expert + 2 * (context + tokens) * kv
    vocabulary = c.vocab_size * c.hidden_size
    return {
        "bytes": 4 * (c.num_hidden_layers * layer + vocabulary + tokens * c.hidden_size + logits_rows * c.vocab_size),
        "flops": c.num_hidden_layers * (2 * tokens * dense + 2 * slots * per_expert + 4 * pairs * heads) + 2 * logits_rows * vocabulary,
    }


def tolerance(case):
    """About four times the largest distance from ``exact`` that the listed and some drawn cases show: 3.8e-3 in
    bfloat16 (the new keys' rounding; 1.7e-3 to 3.5e-3 on the other outputs), 3.7e-7 in float32, where sums of up
    to 4096 terms in another order may move further than these."""
    if case["kind"] in ("attention", "experts") or case.get("dtype") == "bf16":
        return {"rel": 1.5e-2, "max": 0.2}
    return {"rel": 5e-6, "max": 5e-4}


# --------------------------------------------------------------------------------------------------- exact
def _norm(x, scale):
    return x * torch.rsqrt(torch.mean(x * x, dim=-1, keepdim=True) + 1e-5) * scale.double()


def _rotary(c, positions):
    """YaRN rotary cosines and sines [tokens, head_dim / 2] (https://arxiv.org/abs/2309.00071). The inverse
    frequencies are single-precision constants of the graph, as the model states them; what follows is 64-bit."""
    freq = c.rope_theta ** (torch.arange(0, c.head_dim, 2, dtype=torch.float32) / c.head_dim)
    if c.rope_scaling_factor > 1:
        concentration = 0.1 * math.log(c.rope_scaling_factor) + 1.0
        half = c.head_dim / 2
        low = half * math.log(c.initial_context_length / (c.rope_ntk_beta * 2 * math.pi)) / math.log(c.rope_theta)
        high = half * math.log(c.initial_context_length / (c.rope_ntk_alpha * 2 * math.pi)) / math.log(c.rope_theta)
        keep = 1 - ((torch.arange(half, dtype=torch.float32) - low) / (high - low)).clamp(0, 1)
        inverse = 1.0 / (c.rope_scaling_factor * freq) * (1 - keep) + 1.0 / freq * keep
    else:
        concentration, inverse = 1.0, 1.0 / freq
    angles = (positions.cpu().float()[:, None] * inverse[None, :]).double().to(positions.device)
    return angles.cos() * concentration, angles.sin() * concentration


def _rotate(x, cos, sin):
    first, second = x.chunk(2, dim=-1)
    cos, sin = cos[:, None, :], sin[:, None, :]
    return torch.cat((first * cos - second * sin, second * cos + first * sin), dim=-1)


def _attend(c, w, prefix, x, positions, keys, values, live):
    """(x + attention, new keys, new values) of one layer in 64 bits; ``live`` [tokens, past + tokens]."""
    tokens = x.shape[0]
    qkv = _norm(x, w[prefix + "norm.scale"]) @ w[prefix + "qkv.weight"].double().T + w[prefix + "qkv.bias"].double()
    heads, kv_heads, dim = c.num_attention_heads, c.num_key_value_heads, c.head_dim
    q, k, v = qkv.split((heads * dim, kv_heads * dim, kv_heads * dim), dim=1)
    cos, sin = _rotary(c, positions)
    q, k = _rotate(q.reshape(tokens, heads, dim), cos, sin), _rotate(k.reshape(tokens, kv_heads, dim), cos, sin)
    v = v.reshape(tokens, kv_heads, dim)
    all_k = k if keys is None else torch.cat((keys.double(), k))
    all_v = v if values is None else torch.cat((values.double(), v))
    attended = torch.empty(tokens, heads, dim, dtype=torch.float64, device=x.device)
    for head in range(heads):
        kv = head // (heads // kv_heads)
        scores = (q[:, head] @ all_k[:, kv].T) / math.sqrt(dim)
        scores = torch.where(live, scores, -math.inf)
        sink = w[prefix + "sinks"][head].double().expand(tokens, 1)
        attended[:, head] = torch.softmax(torch.cat((scores, sink), dim=1), dim=1)[:, :-1] @ all_v[:, kv]
    out = attended.reshape(tokens, -1) @ w[prefix + "out.weight"].double().T + w[prefix + "out.bias"].double()
    return x + out, k, v


def _mix(c, x, t, chosen, chosen_weights, up, up_bias, down, down_bias):
    """x + the weighted sum of the chosen experts' outputs for the normed rows t, in 64 bits."""
    out = x.clone()
    for expert in range(c.num_experts):
        token, slot = torch.nonzero(chosen == expert, as_tuple=True)
        if not len(token):
            continue
        h = t[token] @ up[expert].double().T + up_bias[expert].double()
        glu, linear = h[:, ::2].clamp(max=c.swiglu_limit), h[:, 1::2].clamp(-c.swiglu_limit, c.swiglu_limit)
        h = glu * torch.sigmoid(1.702 * glu) * (linear + 1)
        h = h @ down[expert].double().T + down_bias[expert].double()
        out.index_add_(0, token, h * chosen_weights[token, slot].double()[:, None])
    return out


def _dev_exact(tokens, rows, window):
    """The dev model's logits of the last ``rows`` tokens in 64 bits."""
    c, w = dev, _dev_weights()
    ids = torch.from_numpy(tokens).cuda()
    x = w["embedding.weight"][ids].double()
    place = torch.arange(len(tokens), device="cuda")
    live = (place[None, :] <= place[:, None]) & (place[None, :] > place[:, None] - window)
    for layer in range(c.num_hidden_layers):
        x, _, _ = _attend(c, w, f"block.{layer}.attn.", x, place.double(), None, None, live)
        p = f"block.{layer}.mlp."
        t = _norm(x, w[p + "norm.scale"])
        chosen = torch.topk(t @ w[p + "gate.weight"].double().T + w[p + "gate.bias"].double(), c.experts_per_token, dim=-1)
        x = _mix(c, x, t, chosen.indices, torch.softmax(chosen.values, -1), w[p + "mlp1_weight"], w[p + "mlp1_bias"], w[p + "mlp2_weight"],
                 w[p + "mlp2_bias"])
    return _norm(x[-rows:], w["norm.scale"]) @ w["unembedding.weight"].double().T


def exact(case, seed):
    kind, inputs = case["kind"], _inputs(case, seed)
    if kind == "mlp":
        w, x = _mlp_weights(case), inputs[0].cuda().double()
        h = _norm(x, w["norm"])
        gate, up = h @ w["gate"].double().T, h @ w["up"].double().T
        return (gate * torch.sigmoid(gate) * up) @ w["down"].double().T + x
    if kind == "chain":
        x, y = (value.double() for value in inputs)
        z = torch.tanh(x * 0.5 + y) * torch.sigmoid(y) - torch.exp(torch.clamp(x, -8, 8)) * 1e-3
        return [torch.softmax(z, -1)]
    if kind == "attention":
        x, positions, keys, values, _ = inputs
        return list(_attend(gpt_oss_20b, _attention_weights(), "", x.double(), positions, keys, values, _live(case, "cuda")))
    if kind == "experts":
        x, chosen, chosen_weights = inputs
        w = _expert_weights()
        return [_mix(gpt_oss_20b, x.double(), _norm(x.double(), w["norm"]), chosen, chosen_weights, w["mlp1_weight"], w["mlp1_bias"],
                     w["mlp2_weight"], w["mlp2_bias"])]
    tokens = inputs[0]
    if kind == "forward":
        return _dev_exact(tokens, len(tokens), len(tokens))
    return _dev_exact(tokens, 1, case["context"])
