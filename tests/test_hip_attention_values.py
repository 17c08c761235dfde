"""Attention over masks and operands of every size: finite fills down to the type's lowest value, large scores."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import chroma_amd
from tests.helpers import as_float
from tests.test_hip_runtime import FreshAttention, SinkAttention

F32, BF16 = torch.float32, torch.bfloat16


def exact_attention(q, k, v, mask, sinks):
    """(out, sum of p |v|) of the attention chain in 64 bits after its own roundings: q and k hold integers, so a float
    dot product is exact, and the score, the scaled and the masked score are rounded to the type as the chain states."""
    dtype, (tokens, kv_heads, group, dim) = q.dtype, q.shape
    dot = torch.einsum("qhmd,khd->hmqk", q.double(), k.double()).to(dtype)
    scores = (dot.float() * (1 / math.sqrt(dim))).to(dtype)
    scores = (scores.float() + mask.float()).to(dtype).double()
    sink = sinks.double().reshape(kv_heads, group, 1, 1).expand(-1, -1, tokens, -1)
    p = torch.softmax(torch.cat((scores, sink), -1), -1)[..., :-1]
    return tuple(torch.einsum("hmqk,khd->qhmd", p, x).numpy() for x in (v.double(), v.double().abs()))


def integers(generator, dtype, *shape, most=3):
    return torch.randint(-most, most + 1, shape, generator=generator).to(dtype)


def operands(tokens, past, kv_heads, group, dim, dtype, window):
    """q, k, v, sinks (one of them -inf) and which keys a query sees: causal, the last ``window`` of them, none for query 1."""
    generator = torch.Generator().manual_seed(tokens * 31 + past + dim)
    keys = past + tokens
    q, k = integers(generator, dtype, tokens, kv_heads, group, dim), integers(generator, dtype, keys, kv_heads, dim)
    v = torch.randn(keys, kv_heads, dim, generator=generator).to(dtype)
    sinks = (torch.randn(kv_heads * group, generator=generator) * 2).to(dtype)
    sinks[0] = -math.inf
    key, last = torch.arange(keys), past + torch.arange(tokens)[:, None]
    seen = (key <= last) & (key > last - window)
    if tokens > 2:
        seen[1] = False
    return q, k, v, sinks, seen


def assert_attention(got, q, k, v, mask, sinks):
    """``got`` within the kernels' own roundings of the exact result. bfloat16: half a spacing (2^-8 relative) of every
    probability and of the output, and 2^-18 for the float steps. Float: sums of up to ``keys`` terms, whose errors walk at random
    (a root of the terms times 2^-24), and some 8 roundings of each exponential and of the rescaled sums; 8 times both
    are allowed. NaN where the chain has it: rows whose keys and sink are all -inf."""
    want, magnitude = exact_attention(q, k, v, mask, sinks)
    got = as_float(got).astype(np.float64)
    error = np.where(got == want, 0.0, np.abs(got - want))
    if q.dtype == BF16:
        limit = 1.02 * 2.0**-8 * (magnitude + np.abs(want)) + 2.0**-18 * magnitude
    else:
        limit = 8 * 2.0**-24 * (math.sqrt(len(k)) + 8) * magnitude
    bad = np.argwhere(np.where(np.isnan(want), ~np.isnan(got), ~(error <= limit + 1e-37)))
    assert not len(bad), (len(bad), [(i, float(want[i]), float(error[i]), float(limit[i])) for i in map(tuple, bad[:3].tolist())])


def compiled(tmp_path, dtype, tokens, past, kv_heads, group, dim):
    """(a call of q, k, v, mask, sinks, the artifact's source) of the fused attention with ``past`` cached rows."""
    keys = past + tokens
    q, k = torch.zeros(tokens, kv_heads, group, dim, dtype=dtype), torch.zeros(keys, kv_heads, dim, dtype=dtype)
    mask, sinks = torch.zeros(tokens, keys, dtype=dtype), torch.zeros(kv_heads * group, dtype=dtype)
    if past:
        model = chroma_amd.compile(torch.export.export(SinkAttention(), (q, k[:past], k[past:], k[:past], k[past:], mask, sinks)), tmp_path / "hip")
        call = lambda q, k, v, mask, sinks: model(q, k[:past], k[past:], v[:past], v[past:], mask, sinks)
    else:
        model = chroma_amd.compile(torch.export.export(FreshAttention(), (q, k, k, mask, sinks)), tmp_path / "hip")
        call = model
    return model, call, (tmp_path / "hip" / "model.hip").read_text()


FLASH = [  # tokens, past, KV heads, group, dim, window
    (F32, 20, 100, 2, 3, 32, 70),      # an odd group: rows of one query in two tiles
    (F32, 17, 40, 2, 2, 16, 400),      # one key block
    (F32, 40, 300, 8, 16, 16, 150),    # two row tiles a wave; a key block of some waves, two of others
    (F32, 33, 700, 1, 1, 64, 400),     # a group of one (17 queries a tile); keys split over workgroups
    (F32, 520, 64, 8, 1, 16, 300),     # the same with two row tiles (33 queries)
    (F32, 130, 1103, 1, 8, 64, 700),   # three splits, ragged keys
    (BF16, 5, 150, 2, 3, 32, 70),      # probabilities divided first; a scale that is no power of two
    (BF16, 1, 299, 8, 8, 64, 200),     # one query
    (BF16, 40, 300, 8, 16, 64, 150),   # two row tiles
    (BF16, 33, 700, 1, 1, 64, 400),    # a group of one; split keys
    (BF16, 70, 900, 1, 8, 128, 500),
    (BF16, 36, 4036, 8, 8, 64, 128),   # long keys, most blocks dead; split
    (BF16, 2, 701, 8, 8, 64, 10**6),   # averages over hundreds of keys
]

HEADS = [  # the group-shared prefill kernel: two heads a wave, one; a power-of-two scale, another
    (BF16, 100, 200, 2, 4, 64, 90),
    (BF16, 130, 101, 1, 3, 64, 70),
    (BF16, 70, 140, 2, 2, 128, 100),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kernel, dtype, tokens, past, kv_heads, group, dim, window",
                         [("attention_flash<", *case) for case in FLASH] + [("attention_heads_mfma_bf16<", *case) for case in HEADS])
def test_attention_with_finite_masks(tmp_path, kernel, dtype, tokens, past, kv_heads, group, dim, window):
    """Masked keys filled with -inf and with finite values down to the type's lowest: rows that see no key in whole key
    blocks, and a row that sees none at all."""
    q, k, v, sinks, seen = operands(tokens, past, kv_heads, group, dim, dtype, window)
    model, call, source = compiled(tmp_path, dtype, tokens, past, kv_heads, group, dim)
    with model:
        assert kernel in source
        for fill in (-math.inf, -3e4, -1e10, -1e30, torch.finfo(dtype).min):
            mask = torch.where(seen, 0.0, torch.tensor(fill)).to(dtype)
            assert_attention(call(q, k, v, mask, sinks), q, k, v, mask, sinks)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens, past, kv_heads, group, dim", [(20, 492, 2, 4, 16), (130, 1103, 1, 8, 64)])
def test_float_attention_with_large_scores(tmp_path, tokens, past, kv_heads, group, dim):
    """Scores around 0, 100 and 400 that differ little within a row: the error does not grow with them. Its norm stays below
    8 x 2^-24 of the result's (a sum of 128 terms in a wave walks some 4 of these)."""
    q, k, v, sinks, seen = operands(tokens, past, kv_heads, group, dim, F32, 10**6)
    mask = torch.where(seen, 0.0, -math.inf)
    model, call, source = compiled(tmp_path, F32, tokens, past, kv_heads, group, dim)
    with model:
        assert "attention_flash<" in source
        for base in (0, 100, 400):
            k[..., 0], q[..., 0] = 4 * math.sqrt(dim), base / 4  # adds ``base`` to every score, exactly
            q[..., 1:] = q[..., 1:].clamp(-1, 1)
            sinks[1:] = base
            got = call(q, k, v, mask, sinks)
            want = exact_attention(q, k, v, mask, sinks)[0]
            live = ~np.isnan(want)
            error = np.linalg.norm((got - want)[live]) / np.linalg.norm(want[live])
            print(f"scores around {base}: {error:.2e}", flush=True)
            assert error < 8 * 2.0**-24, (base, error)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens, past, kv_heads, group, dim, simulated", [(20, 492, 2, 4, 16, 1.8e-7), (20, 492, 2, 4, 64, 1.8e-7)])
def test_float_attention_error(tmp_path, tokens, past, kv_heads, group, dim, simulated):
    """The error of normal operands against 64 bits. The chain simulated in float with the kernel's order of sums (scores in chains of 8
    products, 16 keys a level, 4 waves) gives ``simulated``, with single chains 2.9e-7 and 3.7e-7, with a thread a key and 32
    lanes a sum (the vector units' kernel) 2.2e-7 and 3.2e-7; a fifth more is allowed for another sample."""
    generator = torch.Generator().manual_seed(1)
    q, k, v, sinks = (torch.randn(shape, generator=generator) * scale for shape, scale in (
        ((tokens, kv_heads, group, dim), 1.0), ((past + tokens, kv_heads, dim), 1.0), ((past + tokens, kv_heads, dim), 1.0), ((kv_heads * group,), 2.0)))
    mask = torch.where(torch.arange(past + tokens) <= past + torch.arange(tokens)[:, None], 0.0, -math.inf)
    model, call, source = compiled(tmp_path, F32, tokens, past, kv_heads, group, dim)
    with model:
        assert "attention_flash<" in source
        got = call(q, k, v, mask, sinks)
    scores = torch.einsum("qhmd,khd->hmqk", q.double(), k.double()) / math.sqrt(dim) + mask.double()
    sink = sinks.double().reshape(kv_heads, group, 1, 1).expand(-1, -1, tokens, -1)
    want = torch.einsum("hmqk,khd->qhmd", torch.softmax(torch.cat((scores, sink), -1), -1)[..., :-1], v.double()).numpy()
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"head dimension {dim}: {error:.2e}", flush=True)
    assert error < 1.2 * simulated, (error, simulated)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype, tokens, past, kv_heads, group, dim", [
    (F32, 20, 100, 2, 3, 32), (F32, 130, 1103, 1, 8, 64),                        # one split, three
    (BF16, 5, 150, 2, 3, 32), (BF16, 40, 301, 8, 16, 64), (BF16, 33, 700, 1, 1, 64),  # divided first, in the end, split
])
def test_infinite_last_value_row(tmp_path, dtype, tokens, past, kv_heads, group, dim):
    """The last key block is ragged and the last key's values are infinite: every query sees that key, so every result is
    infinite, and nothing of the block behind it turns it into NaN."""
    q, k, v, sinks, seen = operands(tokens, past, kv_heads, group, dim, dtype, 10**6)
    assert len(k) % 64
    v[-1, :, ::2], v[-1, :, 1::2] = math.inf, -math.inf
    mask = torch.zeros(seen.shape, dtype=dtype)
    model, call, source = compiled(tmp_path, dtype, tokens, past, kv_heads, group, dim)
    with model:
        assert "attention_flash<" in source
        got = as_float(call(q, k, v, mask, sinks))
    assert (got[..., ::2] == math.inf).all() and (got[..., 1::2] == -math.inf).all(), np.isnan(got).sum()
