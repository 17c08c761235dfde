"""Products and attention of few output tiles: the kernels that split K or the keys over waves and workgroups."""

from __future__ import annotations

import re
import subprocess

import numpy as np
import pytest
import torch

import chroma_amd
from chroma_amd._src.build import compiler_command
from chroma_amd._src.codegen import hip
from chroma_amd._src.codegen.hip import HIPCodegen
from chroma_amd._src.compiler import lower_program
from tests.helpers import Function, as_float, export
from tests.test_hip_runtime import SinkAttention


def assert_sums(got, exact, terms, scale, dtype):
    """``got`` against 64-bit sums of ``terms`` products of standard deviation ``scale``: a float sum's partial sums
    grow like a random walk, so its rounding errors add up to about 2^-24 scale terms / sqrt(2) (8 of them are
    allowed), and the stored value is rounded once (half a spacing: 2^-9 relative in bfloat16, 2^-24 in float)."""
    error = np.abs(as_float(got).astype(np.float64) - exact.numpy())
    limit = 8 * 2.0**-24 * scale * terms + np.abs(exact.numpy()) * (2.0**-8 if dtype == torch.bfloat16 else 2.0**-23)
    worst = np.unravel_index(np.argmax(error - limit), error.shape)
    assert (error <= limit).all(), (worst, error[worst], limit[worst])


def plan_of(module, *inputs):
    return lower_program(export(module, *inputs), HIPCodegen()).files["model.hip"]


def linear(rows, inner, columns, dtype, bias=True):
    generator = torch.Generator().manual_seed(rows + inner + columns)
    layer = torch.nn.Linear(inner, columns, bias=bias).eval()
    with torch.no_grad():
        for parameter in layer.parameters():
            parameter.copy_(torch.randn(parameter.shape, generator=generator) * 0.05)
    return layer.to(dtype), torch.randn(rows, inner, generator=generator).to(dtype)


def test_unaligned_operands_keep_the_general_body():
    """The K-split body copies 16-byte chunks: rows that are no whole chunks, or an operand that starts between two,
    stay on the bodies that took them before."""
    x = torch.ones(40 * 256 + 8)
    assert "kwave_linear<float" in plan_of(Function(lambda v, w: torch.nn.functional.linear(v[4:4 + 40 * 256].reshape(40, 256), w)), x, torch.ones(33, 256))
    assert "kwave_linear" not in plan_of(Function(lambda v, w: torch.nn.functional.linear(v[2:2 + 40 * 256].reshape(40, 256), w)), x, torch.ones(33, 256))
    assert "kwave_linear" not in plan_of(Function(torch.nn.functional.linear), torch.ones(40, 258), torch.ones(33, 258))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("stored", [False, True])
def test_rows_beyond_32_bit_offsets_keep_the_general_body(dtype, stored):
    """The K-split body's byte offsets inside a tile have 32 bits; that holds for an X that is still an expression too."""
    from types import SimpleNamespace

    x = SimpleNamespace(dtype=dtype, stored=stored, view=SimpleNamespace(offset=0) if stored else None)
    weight = SimpleNamespace(dtype=dtype, view=SimpleNamespace(offset=0))
    longest = 2**31 // 128 // (4 if dtype == torch.float32 else 2)
    takes = lambda inner: HIPCodegen()._kwave_few_rows(x, weight, 8, 65536, inner)
    assert takes(longest - 1024) and not takes(longest) and not takes(4 * longest)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, inner, columns", [
    (17, 128, 7),       # every wave one bfloat16 unit of K; one partial column tile, odd stores
    (18, 136, 160),     # K ends inside a unit
    (3, 11528, 37),     # few rows too wide for the streaming kernel, ragged last unit
    (16, 4096, 129),
    (100, 1000, 515),   # ragged rows, columns and K; more units than ring slots
    (250, 4096, 128),
    (300, 264, 1024),
    (700, 640, 2880),   # the largest tiles
])
def test_k_split_linear(tmp_path, dtype, rows, inner, columns):
    layer, x = linear(rows, inner, columns, dtype)
    exported = torch.export.export(layer, (x,))
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert "kwave_linear" in (tmp_path / "hip" / "model.hip").read_text()
        got = [model(x) for _ in range(2)]
    exact = x.double() @ layer.weight.detach().double().T + layer.bias.detach().double()
    for result in got:
        assert_sums(result, exact, inner, 0.05, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("rows, inner, columns, levels", [
    (8, 1024, 4096, (8, 2, 8, 2, 4)),     # products, halves of a unit, units, levels of a wave's share of K, waves
    (3, 11520, 2880, (8, 2, 8, 22.5, 4)),
    (40, 4096, 1024, (64, 16, 4)),        # more than 16 rows: levels of 4 units in one chain
])
def test_k_split_float_sums(tmp_path, rows, inner, columns, levels):
    """The rounding errors of float sums in levels. A level of n terms of like size rounds n partial sums whose mean square is
    (n + 1) / 2 / n of its result's, each by 0.42 x 2^-24 (a uniform error of at most half a spacing, over the spacings of
    its values), and the squares of the levels add up; a fifth more is allowed (the variance of a sample, sums of
    unlike size). The weight stream's sums of few rows are as exact: chains of K / 64 products and a tree."""
    layer, x = linear(rows, inner, columns, torch.float32, bias=False)
    exported = torch.export.export(layer, (x,))
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert "kwave_linear" in (tmp_path / "hip" / "model.hip").read_text()
        got = model(x)
    exact = (x.double() @ layer.weight.detach().double().T).numpy()
    error = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    limit = 1.2 * 0.42 * 2.0**-24 * sum((n + 1) / 2 for n in levels) ** 0.5
    print(f"{rows} x {columns} x {inner}: {error:.3e}, limit {limit:.3e}", flush=True)
    assert error < limit, (error, limit)


@pytest.mark.parametrize("dtype, rows, columns, inner, split", [
    (torch.float32, 800, 4096, 1024, True), (torch.float32, 700, 11520, 2880, True), (torch.float32, 1000, 11520, 2880, True), (torch.float32, 2048, 1024, 4096, True),
    (torch.float32, 2048, 4096, 1024, False), (torch.float32, 4096, 4096, 4096, False), (torch.float32, 8192, 512, 512, False),
    (torch.float32, 20000, 256, 128, False), (torch.float32, 1024, 8192, 2048, False), (torch.float32, 2048, 5120, 128, False),
    (torch.bfloat16, 300, 4096, 1024, True), (torch.bfloat16, 2048, 1024, 4096, True), (torch.bfloat16, 1024, 2048, 2048, True),
    (torch.bfloat16, 4096, 1024, 1024, False), (torch.bfloat16, 1500, 2880, 2880, False), (torch.bfloat16, 20000, 256, 128, False),
])
def test_many_rounds_take_the_tiled_bodies(dtype, rows, columns, inner, split):
    """Products of many tiles, each measured faster on the side it takes."""
    assert (HIPCodegen._kwave_beats_tiles(rows, columns, inner, dtype) is not None) == split


@pytest.mark.parametrize("rows, inner, columns, split", [
    (2, 640, 201088, False), (6, 640, 201088, False), (12, 640, 201088, True), (4, 1024, 32000, True), (8, 1024, 4096, True),
    (3, 2880, 11520, True), (3, 11520, 2880, True), (4, 2048, 8192, True),
])
def test_few_float_rows_over_large_weights_stream(rows, inner, columns, split):
    """Each measured faster on the side it takes (the last three behind an MLP's norm)."""
    from types import SimpleNamespace

    view = SimpleNamespace(offset=0)
    x, weight = SimpleNamespace(dtype=torch.float32, stored=True, view=view), SimpleNamespace(dtype=torch.float32, view=view)
    assert HIPCodegen()._kwave_few_rows(x, weight, rows, columns, inner) == split


@pytest.mark.gpu
@pytest.mark.parametrize("rows, inner, columns", [(17, 64, 5), (129, 68, 130), (140, 520, 260), (130, 1540, 128), (64, 4096, 257)])
def test_tiled_float_product_sums_in_levels(tmp_path, monkeypatch, rows, inner, columns):
    """The 128 x 128 float body: one level, whole levels, ragged ones; its error against what sums of 64 products (32), 4 of
    these and the rest give (``test_k_split_float_sums``)."""
    monkeypatch.setattr(HIPCodegen, "_kwave_beats_tiles", lambda *a: None)
    layer, x = linear(rows, inner, columns, torch.float32)
    exported = torch.export.export(layer, (x,))
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert "mfma_linear<float, 5>" in (tmp_path / "hip" / "model.hip").read_text()
        got = model(x)
    exact = x.double() @ layer.weight.detach().double().T + layer.bias.detach().double()
    assert_sums(got, exact, inner, 0.05, torch.float32)
    error = np.linalg.norm(got - exact.numpy()) / np.linalg.norm(exact)
    low = 32 if inner < 256 else 64
    levels = (low, min(4, -(-inner // low)), -(-inner // (4 * low)), 2)  # (the bias is one more)
    limit = 1.2 * 0.42 * 2.0**-24 * sum((n + 1) / 2 for n in levels) ** 0.5
    print(f"{rows} x {columns} x {inner}: {error:.3e}, limit {limit:.3e}", flush=True)
    assert error < limit, (error, limit)


def attention_inputs(tokens, past, kv_heads, group, dim, window):
    """Operands of a cached attention with sinks: causal (or windowed) over a cache of ``past`` rows, one query row
    wholly masked, an additive bias on a band of keys."""
    generator = torch.Generator().manual_seed(tokens * 31 + past + dim)

    def rand(*shape, scale=1.0):
        return (torch.randn(*shape, generator=generator) * scale).to(torch.bfloat16)

    keys = past + tokens
    mask = torch.zeros(tokens, keys)
    mask[:, keys // 3 : keys // 3 + 30] = torch.randn(tokens, 30, generator=generator)[:, : keys - keys // 3] * 0.5
    for t in range(tokens):
        mask[t, past + t + 1 :] = -torch.inf
        if window is not None:
            mask[t, : max(0, past + t - window)] = -torch.inf
    if tokens > 2:
        mask[1, :] = -torch.inf
    return (rand(tokens, kv_heads, group, dim), rand(past, kv_heads, dim), rand(tokens, kv_heads, dim), rand(past, kv_heads, dim),
            rand(tokens, kv_heads, dim), mask.to(torch.bfloat16), rand(kv_heads * group, scale=2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens, past, kv_heads, group, dim, window", [
    (1, 99, 8, 8, 64, None),     # one query, keys a multiple of 4 in a partial block
    (3, 131, 2, 4, 32, 40),      # 12 of 16 rows; heads of 32
    (2, 701, 8, 8, 64, 128),     # odd key count, whole key blocks masked, no split
    (16, 1000, 1, 3, 128, None), # an odd group: rows of one query in two tiles; one KV head, keys split
    (36, 4036, 8, 8, 64, 128),   # many dead blocks per wave
    (63, 17, 2, 8, 64, None),
    (100, 1000, 8, 8, 64, 128),
    (70, 5000, 1, 8, 64, None),  # several blocks per wave and split
])
def test_few_query_attention(tmp_path, tokens, past, kv_heads, group, dim, window):
    """Attention of few query rows with the keys split over waves and workgroups, against the oracle's unfused chain at
    its bfloat16 bar, twice."""
    from oracle import compile_cpu
    from tests.helpers import assert_close, numpy_of

    inputs = attention_inputs(tokens, past, kv_heads, group, dim, window)
    exported = torch.export.export(SinkAttention(), inputs)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert "attention_flash<" in (tmp_path / "hip" / "model.hip").read_text()
        got = [model(*inputs) for _ in range(2)]
    want = compile_cpu(exported, tmp_path / "cpu")(*[numpy_of(v) for v in inputs])
    for result in got:
        assert_close(result, want, rtol=2e-2, atol=1e-2)


@pytest.mark.parametrize("tokens, keys, kv_heads, group, dim, fused", [
    (1, 60, 1, 8, 32, True), (16, 256, 1, 8, 32, True), (4, 128, 1, 2, 64, True),
    (17, 60, 1, 8, 32, False), (1, 257, 1, 8, 32, False), (4, 129, 1, 2, 64, False), (1, 60, 1, 8, 64, False), (1, 60, 2, 4, 32, False),
    (1, 60, 1, 2, 128, False),
])
def test_short_rows_of_one_kv_head_keep_their_product(tokens, keys, kv_heads, group, dim, fused):
    """A bfloat16 attention of one KV head over few keys and the few-row product behind it are one launch, q and k rotated in place."""
    class Block(torch.nn.Module):
        def forward(self, w, angle, q, k_past, k_new, *rest):
            turn = lambda v: torch.cat((v[..., : dim // 2] * angle, v[..., dim // 2 :] * (1 - angle)), -1)
            y = SinkAttention()(turn(q), k_past, turn(k_new), *rest)
            return torch.nn.functional.linear(y.reshape(tokens, -1), w)

    inputs = attention_inputs(tokens, keys - tokens, kv_heads, group, dim, None)
    width = kv_heads * group * dim
    files = lower_program(export(Block(), torch.ones(128, width, dtype=torch.bfloat16), torch.ones(1, dtype=torch.bfloat16), *inputs), HIPCodegen()).files
    launches = [line.split()[1] for line in files["model.plan"].splitlines() if line.startswith("launch ")]
    assert (len(launches) == 1 and "attention_linear" in launches[0]) == fused and fused != ("attention_flash<" in files["model.hip"]), launches


@pytest.mark.gpu
@pytest.mark.parametrize("tokens, keys, group, dim", [(1, 64, 8, 32), (5, 201, 8, 32), (16, 256, 4, 32), (3, 128, 4, 64)])
def test_short_rows_with_their_product(tmp_path, tokens, keys, group, dim):
    """That launch against the oracle's unfused chain at its bfloat16 bar."""
    from oracle import compile_cpu
    from tests.helpers import assert_close, numpy_of

    class Block(torch.nn.Module):
        def forward(self, w, *operands):
            return torch.nn.functional.linear(SinkAttention()(*operands).reshape(tokens, -1), w)

    inputs = (torch.randn(96, group * dim, generator=torch.Generator().manual_seed(keys)).to(torch.bfloat16) * 0.1,
              *attention_inputs(tokens, keys - tokens, 1, group, dim, None))
    exported = torch.export.export(Block(), inputs)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert "stream_block_linear" in (tmp_path / "hip" / "model.hip").read_text()
        got = model(*inputs)
    assert_close(got, compile_cpu(exported, tmp_path / "cpu")(*[numpy_of(v) for v in inputs]), rtol=2e-2, atol=1e-2)


class GroupedExperts(torch.nn.Module):
    def forward(self, weights, indices, x, per_slot):
        selected = weights[indices]
        return torch.einsum("beck,bk->bec", selected, x), torch.einsum("beck,bek->bec", selected, per_slot)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("experts, channels, inner, counts", [
    (3, 100, 136, [1, 63, 0]),          # one slot, an empty expert, K and channels inside a tile
    (12, 256, 128, [16, 17, 32, 33, 64, 65, 1, 0, 0, 28, 60, 4]),  # every count of live 16-row blocks
    (70, 36, 264, [2] * 64 + [0] * 5 + [64]),  # more experts than lanes
])
def test_k_split_expert_products(tmp_path, dtype, experts, channels, inner, counts):
    generator = torch.Generator().manual_seed(sum(counts) + channels)
    slots = torch.cat([torch.full((count,), e, dtype=torch.int64) for e, count in enumerate(counts)])
    slots = slots[torch.randperm(len(slots), generator=generator)]
    selected = 4 if len(slots) % 4 == 0 else 1
    indices = slots.reshape(-1, selected)
    indices[0, 0] -= experts  # ids wrap when negative
    weights = (torch.randn(experts, channels, inner, generator=generator) * 0.05).to(dtype)
    x = torch.randn(len(indices), inner, generator=generator).to(dtype)
    per_slot = torch.randn(*indices.shape, inner, generator=generator).to(dtype)
    exported = export(GroupedExperts(), weights, indices, x, per_slot)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert (tmp_path / "hip" / "model.hip").read_text().count("grouped_expert_kwave") == 2
        up, down = model(weights, indices, x, per_slot)
        bad = indices.clone()
        bad[-1, -1] = experts
        with pytest.raises(IndexError):
            model(weights, bad, x, per_slot)
    w = weights.double()[indices]
    assert_sums(up, torch.einsum("beck,bk->bec", w, x.double()), inner, 0.05, dtype)
    assert_sums(down, torch.einsum("beck,bek->bec", w, per_slot.double()), inner, 0.05, dtype)


def test_k_split_expert_products_have_a_name_of_their_own():
    """Profiles tell the K-split grouped products from the tiled ones by their kernels' names."""
    weights, indices, x, per_slot = few_slots(4, 128, 128, 80)
    names = lambda *inputs: sorted({name.rsplit("_", 1)[0] for name in re.findall(r"\bchroma_experts_\w+", plan_of(GroupedExperts(), *inputs))})
    assert names(weights.float(), indices, x.float(), per_slot.float()) == ["chroma_experts_kwave"]
    weights, indices, x, per_slot = few_slots(4, 384, 128, 80)
    assert names(weights, indices, x, per_slot) == ["chroma_experts_mfma"]


@pytest.mark.parametrize("dtype, experts, channels, inner, slots, split", [
    (torch.float32, 8, 2048, 1024, 2048, True), (torch.float32, 32, 1024, 512, 4096, True), (torch.float32, 12, 256, 128, 16384, True),
    (torch.float32, 32, 1024, 512, 16384, True), (torch.float32, 8, 2048, 1024, 16384, False),
    (torch.bfloat16, 32, 1000, 512, 512, True), (torch.bfloat16, 8, 2048, 1024, 512, True),
    (torch.bfloat16, 32, 1000, 512, 1024, False), (torch.bfloat16, 32, 1000, 512, 2000, False),
])
def test_many_expert_slots_take_the_tiled_bodies(dtype, experts, channels, inner, slots, split):
    """Each measured faster on the side it takes."""
    from types import SimpleNamespace

    operand = SimpleNamespace(dtype=dtype, view=SimpleNamespace(offset=0))
    assert (HIPCodegen()._kwave_experts(operand, operand, slots, experts, channels, inner) is not None) == split


@pytest.mark.gpu
@pytest.mark.parametrize("experts, channels, inner, counts", [(3, 100, 136, [1, 63, 0]), (4, 260, 1540, [129, 0, 40, 300])])
def test_tiled_float_expert_products(tmp_path, monkeypatch, experts, channels, inner, counts):
    """Float expert products on 128 x 128 tiles, their sums in levels."""
    monkeypatch.setattr(HIPCodegen, "_kwave_experts", lambda *a: None)
    generator = torch.Generator().manual_seed(inner)
    slots = torch.cat([torch.full((count,), e, dtype=torch.int64) for e, count in enumerate(counts)])
    indices = slots[torch.randperm(len(slots), generator=generator)].reshape(-1, 1)
    weights = torch.randn(experts, channels, inner, generator=generator) * 0.05
    x, per_slot = torch.randn(len(indices), inner, generator=generator), torch.randn(*indices.shape, inner, generator=generator)
    with chroma_amd.compile(export(GroupedExperts(), weights, indices, x, per_slot), tmp_path / "hip") as model:
        source = (tmp_path / "hip" / "model.hip").read_text()
        assert "grouped_expert_linear<float, false, 5" in source and "grouped_expert_linear<float, true, 5" in source
        up, down = model(weights, indices, x, per_slot)
    w, low = weights.double()[indices], 32 if inner < 256 else 64
    limit = 1.2 * 0.42 * 2.0**-24 * sum((n + 1) / 2 for n in (low, min(4, -(-inner // low)), -(-inner // (4 * low)))) ** 0.5
    for got, exact in ((up, torch.einsum("beck,bk->bec", w, x.double())), (down, torch.einsum("beck,bek->bec", w, per_slot.double()))):
        assert_sums(got, exact, inner, 0.05, torch.float32)
        error = np.linalg.norm(got - exact.numpy()) / np.linalg.norm(exact)
        assert error < limit, (error, limit)


def few_slots(experts, channels, inner, slots):
    generator = torch.Generator().manual_seed(slots + channels)
    weights = (torch.randn(experts, channels, inner, generator=generator) * 0.05).bfloat16()
    indices = torch.randint(0, experts, (slots, 1), generator=generator)
    return weights, indices, torch.randn(slots, inner, generator=generator).bfloat16(), torch.randn(slots, 1, inner, generator=generator).bfloat16()


def test_few_slots_are_grouped_where_slabs_repeat(monkeypatch):
    """From one slot per expert on, and only where the repeated slabs cost more than the routing; an operand that starts
    inside a 16-byte chunk stays on the stream."""
    of = lambda slots, *view: plan_of(GroupedExperts(), *few_slots(6, 384, 64, slots))
    assert "grouped_expert" not in of(12)
    monkeypatch.setattr(hip, "REPEATED_SLAB_BYTES", 1)
    assert of(5).count("chroma::stream_expert_linear") == 2 and of(6).count("chroma::grouped_expert_linear<") == 2
    shifted = lambda w, i, x: torch.einsum("beck,bk->bec", w[4:4 + 6 * 384 * 64].reshape(6, 384, 64)[i], x)
    plan = plan_of(Function(shifted), torch.ones(6 * 384 * 64 + 8, dtype=torch.bfloat16), *few_slots(6, 384, 64, 12)[1:3])
    assert "grouped_expert" not in plan


def test_ring_tiles_of_few_slots():
    """The narrower tile only where it needs fewer rounds of the chip, and never above its range."""
    few, wide = hip.FEW_SLOT_TILE, hip.RING_EXPERT_TILES
    assert [HIPCodegen._ring_tile(slots, 32, 5760) for slots in (32, 200, 2048, 2049)] == [few, wide[0], wide[0], wide[0]]
    assert [HIPCodegen._ring_tile(slots, 32, 2880) for slots in (32, 200, 2048, 2049)] == [wide[1], few, few, wide[1]]
    assert HIPCodegen._ring_tile(64, 32, 192) is None and HIPCodegen._ring_tile(64, 32, 640) == wide[1]


@pytest.mark.gpu
@pytest.mark.parametrize("experts, channels, inner, slots", [
    (5, 384, 64, 5),     # the 192-channel tile in place of the 384-channel one
    (1, 960, 96, 63),    # one expert; the 192-channel tile in place of the 320-channel one
    (9, 320, 160, 23),   # the 320-channel tile
])
def test_few_slots_grouped_by_expert(tmp_path, monkeypatch, experts, channels, inner, slots):
    monkeypatch.setattr(hip, "REPEATED_SLAB_BYTES", 0)
    weights, indices, x, per_slot = few_slots(experts, channels, inner, slots)
    indices[0, 0] -= experts
    exported = export(GroupedExperts(), weights, indices, x, per_slot)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        assert (tmp_path / "hip" / "model.hip").read_text().count("chroma::grouped_expert_linear<") >= 1
        up, down = model(weights, indices, x, per_slot)
        indices[-1, -1] = experts
        with pytest.raises(IndexError):
            model(weights, indices, x, per_slot)
        indices[-1, -1] = 0
    indices = few_slots(experts, channels, inner, slots)[1]
    w = weights.double()[indices]
    assert_sums(up, torch.einsum("beck,bk->bec", w, x.double()), inner, 0.05, torch.bfloat16)
    assert_sums(down, torch.einsum("beck,bek->bec", w, per_slot.double()), inner, 0.05, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("keys, dim", [
    (2, 16), (64, 16), (65, 16), (512, 16),   # one past key, whole and ragged rounds of 64 keys, the longest single batch
    (256, 32), (257, 32), (128, 64), (129, 64),  # value rows requested behind the scores; two batches
    (70, 8), (70, 24),                        # more lanes to a dimension; no power of two
])
def test_one_wave_per_head_attention(tmp_path, dtype, keys, dim):
    """One query on one wave per head, against the oracle: at its bfloat16 bar, or (float) within the errors of sums of up
    to 513 terms and of an exponential of arguments up to about 20 (2^-24 times either, and a few such)."""
    from oracle import compile_cpu
    from tests.helpers import assert_close, numpy_of

    inputs = tuple(v.to(dtype) for v in attention_inputs(1, keys - 1, 2, 4, dim, None))
    exported = torch.export.export(SinkAttention(), inputs)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        got = [model(*inputs) for _ in range(2)]
    want = compile_cpu(exported, tmp_path / "cpu")(*[numpy_of(v) for v in inputs])
    for result in got:
        assert_close(result, want, **({"rtol": 2e-2, "atol": 1e-2} if dtype == torch.bfloat16 else {"rtol": 1e-4, "atol": 1e-5}))


@pytest.mark.gpu
@pytest.mark.parametrize("group, keys, dim", [(9, 320, 16), (16, 512, 16), (16, 100, 64)])
def test_one_wave_per_head_attention_of_many_heads(tmp_path, group, keys, dim):
    """The same in float with more than 8 waves a workgroup, which take their keys in batches."""
    from oracle import compile_cpu
    from tests.helpers import assert_close, numpy_of

    inputs = tuple(v.float() for v in attention_inputs(1, keys - 1, 2, group, dim, None))
    exported = torch.export.export(SinkAttention(), inputs)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        got = model(*inputs)
    assert_close(got, compile_cpu(exported, tmp_path / "cpu")(*[numpy_of(v) for v in inputs]), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("product", [False, True])
@pytest.mark.parametrize("group, keys, dim", [(8, 512, 16), (9, 320, 16), (16, 320, 16), (8, 256, 32), (16, 256, 32), (8, 128, 64), (12, 128, 64), (16, 100, 64)])
def test_one_wave_per_head_attention_fits_its_registers(tmp_path, group, keys, dim, product):
    """A workgroup has a wave per query head: with more than 8 of them a lane's registers don't hold its keys' rows, and the
    kernel takes them in batches: no scratch beyond what q, the sums and the batches of heads of 64 need by themselves."""
    class Block(torch.nn.Module):
        def forward(self, w, *operands):
            y = SinkAttention()(*operands).reshape(1, -1)
            return torch.nn.functional.linear(y, w) if product else y

    inputs = (torch.ones(256, group * dim), *(v.float() for v in attention_inputs(1, keys - 1, 1, group, dim, None)))
    (tmp_path / "model.hip").write_text(plan_of(Block(), *inputs))
    remarks = subprocess.run([*compiler_command(), "-Rpass-analysis=kernel-resource-usage", str(tmp_path / "model.hip"), "-o", str(tmp_path / "out")],
                             capture_output=True, text=True, check=True).stderr
    names = re.findall(r"Function Name: (\S+)", remarks)
    scratch = dict(zip(names, map(int, re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", remarks))))
    kernels = [name for name in names if "attention" in name]
    assert len(kernels) == 1 and product == ("attention_linear" in kernels[0]), names
    assert scratch[kernels[0]] <= {(12, 64): 100, (16, 64): 350}.get((group, dim), 0), scratch


@pytest.mark.gpu
def test_float_activation_epilogue_is_bit_identical(tmp_path, monkeypatch):
    """The float MoE MLP whose clamped SwiGLU is written by its up product's epilogue against the build with a separate
    launch, bit for bit, with the product returned or not."""
    from chroma_amd._src.codegen import hip as codegen
    from tests.helpers import ExpertMLP, leaves

    x = torch.randn(96, 128, generator=torch.Generator().manual_seed(3)) * 2
    for product in (False, True):
        exported = torch.export.export(ExpertMLP(128, 64, seed=1, std=0.08, product=product).float().eval(), (x,))
        runs = []
        for fused in (False, True):
            monkeypatch.setattr(codegen, "ACTIVATION_EPILOGUES", fused)
            with chroma_amd.compile(exported, tmp_path / f"{product}{fused}") as program:
                assert program.stats["expert_epilogues"] == int(fused)
                runs.append([np.asarray(a).copy() for a in leaves(program(x))])
        for plain, fused in zip(*runs):
            np.testing.assert_array_equal(fused, plain)


def test_strides_of_views_match_numpy():
    """``_viewed_strides`` against numpy's own reshaping in place, over random slices and orders of up to 4 dimensions."""
    import itertools
    import random

    rng = random.Random(0)
    in_place = copies = 0
    for _ in range(3000):
        a = np.arange(rng.choice([24, 96, 144])).reshape(rng.choice([(2, 3, 4, -1), (4, -1), (6, 1, -1), (-1,)]))
        order = list(range(a.ndim))
        if rng.random() < 0.3:
            rng.shuffle(order)
        view = a.transpose(order)
        view = view[tuple(slice(rng.randint(0, 1) if s > 1 else 0, s, rng.choice([1, 1, 2])) for s in view.shape)]
        wanted, left = [], view.size
        while left > 1:
            wanted.append(rng.choice([d for d in range(2, left + 1) if left % d == 0]))
            left //= wanted[-1]
            if rng.random() < 0.2:
                wanted.append(1)
        strides = HIPCodegen._viewed_strides(view.shape, [s // a.itemsize for s in view.strides], wanted)
        if strides is None:
            shaped = view.view()
            with pytest.raises(AttributeError):
                shaped.shape = tuple(wanted)
            copies += 1
            continue
        start = (view.__array_interface__["data"][0] - a.__array_interface__["data"][0]) // a.itemsize
        at = [start + sum(i * s for i, s in zip(c, strides)) for c in itertools.product(*map(range, wanted))]
        np.testing.assert_array_equal(a.reshape(-1)[at], view.reshape(-1))
        in_place += 1
    assert in_place > 500 and copies > 500


def test_outputs_take_over_stored_copies():
    """A value stored for a kernel is not evaluated again for the output that returns it, also under another shape; a
    buffer that two outputs return is copied for the second; a strided view is copied once."""
    class Views(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.w = torch.nn.Parameter(torch.ones(64, 64), requires_grad=False)

        def forward(self, x):
            y = torch.nn.functional.linear(x, self.w)
            half = y[:, 32:].contiguous().view(40, 4, 8)
            return torch.nn.functional.linear(y * 2, self.w), y.view(40, 8, 8), y, half

    generated = lower_program(export(Views(), torch.ones(40, 64)), HIPCodegen())
    kinds = [line.split()[1].rsplit("_", 1)[0] for line in generated.files["model.plan"].splitlines() if line.startswith("launch ")]
    # product, y * 2, product; a copy of y for the second output of the same buffer and of the strided half
    assert kinds.count("chroma_linear_kwave") == 2 and len(kinds) == 5, kinds


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [2, 5, 16])
def test_few_row_product_behind_a_norm(tmp_path, dtype, rows):
    """A norm over few rows feeding a K-split product (stored by the norm kernel, in bfloat16 as its cast), a strided half of
    the product viewed as heads, and the norm itself, against eager torch in 64 bits at the stored type's rounding."""
    class Block(torch.nn.Module):
        def __init__(self):
            super().__init__()
            generator = torch.Generator().manual_seed(5)
            self.scale = torch.nn.Parameter(1 + 0.1 * torch.randn(2048, generator=generator), requires_grad=False)
            self.w = torch.nn.Parameter((torch.randn(4096, 2048, generator=generator) * 0.05).to(dtype), requires_grad=False)

        def forward(self, x):
            h = x.float()
            h = (h * torch.rsqrt(torch.mean(h**2, dim=-1, keepdim=True) + 1e-5) * self.scale).to(x.dtype)
            y = torch.nn.functional.linear(h, self.w)
            return y, y[:, 1024:3072].contiguous().view(-1, 32, 64), h

    block = Block()
    x = torch.randn(rows, 2048, generator=torch.Generator().manual_seed(rows)).to(dtype)
    exported = export(block, x)
    with chroma_amd.compile(exported, tmp_path / "hip") as model:
        source = (tmp_path / "hip" / "model.hip").read_text()
        assert ("kwave_linear" in source) == (dtype == torch.bfloat16 or rows > 2)
        got, half, normed = (as_float(a).astype(np.float64) for a in model(x))
    wide = x.double()
    h = wide * torch.rsqrt(torch.mean(wide**2, dim=-1, keepdim=True) + 1e-5) * block.scale.double()
    spacing = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-21  # the norm's own float steps in float
    np.testing.assert_allclose(normed, h.numpy(), rtol=spacing, atol=1e-30)
    assert_sums(got.astype(np.float32), torch.from_numpy(normed) @ block.w.double().T, 2048, 0.05, dtype)
    np.testing.assert_array_equal(half, got[:, 1024:3072].reshape(rows, 32, 64))
