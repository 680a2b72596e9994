"""Which launches a decode step's attention layer takes, decided on the host: the launch that also rotates and stores is for plain
attention of a plain rotation alone."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from turboserve_amd.kernels.ops import Ops
from turboserve_amd.parts.attention import GroupedQueryAttention
from turboserve_amd.parts.base import PartSpec, ResidualStream, Runtime
from turboserve_amd.parts.block import PreNormBlock
from turboserve_amd.parts.mlp import ActivatedMLP, SwiGLU
from turboserve_amd.parts.norm import RMSNorm
from turboserve_amd.parts.registry import POSITION_ENCODINGS, register_position_encoding
from turboserve_amd.parts.rope import RotaryEncoding


class Launches:
    """The operations an attention layer asks for, by name."""

    mfma_attention_supported = staticmethod(Ops.mfma_attention_supported)
    decode_projected_supported = staticmethod(Ops.decode_projected_supported)
    decode_shared_keys = Ops.decode_shared_keys

    def __init__(self):
        self.names = []

    def linear(self, x, weight, bias, **more):
        return torch.zeros(3, x.shape[0], weight.shape[0])

    def rows_buffer(self, rows, width, dtype, device):
        return torch.zeros(rows, width, dtype=dtype)

    def tiled_attention_supported(self, *geometry):
        return False

    def float32_attention_supported(self, *operands):
        return False

    def rope_store(self, proj, k, v, cos, sin, positions, slots, heads, *more):
        self.names.append("store")
        return torch.zeros(proj.shape[1], heads * k.shape[3], dtype=torch.bfloat16), heads * k.shape[3]

    def attention_decode(self, out, q, *more, projected=None, **rest):
        self.names.append("attention" if projected is None else "all in one")

    def paged_attention_generic(self, *more, **rest):
        self.names.append("generic")


class RotaryAndSlopes(RotaryEncoding):
    """A rotation whose scores also fall with the distance."""

    def score_slopes(self, num_heads):
        return torch.full((num_heads,), 0.5)


class RotaryAndTable(RotaryEncoding):
    def score_bias_table(self, num_heads):
        return torch.zeros(num_heads, 4)


class OwnAttention(GroupedQueryAttention):
    """Attends in a way of its own."""

    def attend(self, qkv, q_stride, ctx, cache, **more):
        self.runtime.ops.names.append("own")
        return qkv


@pytest.fixture
def encodings(monkeypatch):
    for name, part in (("rope_slopes", RotaryAndSlopes), ("rope_table", RotaryAndTable)):
        monkeypatch.delitem(POSITION_ENCODINGS, name, raising=False)
        register_position_encoding(name)(part)
    yield
    for name in ("rope_slopes", "rope_table"):
        POSITION_ENCODINGS.pop(name, None)


@pytest.mark.parametrize("kind,encoding,launches", [
    (GroupedQueryAttention, "rope", ["all in one"]),
    (GroupedQueryAttention, "rope_slopes", ["store", "generic"]),
    (GroupedQueryAttention, "rope_table", ["store", "generic"]),
    (OwnAttention, "rope", ["store", "own"]),
])
@pytest.mark.parametrize("offset", [0, 4])
def test_a_decode_step_attends_by_the_layers_rule(encodings, kind, encoding, launches, offset):
    ops = Launches()
    runtime = Runtime(device=torch.device("cpu"), dtype=torch.bfloat16, ops=ops)
    layer = kind("layer", runtime, hidden_size=64, num_heads=4, num_kv_heads=2, head_dim=32, scale=32 ** -0.5, qkv_bias=False, out_bias=False,
                 window=None, position=PartSpec(encoding, {"head_dim": 32, "theta": 1e4, "max_positions": 64}))
    layer.qkv_weight = torch.zeros(8 * 32, 64)
    pages = [torch.zeros(4 * 1024 + 4, dtype=torch.bfloat16)[offset:offset + 4096] for _ in range(2)]
    cache = SimpleNamespace(group=0, writable=True, block_size=16, k=pages[0].view(4, 2, 16, 32), v=pages[1].view(4, 2, 32, 16))
    if offset and launches == ["all in one"]:  # the launch that stores wants pages on 16 bytes
        launches = ["store", "attention"]
    ints = torch.zeros(3, dtype=torch.int32)
    ctx = SimpleNamespace(num_tokens=3, num_seqs=3, num_prefill_seqs=0, num_decode_seqs=3, max_context_len=20, max_decode_context_len=20,
                          block_tables=[torch.zeros(3, 4, dtype=torch.int32)], slot_mapping=[ints], positions=ints, token_seq=ints,
                          query_start_loc=ints, context_lens=ints, max_decode_context_dev=ints[:1], carried={})
    asked, plain_store = [], layer.position.plain_store
    layer.position.plain_store = lambda head_dim: asked.append(head_dim) or plain_store(head_dim)
    layer.heads_out(torch.zeros(3, 64), ctx, cache)
    assert ops.names == launches
    ctx.num_prefill_seqs, ctx.num_decode_seqs = 1, 2  # a step with a prompt never goes to the launch that stores
    assert layer._attend_projected(torch.zeros(3, 3, 256), ctx, cache) is None
    assert layer._plain_store == plain_store(32) and len(asked) <= (2 if launches == ["all in one"] else 1)  # worked out once


class Steps:
    """What a block of a step of one token asks for, and what its products get."""

    normed_max_rows = Ops.normed_max_rows

    def __init__(self):
        self.names = []

    def waiting_norm(self, residual, *more, **rest):
        self.names.append("waits")
        return SimpleNamespace(after=residual, dtype=torch.bfloat16, device=residual.device)

    def add_rmsnorm(self, residual, *more, **rest):
        self.names.append("norm")
        return residual.bfloat16()

    def linear(self, x, weight, bias=None, **more):
        return torch.zeros(1, 1, weight.shape[0])

    def linear_swiglu(self, x, weight, rule, bias):
        return torch.zeros(1, weight.shape[0] // 2)

    def activate(self, x, *more):
        return x[0]


class ReadingAttention(GroupedQueryAttention):
    """An adapter's way: looks at its rows, then runs the layer."""

    def forward(self, x, ctx, cache):
        assert x.shape == (1, 64)
        return super().forward(x, ctx, cache)

    def _attend_projected(self, *more):
        return torch.zeros(1, 128)


class ReadingHeads(GroupedQueryAttention):
    def heads_out(self, x, ctx, cache, *, scale=1.0, out=None):
        assert x.shape == (1, 64)
        return torch.zeros(1, 128)


class PlainAttention(GroupedQueryAttention):
    def _attend_projected(self, qkv, ctx, cache, waits_for=None):
        assert waits_for is self.o_weight
        return torch.zeros(1, 128)


class ReadingSwiGLU(SwiGLU):
    def forward(self, x, ctx):
        assert x.shape == (1, 64)
        return super().forward(x, ctx)


class ReadingMLP(ActivatedMLP):
    def forward(self, x, ctx):
        assert x.shape == (1, 64)
        return super().forward(x, ctx)


class OwnNorm(RMSNorm):
    def forward_residual(self, stream, rows=None):
        self.runtime.ops.names.append("own")
        return stream.residual.bfloat16()


@pytest.mark.parametrize("mixer,feed_forward,norm,asked", [
    (PlainAttention, SwiGLU, RMSNorm, ["waits", "waits"]),
    (PlainAttention, ActivatedMLP, RMSNorm, ["waits", "waits"]),
    (ReadingAttention, ReadingSwiGLU, RMSNorm, ["norm", "norm"]),
    (ReadingHeads, ReadingMLP, RMSNorm, ["norm", "norm"]),
    (PlainAttention, SwiGLU, OwnNorm, ["own", "own"]),
])
@pytest.mark.parametrize("on_the_instance", [False, True])
def test_a_part_of_its_own_ways_gets_rows(mixer, feed_forward, norm, asked, on_the_instance):
    """A norm waits for its product only where the part that reads it is known to read nothing but the product, and the norm is the plain one: a
    subclass's ways, or those set on an instance, get the rows in a step of one token, too."""
    runtime = Runtime(device=torch.device("cpu"), dtype=torch.bfloat16, ops=Steps())
    block = PreNormBlock.__new__(PreNormBlock)
    block.runtime = runtime
    block.mixer = mixer("mixer", runtime, hidden_size=64, num_heads=4, num_kv_heads=2, head_dim=32, scale=32 ** -0.5, qkv_bias=False, out_bias=False,
                        window=None, position=PartSpec("rope", {"head_dim": 32, "theta": 1e4, "max_positions": 64}))
    block.mixer.qkv_weight, block.mixer.o_weight = torch.zeros(8 * 32, 64), torch.zeros(64, 4 * 32)
    more = {"activation": "relu"} if issubclass(feed_forward, ActivatedMLP) else {}
    block.feed_forward = feed_forward("mlp", runtime, hidden_size=64, intermediate_size=32, **more)
    block.feed_forward.gate_up_weight = block.feed_forward.up_weight = torch.zeros(64, 64)
    block.feed_forward.down_weight = torch.zeros(64, 32)
    block.mixer_norm, block.ff_norm = (norm(name, runtime, size=64, eps=1e-6) for name in ("a", "b"))
    if on_the_instance:
        for part in (block.mixer, block.feed_forward):
            def looks(x, *rest, forward=part.forward):
                assert x.shape == (1, 64)
                return forward(x, *rest)
            part.forward = looks
        asked = [name.replace("waits", "norm") for name in asked]
    ctx = SimpleNamespace(num_prefill_seqs=0, num_tokens=1)
    block.forward(ResidualStream(torch.zeros(1, 64), torch.zeros(2, 1, 64)), ctx, None)
    assert runtime.ops.names == asked


@pytest.mark.parametrize("workgroups,span,head_dim,waves", [
    (256, 128, 128, 8), (257, 1024, 128, 4), (1023, 512, 128, 4), (1024, 512, 128, 2), (1024, 1024, 128, 4), (257, 1025, 128, 8),
    (320, 2048, 80, 4), (320, 2049, 80, 8), (512, 64, 64, 4), (2048, 64, 64, 2), (257, 2048, 256, 2), (256, 2048, 256, 8), (2048, 4096, 256, 8),
])
def test_more_workgroups_than_units_over_short_spans_share_units(workgroups, span, head_dim, waves):
    """A workgroup of eight wavefronts has a unit to itself: 64 requests of 100 keys with 32 KV heads took eight turns of starts, 55 us
    where a wavefront per stretch of keys had taken 34."""
    assert Ops._decode_waves(SimpleNamespace(compute_units=256), workgroups, span, head_dim) == waves


def shares(lengths, rows, pairs, head_dim=128, window=None):
    ops = SimpleNamespace(compute_units=256, decode_shared_keys=Ops.decode_shared_keys)
    return Ops.decode_shares(ops, lengths, rows, pairs, head_dim, window)


@pytest.mark.parametrize("lengths,rows,pairs,parts", [
    ([16384] + [600] * 40, 64, 4, 4),                        # a long request ends last, alone
    ([16384] + [600] * 16, 32, 8, 4),
    ([8192] * 65, 128, 4, 4), ([8192] * 33, 64, 8, 4),       # a few workgroups more than a round
    ([8192] * 64, 64, 4, 1), ([8192] * 128, 128, 4, 1), ([8192] * 33, 64, 4, 1),
    ([2048] * 65, 128, 4, 1), ([16384] + [600] * 16, 32, 4, 1), ([16384], 1, 4, 1), ([], 64, 4, 1),
])
def test_long_requests_among_short_ones_are_divided(lengths, rows, pairs, parts):
    """From half the compute units on, a request was one workgroup's whatever the others brought: 151 us a layer for 16,384 keys among 40
    short requests where 131 had been enough."""
    assert shares(lengths, rows, pairs) == parts
    assert shares(lengths, rows, pairs, window=1024) == 1


def test_a_recorded_step_is_for_lengths_that_divide_alike():
    """Uneven lengths are another recorded shape; the layers find their parts in its context."""
    from turboserve_amd.engine.decode_graph import DecodeGraphs

    geometry, windowed = (4, 128, None), (4, 128, 1024)
    ops = SimpleNamespace(compute_units=256, decode_shared_keys=Ops.decode_shared_keys)
    ops.decode_shares = lambda *of: Ops.decode_shares(ops, *of)
    model = SimpleNamespace(runtime=SimpleNamespace(device=torch.device("cpu"), ops=ops, decode_geometries={geometry, windowed}))
    graphs = DecodeGraphs(model, [], page_size=16, num_groups=1, pad_state_slot=0)
    entries = lambda lengths: [SimpleNamespace(start=n - 1, tables=[[0] * -(-n // 16)]) for n in lengths]
    uneven, even = graphs._key(entries([16384] + [600] * 40)), graphs._key(entries([16384] * 41))
    assert uneven[:2] == even[:2] and even[2] == () and dict(uneven[2]) == {geometry: 4}
    assert graphs._key(entries([600] * 41))[2] == ()
    layer = SimpleNamespace(decode_geometry=geometry, runtime=model.runtime)
    step = SimpleNamespace(recorded=True, max_decode_context_len=16384, decode_shares=dict(uneven[2]))
    assert GroupedQueryAttention._decode_shares(layer, step) == 4
    step.decode_shares = {}
    assert GroupedQueryAttention._decode_shares(layer, step) == 1


@pytest.mark.parametrize("pairs,span,head_dim,shares,parts", [
    (4, 512, 128, 1, 1), (4, 513, 128, 1, 5), (4, 256, 256, 1, 1), (4, 300, 256, 1, 5), (1, 500, 256, 1, 5), (132, 300, 256, 1, 1),
    (64, 8192, 128, 4, 4), (128, 8192, 128, 4, 2), (132, 8192, 128, 4, 4), (132, 2048, 128, 4, 1), (512, 8192, 128, 1, 1),
])
def test_spans_that_are_divided(pairs, span, head_dim, shares, parts):
    """Four wavefronts of heads of more than 128 took four turns over 512 keys in one workgroup."""
    ops = object.__new__(Ops)
    ops.compute_units = 256
    assert ops._decode_parts(pairs, span, head_dim, shares) == parts


@pytest.mark.parametrize("pairs,span,parts", [(4, 64, 1), (4, 65, 2), (4, 128, 2), (4, 256, 4), (4, 300, 4), (4, 512, 4), (4, 513, 5), (4, 1024, 8), (32, 512, 4),
                                              (100, 512, 2), (129, 512, 1)])
def test_spans_whose_parts_the_output_product_joins(pairs, span, parts):
    """No more parts than that product takes, and none without a unit of its own."""
    ops = object.__new__(Ops)
    ops.compute_units = 256
    assert ops._joined_parts(pairs, span) == parts


@pytest.mark.parametrize("head_dim,keys,parts", [
    (32, 128, 1), (32, 256, 1), (32, 257, 4), (32, 512, 4), (64, 128, 1), (64, 129, 3), (64, 256, 4), (96, 128, 1), (96, 129, 3), (128, 64, 1), (128, 65, 2),
    (128, 512, 4), (192, 65, 2), (256, 64, 1), (256, 128, 2), (64, 640, 5),
])
def test_a_short_span_stays_whole_where_parts_cost_more_to_join_than_they_save(monkeypatch, head_dim, keys, parts):
    """One request's attention in front of a product that joins parts: a workgroup a KV head over spans that it reads about as soon as that product has put
    the parts together, by the head's size."""
    from turboserve_amd.kernels import ops as module

    launched = []
    monkeypatch.setattr(module, "load_module", lambda name: SimpleNamespace(**{f"ts_attention_decode_d{head_dim}": lambda *of: launched.append(of) or 0}))
    monkeypatch.setattr(module, "_gpu", lambda *tensors: None)
    ops = object.__new__(Ops)
    ops.compute_units, ops.stream, ops._stream_plans = 256, lambda: None, {}
    heads, ints = 1024 // head_dim * 2, torch.zeros(2, dtype=torch.int32)
    heads -= heads % 2
    out = torch.zeros(1, heads * head_dim, dtype=torch.bfloat16)
    pages, table = torch.zeros(2, 2, 16, head_dim, dtype=torch.bfloat16), torch.zeros(1, 64, dtype=torch.int32)
    matrix = torch.zeros(512, heads * head_dim, dtype=torch.bfloat16)
    waiting = ops.attention_decode(out, out, out.shape[1], pages, pages.view(2, 2, head_dim, 16), table, ints, ints[:1], 0, 1, heads, 1.0, None, keys, waits_for=matrix)
    assert launched[0][19] == parts and (waiting is None) == (parts == 1)
    assert parts == 1 or waiting.sums.shape == (heads, parts, head_dim)
