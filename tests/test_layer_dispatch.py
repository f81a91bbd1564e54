"""A decoder layer takes its norms into the products behind them only where nobody could tell: on the host, with stand-ins for the kernels."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from infer_amd import attention as attention_module, ops, qwen3


def _norm(x, weight, eps, residual=None, out=None):
    x = x if residual is None else residual.add_(x)
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight
    return y if residual is None else (y, residual)


class Mixed(torch.nn.Module):
    k_cache = v_cache = torch.zeros(0)

    def forward(self, q, k, v, kv_stored):
        return q.reshape(q.shape[0], -1) * 2 + k.reshape(k.shape[0], -1).repeat(1, 2)


@pytest.fixture
def layer(monkeypatch):
    torch.manual_seed(0)
    config = SimpleNamespace(hidden_size=16, num_attention_heads=2, num_key_value_heads=1, max_position_embeddings=8, rms_norm_eps=1e-6, head_dim=8,
                             intermediate_size=24)
    it = qwen3.QwenDecoderLayer(config, 0).float()
    for p in it.parameters():
        torch.nn.init.normal_(p)
    it.fused = 0

    def fused(x, gain, eps, residual, weight, gated=False):
        it.fused += 1
        total = x if residual is None else x + residual
        y = F.linear(_norm(total, gain, eps), weight)
        return (F.silu(y[:, :24]) * y[:, 24:] if gated else y), total

    monkeypatch.setattr(ops, "norm_linear", fused)
    monkeypatch.setattr(ops, "rms_norm", _norm)
    monkeypatch.setattr(ops, "silu_and_mul", lambda out, y: out.copy_(F.silu(y[..., :24]) * y[..., 24:]))
    monkeypatch.setattr(ops, "gate_up_silu", lambda x, w: F.silu(F.linear(x, w)[:, :24]) * F.linear(x, w)[:, 24:])
    monkeypatch.setattr(ops, "qk_norm_rope_store_kvcache", lambda *a, **k: None)
    monkeypatch.setattr(qwen3, "cos_sin_table", lambda *a: None)
    monkeypatch.setattr(qwen3, "get_context", lambda: SimpleNamespace(slot_mapping=torch.zeros(0), is_prefill=False, block_tables=None))
    it.self_attn.attn = Mixed()
    return it


def _plain(it, x, residual):
    """The layer in plain calls."""
    s = x if residual is None else x + residual
    a = it.self_attn
    qkv = a.qkv_proj(_norm(s, it.input_layernorm.weight, 1e-6))
    o = a.o_proj(qkv[:, :16] * 2 + qkv[:, 16:24].repeat(1, 2))
    s = s + o
    y = it.mlp.gate_up_proj(_norm(s, it.post_attention_layernorm.weight, 1e-6))
    return it.mlp.down_proj(F.silu(y[:, :24]) * y[:, 24:]), s


@pytest.mark.parametrize("rows,fused", [(1, 2), (ops.FEW_ROWS, 2), (ops.FEW_ROWS + 1, 0)])
@pytest.mark.parametrize("first", [False, True])
def test_layers_of_few_rows(layer, rows, fused, first):
    x, residual = torch.randn(rows, 16), None if first else torch.randn(rows, 16)
    want = _plain(layer, x, residual)
    got = layer(None, x, None if first else residual.clone())
    assert layer.fused == fused
    torch.testing.assert_close(got, want, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("where,left", [("input_layernorm", 1), ("self_attn", 1), ("self_attn.qkv_proj", 1), ("post_attention_layernorm", 1), ("mlp", 1),
                                        ("mlp.gate_up_proj", 1), ("mlp.down_proj", 2), ("self_attn.o_proj", 2)])
def test_somebody_who_looks_sees_the_call(layer, where, left):
    seen = []
    layer.get_submodule(where).register_forward_hook(lambda m, args, out: seen.append((args, out)))
    x, residual = torch.randn(2, 16), torch.randn(2, 16)
    want = _plain(layer, x, residual)
    seen.clear()
    torch.testing.assert_close(layer(None, x, residual.clone()), want, atol=1e-4, rtol=1e-4)
    assert layer.fused == left and len(seen) == 1
    assert all(isinstance(a, torch.Tensor) or a is None for a in seen[0][0])


def test_a_forward_of_its_own_is_called(layer):
    inner = layer.input_layernorm.forward
    layer.input_layernorm.forward = lambda x, residual=None: tuple(2 * t for t in inner(x, residual))
    layer(None, torch.randn(2, 16), torch.randn(2, 16))
    assert layer.fused == 1


class Echo(torch.nn.Module):
    def forward(self, *args):
        return args[-1] * 2


@pytest.mark.parametrize("where,fused", [("self_attn", 1), ("mlp", 1)])
def test_a_module_of_its_own_needs_none_of_the_parts(layer, where, fused):
    """A block put in the place of the attention or the MLP is called, whatever it is made of."""
    setattr(layer, where, Echo())
    layer(None, torch.randn(2, 16), torch.randn(2, 16))
    assert layer.fused == fused


def test_calls_that_the_launch_with_the_front_leaves_to_two():
    """One length for the whole batch, which decode attention takes, no lengths, other types: not this launch's, and nothing is raised here."""
    rows, w, cache = torch.zeros(2, 8, 128, dtype=torch.bfloat16), torch.ones(128, dtype=torch.bfloat16), torch.zeros(4, 256, 8, 128, dtype=torch.bfloat16)
    table, lens, at = torch.zeros(2, 2, dtype=torch.int32), torch.ones(2, dtype=torch.int32), torch.zeros(2, dtype=torch.int64)

    def call(lens=lens, table=table, rows=rows, slots=lens):
        return ops.few_decode_with_front(rows, rows, rows, at, w, w, 1e-6, w.expand(9, 128).contiguous(), cache, cache, slots, table, lens, 0.1)
    assert ops._lib.load().infer_few_decode_workspace_bytes(2, 8, 8, 128, 512) > 0
    for change in ({"lens": 64}, {"lens": None}, {"lens": lens.long()}, {"table": None}, {"table": table[0]}, {"table": table.long()}, {"rows": rows.float()},
                   {"rows": rows[:, :, :64]}, {"slots": lens.long()}, {}):
        assert call(**change) is None


@pytest.fixture
def attention(monkeypatch):
    """An attention with its cache, in a decode step; ``given``: what the launch with the front was given as the product behind it, call by call."""
    torch.manual_seed(1)
    it = qwen3.QwenAttention(16, 2, 1, max_position=8, head_dim=8).float()
    for p in it.parameters():
        torch.nn.init.normal_(p)
    it.attn.k_cache = it.attn.v_cache = torch.zeros(1, 4, 1, 8)
    it.given = []
    context = SimpleNamespace(slot_mapping=torch.zeros(2, dtype=torch.int32), is_prefill=False, block_tables=torch.zeros(2, 1), context_lens=torch.ones(2))

    def few(q, *rest):
        it.given.append(rest[-1])
        return q * 2
    monkeypatch.setattr(ops, "few_decode_with_front", few)
    monkeypatch.setattr(ops, "flash_attn_with_kvcache", lambda q, *a, **k: q * 2)
    monkeypatch.setattr(ops, "qk_norm_rope_store_kvcache", lambda *a, **k: None)
    monkeypatch.setattr(qwen3, "cos_sin_table", lambda *a: None)
    for module in (qwen3, attention_module):
        monkeypatch.setattr(module, "get_context", lambda: context)
    return it


def _attend(it):
    x = torch.randn(2, 16, generator=torch.Generator().manual_seed(2))
    torch.testing.assert_close(it(None, x), F.linear(2 * it.qkv_proj(x)[:, :16], it.o_proj.weight, it.o_proj.bias))


def test_attention_of_a_few_rows_takes_the_front_and_the_product(attention):
    _attend(attention)
    assert len(attention.given) == 1 and attention.given[0] is attention.o_proj.weight


def test_sums_of_the_product_are_passed_on(attention, monkeypatch):
    sums = ops.SplitKSum(torch.zeros(2, 2, 16), torch.float32)
    monkeypatch.setattr(ops, "few_decode_with_front", lambda *a: sums)
    attention.o_proj.forward = None
    assert attention(None, torch.randn(2, 16)) is sums


@pytest.mark.parametrize("how", ["hook", "pre-hook", "forward"])
@pytest.mark.parametrize("where", ["q_norm", "k_norm", "attn"])
def test_no_front_where_somebody_looks_at_its_parts(attention, where, how):
    part = getattr(attention, where)
    if how == "hook":
        part.register_forward_hook(lambda *a: None)
    elif how == "pre-hook":
        part.register_forward_pre_hook(lambda *a: None)
    else:
        inner = part.forward
        part.forward = lambda *a, **k: inner(*a, **k)
    _attend(attention)
    assert attention.given == []


def test_no_front_where_decode_is_somebody_elses(attention):
    seen, inner = [], attention.attn._decode
    attention.attn._decode = lambda *a: seen.append(1) or inner(*a)
    _attend(attention)
    assert attention.given == [] and seen == [1]


@pytest.mark.parametrize("how", ["hook", "pre-hook", "forward", "bias", "class"])
def test_no_product_where_the_projection_is_more_than_its_weight(attention, how):
    seen, proj = [], attention.o_proj
    if how == "hook":
        proj.register_forward_hook(lambda *a: seen.append(1))
    elif how == "pre-hook":
        proj.register_forward_pre_hook(lambda *a: seen.append(1))
    elif how == "forward":
        inner = proj.forward
        proj.forward = lambda *a, **k: seen.append(1) or inner(*a, **k)
    elif how == "bias":
        proj.register_parameter("bias", torch.nn.Parameter(torch.randn(16)))
        seen.append(1)
    else:
        class Other(type(proj)):
            def forward(self, *a, **k):
                seen.append(1)
                return super().forward(*a, **k)
        proj.__class__ = Other
    _attend(attention)
    assert attention.given == [None] and seen == [1]
