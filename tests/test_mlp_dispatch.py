"""`MLP.forward` takes its first projection and the gate in one launch, and `Linear.forward` leaves sums in pieces, only where nobody could
tell: on the host, with stand-ins for the kernels."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F
from torch import nn
from torch.nn.modules import module as modules

from infer_amd import layers, ops


@pytest.fixture
def mlp(monkeypatch):
    torch.manual_seed(0)
    m = layers.MLP(16, 24).float()
    for p in m.parameters():
        nn.init.normal_(p)
    m.fused = 0

    def fused(x, weight):
        m.fused += 1
        y = F.linear(x, weight)
        return F.silu(y[:, :24]) * y[:, 24:]

    monkeypatch.setattr(ops, "gate_up_silu", fused)
    monkeypatch.setattr(ops, "silu_and_mul", lambda out, y: out.copy_(F.silu(y[..., :24]) * y[..., 24:]))
    return m


class Adapted(nn.Module):
    """Another module around the projection, as an adapter or a quantised layer is."""
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    @property
    def weight(self):
        return self.inner.weight

    def forward(self, x):
        return 2 * self.inner(x)


class Doubled(layers.MergeLinear):
    def forward(self, input, defer=False):
        return 2 * super().forward(input, defer)


def replaced(m):
    m.gate_up_proj = Adapted(m.gate_up_proj)


def own_class(m):
    m.gate_up_proj.__class__ = Doubled


def own_forward(m):
    inner = m.gate_up_proj.forward
    m.gate_up_proj.forward = lambda x: 2 * inner(x)


def patched_class(m):
    inner = layers.Linear.forward
    m.undo = lambda: setattr(layers.Linear, "forward", inner)
    layers.Linear.forward = lambda self, x, defer=False: (2 if self is m.gate_up_proj else 1) * inner(self, x, defer)


def hook(m):
    m.gate_up_proj.register_forward_hook(lambda module, args, y: 2 * y)


def pre_hook(m):
    m.gate_up_proj.register_forward_pre_hook(lambda module, args: (2 * args[0],))


def global_hook(m):
    m.undo = modules.register_module_forward_hook(lambda module, args, y: 2 * y if module is m.gate_up_proj else None).remove


def global_pre_hook(m):
    m.undo = modules.register_module_forward_pre_hook(lambda module, args: (2 * args[0],) if module is m.gate_up_proj else None).remove


def bias(m):
    # the bias that makes the product twice as large for the rows below
    m.gate_up_proj.bias = nn.Parameter(F.linear(rows()[0], m.gate_up_proj.weight).detach())


def rows():
    return torch.linspace(-1, 1, 16).expand(5, 16)


@pytest.mark.parametrize("change", [replaced, own_class, own_forward, patched_class, hook, pre_hook, global_hook, global_pre_hook, bias])
def test_a_changed_projection_is_called(mlp, change):
    plain = mlp(rows())
    assert mlp.fused == 1
    y = 2 * F.linear(rows(), mlp.gate_up_proj.weight)
    want = F.linear(F.silu(y[:, :24]) * y[:, 24:], mlp.down_proj.weight)
    change(mlp)
    try:
        got = mlp(rows())
    finally:
        getattr(mlp, "undo", lambda: None)()
    assert mlp.fused == 1
    torch.testing.assert_close(got, want)
    assert not torch.allclose(got, plain)


def test_backward_hooks_are_called(mlp):
    seen = []
    mlp.gate_up_proj.register_full_backward_hook(lambda module, inputs, outputs: seen.append(module))
    mlp(rows().clone().requires_grad_()).sum().backward()
    assert seen == [mlp.gate_up_proj] and mlp.fused == 0


@pytest.mark.parametrize("register", [nn.Module.register_forward_hook, nn.Module.register_full_backward_hook,
                                      lambda layer, hook: modules.register_module_forward_hook(hook),
                                      lambda layer, hook: modules.register_module_full_backward_hook(hook)])
def test_hooks_see_a_tensor_and_not_sums_in_pieces(monkeypatch, register):
    monkeypatch.setattr(ops, "linear", lambda x, weight, defer=False: "pieces" if defer else "tensor")
    layer, x = layers.Linear(256, 64), SimpleNamespace(shape=torch.Size((4, 256)), is_cuda=True, dim=lambda: 2)
    assert layer.forward(x, defer=True) == "pieces" and layer.forward(x) == "tensor"
    handle = register(layer, lambda module, args, result: None)
    try:
        assert layer.forward(x, defer=True) == "tensor"
    finally:
        handle.remove()
    assert layer.forward(x, defer=True) == "pieces"
