"""Which products `ops.linear` and `ops.gate_up_silu` may hand to the kernels of this package: on the host, with stand-ins for tensors,
kernels and the vendor's product, so nothing is launched."""
from types import SimpleNamespace

import pytest
import torch

from infer_amd import ops


class Library:
    """Stands in for the C library: every product is one launch."""
    def __init__(self):
        self.launched = []

    def infer_skinny_gemm_workspace_bytes(self, m, n, k):
        return 0

    def __getattr__(self, name):
        def call(*args):
            self.launched.append(name)
            return 0
        return call


def stand_in(rows, columns, device="cuda:0"):
    device = torch.device(device)
    return SimpleNamespace(shape=torch.Size((rows, columns)), device=device, dtype=torch.bfloat16, is_cuda=device.type == "cuda",
                           requires_grad=False, dim=lambda: 2, stride=lambda i: (columns, 1)[i], is_contiguous=lambda: True,
                           get_device=lambda: -1 if device.type == "cpu" else device.index, data_ptr=lambda: 4096)


@pytest.fixture
def library(monkeypatch):
    lib = Library()

    def vendor(x, weight, bias=None):
        raise RuntimeError("vendor's product")

    monkeypatch.setattr(ops._lib, "load", lambda: lib)
    monkeypatch.setattr(ops, "_stream_ptr", lambda t: 0)
    monkeypatch.setattr(torch.nn.functional, "linear", vendor)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: stand_in(4, 512))
    return lib


@pytest.mark.parametrize("product", [ops.gate_up_silu, ops.linear])
def test_products_that_the_kernels_take_are_launched(library, product):
    product(stand_in(4, 256), stand_in(512, 256))
    assert len(library.launched) == 1


@pytest.mark.parametrize("product", [ops.gate_up_silu, ops.linear])
@pytest.mark.parametrize("x,weight", [("cuda:0", "cpu"), ("cuda:0", "cuda:1"), ("cuda:1", "cuda:1"), ("cuda:1", "cuda:0"), ("cpu", "cuda:0")])
def test_operands_elsewhere_than_the_launch_are_the_vendors(library, product, x, weight):
    """A pointer of the host or of another GPU never reaches a kernel: the vendor's product runs there, or refuses."""
    with pytest.raises(RuntimeError, match="vendor"):
        product(stand_in(4, 256, x), stand_in(512, 256, weight))
    assert not library.launched
