"""Which products `ops.linear` and `ops.gate_up_silu` may hand to the kernels of this package.  On the host with stand-ins for tensors,
kernels and the vendor's product, so nothing is launched; what follows or transforms operators with real tensors on the GPU."""
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

    def infer_skinny_gemm_pays(self, m, n, k, reduced):
        return 1

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
    monkeypatch.setattr(ops, "_plain", lambda t: True)
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


# ------------------------------------------------------------------ on the GPU: 600 rows of weights would go to the streaming kernel
def operands(gpu):
    g = torch.Generator(device=gpu).manual_seed(1)
    return [torch.randn(n, 256, generator=g, device=gpu).to(torch.bfloat16) for n in (4, 600)]


def near(got, want):
    # both are rounded to bfloat16 once: 2^-8 of each other, and of the largest where terms cancel
    assert (got.float() - want.float()).abs().max() <= 2.0 ** -7 * want.float().abs().max()


@pytest.mark.gpu
def test_a_tangent_passes_through(gpu):
    x, w = operands(gpu)
    with torch.autograd.forward_ad.dual_level():
        for a, b, want in ((torch.autograd.forward_ad.make_dual(x, x.flip(0)), w, x.flip(0) @ w.t()),
                           (x, torch.autograd.forward_ad.make_dual(w, w.flip(0)), x @ w.flip(0).t())):
            near(torch.autograd.forward_ad.unpack_dual(ops.linear(a, b)).tangent, want)
    near(torch.func.jvp(lambda x: ops.linear(x, w), (x,), (x.flip(0),))[1], x.flip(0) @ w.t())


@pytest.mark.gpu
def test_a_batch_of_products_by_vmap(gpu):
    x, w = operands(gpu)
    got = torch.vmap(ops.linear, (0, None))(torch.stack([x, -x]), w)
    near(got, torch.stack([x @ w.t(), -(x @ w.t())]))


@pytest.mark.gpu
def test_a_trace_holds_the_product_and_not_its_result(gpu):
    x, w = operands(gpu)
    traced = torch.jit.trace(lambda x, w: ops.linear(x, w), (x, w), check_trace=False)
    near(traced(-x, w), -(x @ w.t()))


@pytest.mark.gpu
def test_modes_and_subclasses_see_the_product(gpu):
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    x, w = operands(gpu)
    seen = []

    class Calls(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Operators(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Named(torch.Tensor):
        pass

    for mode in (Calls(), Operators()):
        seen.clear()
        with mode:
            ops.linear(x, w)
        assert any("linear" in str(f) or "mm" in str(f) for f in seen)
    assert type(ops.linear(x.as_subclass(Named), w)) is Named
    with FakeTensorMode() as fake:
        assert ops.linear(fake.from_tensor(x), fake.from_tensor(w)).shape == (4, 600)


@pytest.mark.gpu
def test_autocast_to_another_type(gpu):
    x, w = operands(gpu)
    with torch.autocast("cuda", torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.linear(x, w).dtype == torch.bfloat16


@pytest.mark.gpu
def test_a_default_device_and_parameters_keep_the_kernel(gpu, monkeypatch):
    x, w = operands(gpu)
    monkeypatch.setattr(torch.nn.functional, "linear", None)
    for weight in (w, torch.nn.Parameter(w, requires_grad=False)):
        with torch.device(gpu):
            near(ops.linear(x, weight), x @ w.t())
