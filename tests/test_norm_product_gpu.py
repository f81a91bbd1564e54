"""A product of few rows with the norm of its input in front: the bits of the two launches, and what is refused."""
import pytest
import torch

from infer_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen) * std).to(BF16).cuda()


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("m,n,k", [
    (1, 4096, 1024), (2, 6144, 1024), (2, 4112, 1024), (1, 6144, 4096), (2, 4096, 2048), (1, 24576, 4096), (2, 16384, 2048), (1, 16400, 1024),
    (2, 5136, 896), (1, 4096, 640), (1, 4096, 128), (2, 8208, 1920), (1, 5120, 3584), (2, 24592, 512),
])
@pytest.mark.parametrize("source", ["rows", "rows and residual", "pieces"])
def test_bits_of_the_two_launches(gpu, m, n, k, gated, source):
    gen = torch.Generator().manual_seed(m + n + k)
    w, gain = _rand(gen, n, k, std=0.05), _rand(gen, k)
    residual = None if source == "rows" else _rand(gen, m, k)
    assert ops._lib.load().infer_norm_product_supported(m, n, k, int(gated))
    if source == "pieces":
        x = ops.SplitKSum(torch.randn(5, m, k, generator=gen).cuda(), BF16)
        plain = x.materialize()
    else:
        x = plain = _rand(gen, m, k)
    kept = residual.clone() if residual is not None else None
    got, total = ops.norm_linear(x, gain, 1e-6, residual, w, gated)
    normed = ops.rms_norm(plain, gain, 1e-6, kept)
    normed, want_total = normed if kept is not None else (normed, plain)
    want = ops.gate_up_silu(normed, w) if gated else ops.linear(normed, w)
    assert torch.equal(total, want_total) and torch.equal(got, want)
    if residual is not None:
        assert total.data_ptr() != residual.data_ptr()


def test_rows_of_other_strides_and_what_is_left_to_two_launches(gpu):
    gen = torch.Generator().manual_seed(3)
    w, gain, wide, res = _rand(gen, 4096, 1024, std=0.05), _rand(gen, 1024), _rand(gen, 2, 2048), _rand(gen, 2, 1536)
    x, residual = wide[:, 1024:], res[:, 256:1280]
    got, total = ops.norm_linear(x, gain, 1e-6, residual, w)
    normed, want = ops.rms_norm(x.contiguous(), gain, 1e-6, residual.contiguous())
    assert torch.equal(total, want) and torch.equal(got, ops.linear(normed, w))
    assert ops.norm_linear(wide[:, 4:1028], gain, 1e-6, residual, w) is None                     # rows off a vector's start
    assert ops.norm_linear(x, gain, 1e-6, res[:, 4:1028], w) is None
    assert ops.norm_linear(x, gain.float(), 1e-6, residual, w) is None
    assert ops.norm_linear(x, gain[:512], 1e-6, residual, w) is None
    assert ops.norm_linear(x, gain, 1e-6, residual[:1], w) is None
    assert ops.norm_linear(_rand(gen, 3, 1024), gain, 1e-6, None, w) is None                     # more rows
    assert ops.norm_linear(_rand(gen, 2, 4096), _rand(gen, 4096), 1e-6, None, _rand(gen, 6144, 4096)) is None
    assert ops.norm_linear(x, gain, 1e-6, residual, _rand(gen, 1024, 1024)) is None              # a split product


def test_stale_pieces_are_refused(gpu):
    gen = torch.Generator().manual_seed(4)
    part = torch.randn(4, 2, 1024, generator=gen).cuda()
    old = ops.SplitKSum(part, BF16)
    ops.SplitKSum(part, BF16)
    with pytest.raises(RuntimeError, match="overwritten"):
        ops.norm_linear(old, _rand(gen, 1024), 1e-6, _rand(gen, 2, 1024), _rand(gen, 4096, 1024))


@pytest.mark.parametrize("n,k", [(4112, 4096), (16400, 2176), (40976, 4096)])
@pytest.mark.parametrize("gated", [False, True])
def test_bits_of_the_two_launches_wherever_a_row_begins(gpu, n, k, gated):
    """As above with a long k, whose sums begin at different places of it: workgroups of 16 and of 32 rows of weights begin alike for the same row."""
    gen = torch.Generator().manual_seed(n + k)
    w, gain, x = _rand(gen, n, k, std=0.05), _rand(gen, k), _rand(gen, 1, k)
    got, _ = ops.norm_linear(x, gain, 1e-6, None, w, gated)
    want = ops.skinny_linear(ops.rms_norm(x, gain, 1e-6), w)
    if gated:
        both, want = want, torch.empty(1, n // 2, dtype=BF16, device=gpu)
        ops.silu_and_mul(want, both)
    assert torch.equal(got, want)
