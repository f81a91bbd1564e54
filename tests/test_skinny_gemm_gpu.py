"""Split-K weight-streaming GEMM (decode-sized batches) against a float32 reference.

Bar: the bf16 result is within two bf16 steps of the float32 product rounded once (the vendor GEMM
meets the same bar: both accumulate in float32, in different orders)."""
import pytest
import torch

from infer_amd import ops

pytestmark = pytest.mark.gpu


def reference(x, w):
    return x.float() @ w.float().T


def close(got, want):
    assert torch.isfinite(got.float()).all()
    err = (got.float() - want).abs()
    assert (err <= 2.0 ** -6 * want.abs() + 2e-2).all(), float(err.max())


@pytest.mark.parametrize("m,n,k", [
    (128, 4096, 12288),      # down_proj of Qwen3-8B: split over K
    (128, 4096, 4096),       # o_proj
    (64, 6144, 4096), (16, 4096, 4096), (1, 4096, 4096), (17, 1024, 1024), (100, 5120, 8192),
    (128, 24576, 4096),      # gate_up: enough tiles, no split
    (33, 136, 128),          # ragged N (not a multiple of the tile), a single chunk
    (128, 264, 384), (5, 8, 128),
])
def test_against_float32(gpu, m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(gpu)
    w = (torch.randn(n, k, generator=g) * 0.05).to(torch.bfloat16).to(gpu)
    got = ops.skinny_linear(x, w)
    torch.cuda.synchronize()
    close(got, reference(x, w))
    lib = torch.nn.functional.linear(x, w)
    assert (got.float() - lib.float()).abs().max() <= 2.0 ** -6 * reference(x, w).abs().max() + 2e-2


def test_strided_input_and_output_views(gpu):
    g = torch.Generator().manual_seed(0)
    wide = torch.randn(48, 1024 + 256, generator=g).to(torch.bfloat16).to(gpu)
    x = wide[:, 256:]                                   # row stride 1280, 16-byte aligned start
    w = (torch.randn(512, 1024, generator=g) * 0.05).to(torch.bfloat16).to(gpu)
    out_wide = torch.zeros(48, 512 + 64, dtype=torch.bfloat16, device=gpu)
    ops.skinny_linear(x, w, out_wide[:, :512])
    torch.cuda.synchronize()
    close(out_wide[:, :512], reference(x, w))
    assert not out_wide[:, 512:].any()


def test_exact_small_integers(gpu):
    """Products and sums of small integers are exact in bf16 x bf16 -> float32: any indexing mistake
    (a wrong row, a dropped or doubled K chunk, a misplaced partial sum) changes the result."""
    g = torch.Generator().manual_seed(1)
    x = torch.randint(-1, 2, (77, 1536), generator=g).to(torch.bfloat16).to(gpu)
    w = torch.randint(-1, 2, (4096, 1536), generator=g).to(torch.bfloat16).to(gpu)
    got = ops.skinny_linear(x, w)
    want = reference(x, w)
    assert want.abs().max() < 256                       # representable in bf16 without rounding
    assert torch.equal(got.float(), want)


def test_unsupported_shapes_are_refused(gpu):
    w = torch.zeros(64, 192, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(RuntimeError):
        ops.skinny_linear(torch.zeros(4, 192, dtype=torch.bfloat16, device=gpu), w)        # K % 128 != 0
    w = torch.zeros(64, 256, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(RuntimeError):
        ops.skinny_linear(torch.zeros(129, 256, dtype=torch.bfloat16, device=gpu), w)      # M > 128
    assert not ops.skinny_linear_supported(129, 64, 256)
    assert not ops.skinny_linear_supported(4, 64, 192)


def test_linear_picks_one_kernel_per_shape_and_matches(gpu):
    g = torch.Generator().manual_seed(2)
    x = torch.randn(128, 12288, generator=g).to(torch.bfloat16).to(gpu)
    w = (torch.randn(4096, 12288, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    a = ops.linear(x, w)
    b = ops.linear(x, w)
    assert torch.equal(a, b)                             # the choice is sticky: same kernel, same bits
    close(a, reference(x, w))
    big = torch.randn(300, 12288, generator=g).to(torch.bfloat16).to(gpu)
    close(ops.linear(big, w), reference(big, w))         # larger batches take the vendor GEMM


@pytest.mark.parametrize("m,n,k,with_residual", [(128, 4096, 12288, True), (40, 4096, 4096, True), (7, 1024, 2048, False)])
def test_rms_norm_adds_unreduced_partial_sums_to_the_same_bits(gpu, m, n, k, with_residual):
    """RMSNorm fed with the unreduced split-K result must give exactly what reducing first gives."""
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(gpu)
    w = (torch.randn(n, k, generator=g) * 0.03).to(torch.bfloat16).to(gpu)
    gamma = (1 + 0.2 * torch.randn(n, generator=g)).to(torch.bfloat16).to(gpu)
    res_a = torch.randn(m, n, generator=g).to(torch.bfloat16).to(gpu) if with_residual else None
    res_b = res_a.clone() if with_residual else None
    finished = ops.skinny_linear(x, w)
    want = ops.rms_norm(finished, gamma, 1e-6, res_a)
    deferred = ops.skinny_linear_deferred(x, w)
    assert isinstance(deferred, ops.SplitKSum) and deferred.partial.shape[0] > 1
    assert torch.equal(deferred.materialize(), finished)
    got = ops.rms_norm(deferred, gamma, 1e-6, res_b)
    torch.cuda.synchronize()
    if with_residual:
        assert torch.equal(got[0], want[0]) and torch.equal(res_b, res_a)
    else:
        assert torch.equal(got, want)


def test_partial_sums_cannot_be_used_after_a_later_split_gemm(gpu):
    x = torch.zeros(8, 4096, dtype=torch.bfloat16, device=gpu)
    w = torch.zeros(1024, 4096, dtype=torch.bfloat16, device=gpu)
    first = ops.skinny_linear_deferred(x, w)
    assert isinstance(first, ops.SplitKSum)
    ops.skinny_linear_deferred(x, w)
    with pytest.raises(RuntimeError, match="overwritten"):
        ops.rms_norm(first, torch.ones(1024, dtype=torch.bfloat16, device=gpu), 1e-6)


@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(8, 128), (136, 256), (1024, 2048), (4096, 640), (5120, 512), (5128, 128), (6152, 384), (8200, 256), (12296, 128), (16400, 128),
                                 (20488, 128), (24584, 256), (40968, 128), (65544, 128)])
def test_streamed_weights_around_tiles_and_rules(gpu, m, n, k):
    """Small integers, whose products and sums are exact: every number of rows per workgroup, the last rows of the weights and of the
    batch, k of one step per wavefront and fewer; unreduced sums add up to the same."""
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randint(-1, 2, (m, k + 8), generator=g, device=gpu).to(torch.bfloat16)[:, 8:]
    w = torch.randint(-1, 2, (n, k), generator=g, device=gpu).to(torch.bfloat16)
    want = reference(x, w)
    assert want.abs().max() <= 256                      # representable in bf16 without rounding
    assert torch.equal(ops.skinny_linear(x, w).float(), want)
    deferred = ops.linear(x, w, defer=True)
    assert torch.equal((deferred.materialize() if isinstance(deferred, ops.SplitKSum) else deferred).float(), want)


@pytest.mark.parametrize("m", [8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("n,k", [(136, 8192), (4104, 8320), (5120, 8064), (5128, 8192)])
def test_streamed_weights_of_a_long_k(gpu, m, n, k):
    """As above around the line from which few weight rows are cut over k; one in four activations is not zero, so that sums stay below 256."""
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = (torch.randint(-1, 2, (m, k), generator=g, device=gpu) * (torch.rand((m, k), generator=g, device=gpu) < 0.25)).to(torch.bfloat16)
    w = torch.randint(-1, 2, (n, k), generator=g, device=gpu).to(torch.bfloat16)
    want = reference(x, w)
    assert want.abs().max() <= 256                      # representable in bf16 without rounding
    assert torch.equal(ops.skinny_linear(x, w).float(), want)
    deferred = ops.linear(x, w, defer=True)
    assert torch.equal((deferred.materialize() if isinstance(deferred, ops.SplitKSum) else deferred).float(), want)


@pytest.mark.parametrize("m", [33, 48, 64])
@pytest.mark.parametrize("n,k", [(1536, 9728), (1000, 9728), (4616, 6656), (4608, 3072), (5120, 3200)])
def test_streamed_weights_cut_into_more_workgroups_than_compute_units_and_fewer(gpu, m, n, k):
    """As above: more workgroups than compute units, and factors that leave 146 and 216 of them."""
    test_streamed_weights_of_a_long_k(gpu, m, n, k)


@pytest.mark.parametrize("m", [1, 16, 17, 40, 64, 65])
@pytest.mark.parametrize("ff,k", [(8, 128), (2568, 256), (3072, 1024), (4104, 384), (6160, 256), (10248, 128), (12288, 512)])
def test_gate_and_up_in_one_launch_have_the_bits_of_two(gpu, m, ff, k):
    g = torch.Generator(device=gpu).manual_seed(m + ff)
    x = torch.randn(m, k, generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randn(2 * ff, k, generator=g, device=gpu) * 3 * k ** -0.5).to(torch.bfloat16)
    want = torch.empty(m, ff, dtype=torch.bfloat16, device=gpu)
    ops.silu_and_mul(want, ops.linear(x, w))
    got = ops.gate_up_silu(x, w)
    assert torch.equal(got, want)
    # neither may be wrong: roundings to bfloat16 (half of the last of 8 bits: 2^-8 each) of the gate, the up column, the activation and the
    # result, to second order in the gate's, where the activation's slope may be zero (its second derivative is 0.5 at most); float32 sums
    gate, up = (x.double() @ half.double().t() for half in (w[:ff], w[ff:]))
    sums = [1e-6 * x.double().abs() @ half.double().abs().t() for half in (w[:ff], w[ff:])]
    silu, slope = torch.sigmoid(gate) * gate, torch.sigmoid(gate) * (1 + gate * (1 - torch.sigmoid(gate)))
    shift = 2.0 ** -8 * gate.abs() + sums[0]
    bound = 1.02 * (2.0 ** -8 * 3 * silu.abs() * up.abs() + sums[1] * silu.abs() + (slope.abs() * shift + 0.25 * shift ** 2) * up.abs())
    assert ((got.double() - silu * up).abs() <= bound + 1e-30).all()


def test_linear_takes_what_the_streaming_kernel_cannot(gpu):
    """Odd strides and starts, rows on top of each other, a gradient: the vendor GEMM, as before."""
    g = torch.Generator(device=gpu).manual_seed(3)
    w = torch.randn(512, 256, generator=g, device=gpu).to(torch.bfloat16)
    wide = torch.randn(9, 300, generator=g, device=gpu).to(torch.bfloat16)
    for x in (wide[:, 3:259], wide[1:2, 8:264], wide[:1, :256].expand(5, 256), wide[:, :256]):
        close(ops.linear(x, w), reference(x, w))
    x = wide[:, :256].contiguous().requires_grad_()
    ops.linear(x, w).float().sum().backward()
    assert torch.isfinite(x.grad.float()).all()


def test_split_products_on_two_streams_do_not_meet(gpu):
    g = torch.Generator(device=gpu).manual_seed(4)
    x = torch.randn(8, 4096, generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randn(1024, 4096, generator=g, device=gpu) * 0.05).to(torch.bfloat16)
    gamma = torch.ones(1024, dtype=torch.bfloat16, device=gpu)
    first = ops.skinny_linear_deferred(x, w)
    want = ops.rms_norm(first, gamma, 1e-6)
    first = ops.skinny_linear_deferred(x, w)
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        second = ops.skinny_linear_deferred(-x, w)
        assert second.partial.data_ptr() != first.partial.data_ptr()
        minus = ops.rms_norm(second, gamma, 1e-6)
    other.synchronize()
    assert torch.equal(ops.rms_norm(first, gamma, 1e-6), want) and torch.equal(minus, -want)


@pytest.mark.parametrize("m", [9, 24, 64])
@pytest.mark.parametrize("n", [8176, 16368, 24560, 32752, 40944, 49136, 57328, 65520, 81904])
@pytest.mark.parametrize("k", [2176, 256])
def test_steps_that_wavefronts_share(gpu, m, n, k):
    """Exact sums for 2 to 20 tiles of weight rows per workgroup, the last one ragged: fewer steps of k than are under way at a time, and a walk over k that
    begins somewhere else in every workgroup and goes on at the front.  Gate and up in one launch round where the two do."""
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randint(-1, 2, (m, k + 8), generator=g, device=gpu).to(torch.bfloat16)[:, 8:]
    w = torch.randint(-1, 2, (n, k), generator=g, device=gpu, dtype=torch.int8).to(torch.bfloat16)
    want = reference(x, w)
    assert want.abs().max() <= 256                      # representable in bf16 without rounding
    assert torch.equal(ops.skinny_linear(x, w[:-8]).float(), want[:, :-8])
    both, fused = (torch.empty(m, n // 2, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    ops.silu_and_mul(both, want.to(torch.bfloat16))
    rc = ops._lib.load().infer_skinny_gate_silu_bf16(x.data_ptr(), x.stride(0), w.data_ptr(), fused.data_ptr(), n // 2, m, n // 2, k,
                                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(fused, both)


@pytest.mark.parametrize("m", [65, 96, 113, 128])
@pytest.mark.parametrize("n,k", [(8, 128), (136, 256), (1024, 1536), (4104, 2176), (8184, 2304), (24584, 256)])
def test_more_than_64_of_the_batch(gpu, m, n, k):
    """Exact sums for four and eight tiles of weight rows, cut over k and whole, around the last rows of both."""
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randint(-1, 2, (m, k + 8), generator=g, device=gpu).to(torch.bfloat16)[:, 8:]
    w = torch.randint(-1, 2, (n, k), generator=g, device=gpu).to(torch.bfloat16)
    want = reference(x, w)
    assert want.abs().max() <= 256                      # representable in bf16 without rounding
    assert torch.equal(ops.skinny_linear(x, w).float(), want)
    deferred = ops.skinny_linear_deferred(x, w)
    assert torch.equal((deferred.materialize() if isinstance(deferred, ops.SplitKSum) else deferred).float(), want)


@pytest.mark.parametrize("m", [32, 33, 64])
@pytest.mark.parametrize("n,k", [(4096, 16384), (4104, 16384), (5120, 16256), (5120, 16384)])
def test_a_very_long_k(gpu, m, n, k):
    """Around the line from which more than 4096 weight rows go 128 to a workgroup; one in eight activations is not zero, so that sums stay below 256."""
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = (torch.randint(-1, 2, (m, k), generator=g, device=gpu) * (torch.rand((m, k), generator=g, device=gpu) < 0.125)).to(torch.bfloat16)
    w = torch.randint(-1, 2, (n, k), generator=g, device=gpu).to(torch.bfloat16)
    want = reference(x, w)
    assert want.abs().max() <= 256                      # representable in bf16 without rounding
    assert torch.equal(ops.skinny_linear(x, w).float(), want)


@pytest.mark.parametrize("m", [1, 3, 9, 17, 33, 64])
@pytest.mark.parametrize("ff", [2632, 4104, 6152, 8200, 9728, 12288, 12296, 20496])
@pytest.mark.parametrize("k", [2048, 2176, 4096])
def test_gate_and_up_of_a_long_k_have_the_bits_of_two(gpu, m, ff, k):
    """Walks over k begin at different places of it, so every sum has an order of its own: the same one in both, for 16 to 256 weight rows per workgroup, halves that
    are whole workgroups and halves that are not."""
    g = torch.Generator(device=gpu).manual_seed(m + ff + k)
    x = torch.randn((m, k), generator=g, device=gpu).to(torch.bfloat16)
    w = (0.05 * torch.randn((2 * ff, k), generator=g, device=gpu)).to(torch.bfloat16)
    want, got = (torch.empty(m, ff, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    ops.silu_and_mul(want, ops.skinny_linear(x, w))
    rc = ops._lib.load().infer_skinny_gate_silu_bf16(x.data_ptr(), k, w.data_ptr(), got.data_ptr(), ff, m, ff, k, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(got, want)
