"""Which products the decode kernels take by size, and the scratch memory they ask for: the library's own answers, nothing is launched."""
import itertools

import pytest

from infer_amd import _lib

ROWS = (1, 8, 9, 16, 17, 32, 33, 48, 64, 65, 128)
LONG = (1024, 1536, 2048, 4096, 6656, 8192, 9728, 12288, 25600)


@pytest.mark.parametrize("n", [8, 648, 1024, 2560, 3072, 4096, 5120, 5128, 12288, 32584])
def test_scratch_for_a_batch_is_enough_for_smaller_ones(n):
    need = _lib.load().infer_skinny_gemm_workspace_bytes
    for k in LONG:
        sizes = [need(m, n, k) for m in ROWS]
        assert sizes == sorted(sizes), (n, k, sizes)


def test_split_products_of_up_to_64_rows_run_in_one_round():
    """A workgroup of 64 weight rows past 33 to 64 of the batch takes a compute unit; a factor that makes 320 of them takes as long as 512."""
    need = _lib.load().infer_skinny_gemm_workspace_bytes
    for n, k in itertools.product((2560, 3072, 4608, 5120), (2048, 3072, 4096, 5120, 6144)):
        factor = need(64, n, k) // (64 * n * 4) or 1
        assert factor * -(-n // 64) <= 256, (n, k, factor)


@pytest.mark.parametrize("m,n,k,reduced,own", [
    # the projections of a decode step: hidden 1024 to 5120
    *[(m, n, k, r, 1) for m in (1, 16, 32, 64) for n, k, r in ((6144, 1024, 1), (1024, 3072, 0), (6144, 4096, 1), (24576, 4096, 1), (4096, 4096, 0),
                                                              (4096, 12288, 0), (34816, 5120, 1), (5120, 25600, 0), (151936, 4096, 1))],
    # where the vendor's product is ahead
    (16, 36864, 128, 1, 0), (64, 262144, 256, 1, 0), (1, 5128, 16384, 1, 0), (64, 24584, 28672, 1, 0), (48, 24584, 4096, 1, 0),
    (64, 65528, 5120, 1, 0), (32, 16384, 5120, 1, 0), (64, 5120, 1536, 1, 0), (16, 262144, 5120, 1, 0), (40, 512, 768, 1, 0), (24, 256, 1024, 1, 0), (65, 5128, 4096, 0, 0), (65, 4096, 1024, 0, 0),
    # pieces that a norm takes have no launch of their own
    (64, 5120, 1536, 0, 1), (65, 5120, 2048, 0, 1),
    # what they do not take at all
    (0, 4096, 4096, 1, 0), (129, 4096, 4096, 1, 0), (8, 4100, 4096, 1, 0), (8, 4096, 4160, 1, 0)])
def test_sizes_that_go_to_the_kernels(m, n, k, reduced, own):
    assert _lib.load().infer_skinny_gemm_pays(m, n, k, reduced) == own
