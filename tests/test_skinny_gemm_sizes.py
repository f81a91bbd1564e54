"""The scratch memory that split products of a decode step ask for: the library's own answers, nothing is launched."""
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
