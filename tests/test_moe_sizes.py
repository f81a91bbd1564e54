"""Rows per tile of the experts' products by size: the library's own answer, nothing is launched.  With 18 to 112 choices per expert and k in whole steps tiles of 32
and 128 rows say no more than where spans of 128 begin, and tiles of 256 that experts with more rows than that go in blocks."""
import ctypes

import pytest

from infer_amd import _lib


def layout(n, width, ff, experts, top, elem):
    out = (ctypes.c_int64 * 3)()
    assert _lib.load().infer_moe_layout(elem, n, width, -(-ff // 8) * 8, experts, top, ctypes.addressof(out)) == 0
    return list(out)


@pytest.mark.parametrize("width,ff,experts,top,n,rows", [
    # few choices per expert, of few and of many weights and experts
    (4096, 3072, 14, 3, 64, 32), (4096, 3072, 14, 3, 130, 32), (4096, 3072, 14, 3, 140, 256), (1024, 768, 14, 3, 149, 32), (1536, 4096, 8, 2, 128, 32),
    (2048, 768, 128, 8, 384, 32), (2048, 768, 128, 8, 400, 256), (2880, 2880, 32, 4, 192, 32), (2880, 2880, 32, 4, 200, 256), (4096, 14336, 8, 2, 104, 256),
    # blocks: many, or of much to do
    (4096, 3072, 14, 3, 8000, 256), (4096, 3072, 14, 3, 160, 256), (1024, 3072, 14, 3, 200, 128), (1024, 3072, 14, 3, 900, 256), (2048, 3072, 24, 4, 210, 128),
    (2048, 3072, 24, 4, 340, 256), (2048, 8192, 8, 2, 200, 128), (2048, 8192, 8, 2, 440, 256), (1536, 4096, 8, 2, 224, 256), (768, 64, 4, 1, 300, 128)])
def test_rows_per_tile(width, ff, experts, top, n, rows):
    from infer_amd.hybrid_ops import ELEM
    import torch
    places, tiles, per = layout(n, width, ff, experts, top, ELEM[torch.bfloat16])
    assert per == rows and places == n * top
    assert tiles >= -(-n * top // per) and tiles <= n * top // per + experts
