"""Which rows the chunk kernels of the delta rule read for their convolution, from the header that says so, compiled for the host."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "infer_amd", "csrc")


@pytest.fixture(scope="module")
def window_row(tmp_path_factory):
    d = tmp_path_factory.mktemp("window")
    (d / "w.cpp").write_text('#include "conv_window.h"\n'
                             'extern "C" int window(int count, int pos0, int first_pos, int t) { return (int)window_row(count, pos0, first_pos, t); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-I", CSRC, str(d / "w.cpp"), "-o", str(d / "w.so")], check=True)
    return ctypes.CDLL(str(d / "w.so")).window


def test_rows_lie_in_the_portion_or_the_ring(window_row):
    """Portions of 0 to 40 tokens that begin at positions 0 to 20, chunks of 16, an empty one at every place between them: a row of the batch is one of the portion
    that does not lie behind the chunk, an entry of the ring one of the three positions in front of the portion, all others are not read."""
    for first in range(21):
        for n in range(41):
            chunks = [(lo, min(16, n - lo)) for lo in range(0, n, 16)]
            for lo, count in chunks + [(lo, 0) for lo in range(0, n + 1)]:
                for t in range(-3, 16):
                    pos = first + lo + t
                    want = 2 if count == 0 or t >= count or pos < 0 else 0 if lo + t >= 0 else 1
                    assert window_row(count, first + lo, first, t) == want, (first, n, lo, count, t)
                    if want == 1:
                        assert first - 3 <= pos < first
