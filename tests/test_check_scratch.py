"""The look over the compiler's report on spilled registers, and the report of the last build where there is one."""
import importlib.util
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "infer_amd", "csrc")
spec = importlib.util.spec_from_file_location("check_scratch", os.path.join(CSRC, "check_scratch.py"))
check_scratch = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_scratch)


def report(**spills):
    return "".join(f"a.hip:3:1: remark: Function Name: {name} [-Rpass]\na.hip:3:1: remark:     VGPRs: 256 [-Rpass]\n"
                   f"a.hip:3:1: remark:     SGPRs Spill: 7 [-Rpass]\na.hip:3:1: remark:     VGPRs Spill: {n} [-Rpass]\n" for name, n in spills.items())


def test_the_first_name_that_fits_decides():
    text = report(_Z5walkILi8EEvv=20, _Z5walkILi4EEvv=1, _Z4sumsv=3)
    assert check_scratch.check(text, {"walkILi8E": 20, "walk": 1}) == []
    assert len(check_scratch.check(text, {"walkILi8E": 19, "walk": 1})) == 1
    assert len(check_scratch.check(text, {"walkILi8E": 20, "walk": 0})) == 1
    assert len(check_scratch.check(text, {"walk": 1})) == 1
    assert check_scratch.check(text, {"sums": 3}) == [] and check_scratch.check(text, {"sums": 2})


def test_a_kernel_that_is_not_there():
    assert check_scratch.check(report(_Z4sumsv=0), {"walk": 100})
    assert check_scratch.check("", {"walk": 100})


@pytest.mark.parametrize("source,limits", [("talking_prefill", {"talk_mix_kernelILi4ELi8ELi4E": 20, "talk_mix_kernel": 9, "talk_lse_kernel": 0}),
                                           ("dense_prefill", {"dense_prefill_kernelILi8E": 33, "dense_prefill": 0})])
def test_last_build(source, limits):
    path = os.path.join(CSRC, source + ".resources.txt")
    if not os.path.exists(path):
        pytest.skip("not built here")
    with open(path) as f:
        text = f.read()
    assert check_scratch.check(text, limits) == []
