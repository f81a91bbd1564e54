"""The look over the assembly of hand-written products, on assembly with and without the mistakes that it is for."""
import importlib.util
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
spec = importlib.util.spec_from_file_location("check_products", os.path.join(HERE, "..", "infer_amd", "csrc", "check_products.py"))
check_products = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_products)

PRODUCT = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"
OTHERS = [f"v_mfma_f32_16x16x32_bf16 a[{4 * i}:{4 * i + 3}], v[0:3], v[4:7], a[{4 * i}:{4 * i + 3}]" for i in range(1, 21)]


def kernel(body, scratch=0, name="_Z12block_kernelv"):
    return "\n".join([f"{name}:", *("\t" + line if not line.startswith(".") else line for line in body), "\ts_endpgm", ".Lfunc_end0:",
                      f"\t.amdhsa_kernel {name}", "\t\t.amdhsa_group_segment_fixed_size 0", f"\t\t.amdhsa_private_segment_fixed_size {scratch}"])


GOOD = {
    "reads, products, a pause, results": ["ds_read_b128 v[0:3], v9", "s_waitcnt lgkmcnt(0)", PRODUCT, *OTHERS, "s_nop 15", "s_nop 15", "v_accvgpr_read_b32 v8, a0"],
    "a copy far enough in front": ["v_mov_b32_e32 v5, v12", "s_nop 2", PRODUCT],
    "a loop around them": [".LBB0_1:", PRODUCT, *OTHERS, "ds_read_b128 v[0:3], v9", "s_cbranch_scc1 .LBB0_1"],
    "others' registers": ["v_mov_b32_e32 v8, v12", PRODUCT, "v_add_f32_e32 v8, v8, v8 ; v[0:3]"],
}
BAD = {
    "a copy right in front": ["v_mov_b32_e32 v5, v12", "s_nop 0", PRODUCT],
    "an accumulator written right in front": ["v_accvgpr_write_b32 a2, v12", PRODUCT],
    "a result read at once": [PRODUCT, "s_nop 7", "v_accvgpr_read_b32 v8, a3"],
    "a result stored at once": [PRODUCT, "scratch_store_dwordx4 off, a[0:3], off"],
    "a result moved at once": [PRODUCT, "v_accvgpr_mov_b32 a99, a1"],
    "a copy at the end of a loop": [".LBB0_1:", PRODUCT, *OTHERS, "v_mov_b32_e32 v5, v12", "s_cbranch_scc1 .LBB0_1"],
    "a result read behind a branch": [PRODUCT, "s_cbranch_scc1 .LBB0_2", "s_nop 15", "s_nop 15", ".LBB0_2:", "v_accvgpr_read_b32 v8, a3"],
    "a result that enters the next product": [PRODUCT, PRODUCT],
}
INLINE = [";;#ASMSTART", PRODUCT, ";;#ASMEND"]
GOOD["products of the compiler's, which keeps their distances"] = [*INLINE, *OTHERS, OTHERS[0], "v_accvgpr_read_b32 v8, a4"]
BAD["a product in assembly beside others, its result read at once"] = [*OTHERS, *INLINE, "v_accvgpr_read_b32 v8, a0"]
BAD["a result that enters a product of the compiler's"] = [*INLINE, PRODUCT]
BAD["a result of a product of the compiler's"] = [PRODUCT, *INLINE]
BAD["a copy in front of assembly"] = ["v_mov_b32_e32 v5, v12", *INLINE]


@pytest.mark.parametrize("body", GOOD.values(), ids=GOOD)
def test_passes(body):
    assert check_products.check(kernel(body), "block_kernel") == []


@pytest.mark.parametrize("body", BAD.values(), ids=BAD)
def test_reports(body):
    assert check_products.check(kernel(body), "block_kernel")


def test_reports_scratch_memory_and_a_kernel_that_is_not_there():
    assert check_products.check(kernel([PRODUCT], scratch=16), "block_kernel")
    assert check_products.check(kernel([PRODUCT]), "other_kernel")
    assert check_products.check(kernel(["s_nop 0"]), "block_kernel")
