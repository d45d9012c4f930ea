"""The runtime loads a module's whole code at the first launch out of it: the kernels of the products on the matrix cores lie in three modules
for each type of x and of the scales (cubek_amd/csrc/Makefile), so that a launch loads one kind of them."""
import os
import subprocess

from test_build_flags import ROOT, compile_lines


def test_products_on_the_matrix_cores_load_one_kind_of_kernel():
    lines = compile_lines()
    batches = [line for line in lines if "cq_kernels_gemv_batch" in line]
    assert len(batches) == 6
    for line in batches:
        compiled = [command for command in line.split("&&") if " -c " in command]
        assert [("cq_kernels_gemv_quads.hip" in c, "-DCQ_GEMV_LINES=0" in c, "-DCQ_GEMV_LINES=1" in c) for c in compiled] == \
            [(True, False, False), (False, True, False), (False, False, True)]
    symbols = subprocess.run(["nm", os.path.join(ROOT, "cubek_amd", "lib", "libcubek_quant_hip.so")], stdout=subprocess.PIPE, text=True, check=True).stdout
    assert symbols.count(" __hip_module_ctor\n") == sum(line.count(" -c ") for line in lines) == 51 + 2 * 6
