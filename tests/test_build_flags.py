"""What the objects of the library are compiled with (cubek_amd/csrc/Makefile)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def compile_lines():
    out = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "cubek_amd", "csrc"), "../lib/libcubek_quant_hip.so"],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert out.returncode == 0, out.stdout
    return [line for line in out.stdout.replace("\\\n", " ").splitlines() if " -c " in line]


def test_arguments_are_preloaded_except_for_the_flat_dequantize_kernels():
    """Preloaded arguments cost those kernels 2 - 5 %."""
    lines = compile_lines()
    dequantize = [line for line in lines if "cq_kernels_flat_dequantize.hip" in line]
    assert len(lines) == 51 and len(dequantize) == 11
    for line in lines:
        assert ("-amdgpu-kernarg-preload-count=16" in line) == (line not in dequantize), line


def test_every_object_is_compiled_without_packed_f32_arithmetic():
    for line in compile_lines():
        assert "-Xclang -target-feature -Xclang -packed-fp32-ops" in line and "-ffp-contract=off" in line, line
