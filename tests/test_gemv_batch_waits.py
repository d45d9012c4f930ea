"""The product with several vectors (cubek_amd/csrc/cq_kernels_gemv_batch.hip), looked up in the assembly of one of the file's objects.

It overwrites the half of its shared memory that the previous stage was read from: whatever a wave has asked of shared memory has to have
come back before it arrives at the barrier that lets the others overwrite it.

Codes are streamed past the caches where rows are whole lines and not where they are parts of them, by a kernel each: a choice in every
stage cost whole lines up to 5 %.  It stays where parts of lines are the faster with it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    asm = tmp_path_factory.mktemp("gemv_batch") / "gemv_batch.s"
    build = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-fast-math",
                            "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-DCQ_GEMV_PART=5",
                            "--cuda-device-only", "-S", os.path.join(ROOT, "cubek_amd", "csrc", "cq_kernels_gemv_batch.hip"), "-o", str(asm)],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout
    lines = [line.split(";")[0].strip() for line in asm.read_text().splitlines()]
    return [line for line in lines if line]


def test_every_barrier_stands_behind_a_wait_for_shared_memory(lines):
    barriers = [i for i, line in enumerate(lines) if line == "s_barrier"]
    assert len(barriers) >= 40 * 3  # five codes in four shapes for two kinds of rows, one barrier in the loop and two behind it
    for i in barriers:
        before = i - 1
        while not lines[before].startswith("s_waitcnt"):
            assert re.match(r"s_|v_", lines[before]), lines[before:i + 1]  # no access and no label between the wait and the barrier
            before -= 1
        assert "lgkmcnt(0)" in lines[before], lines[before:i + 1]


def test_whole_lines_are_streamed_without_a_choice(lines):
    loads, kernel = {}, ""
    for line in lines:
        if re.match(r"_Z\w+:$", line):
            kernel = line
        elif line.startswith("global_load_lds_dwordx4") and "gemv_batch_kernel" in kernel:
            loads.setdefault(kernel, []).append(line.endswith(" nt"))
    assert len(loads) == 40  # five codes in four shapes, whole lines and parts of lines
    for kernel, nt in loads.items():
        # the codes' loads are those of a stage of eight units of 16 rows, two to a stage, for the first stage and the others
        assert sum(nt) == (4 if "ELb1E" in kernel or "ELi4ELi2ELb0E" in kernel else 0), (kernel, nt)
    plain = {re.sub("ELb[01]E", "", kernel): len(nt) - sum(nt) for kernel, nt in loads.items() if "ELb1E" in kernel}
    for kernel, nt in loads.items():  # parts of lines: the codes' four as well
        assert "ELb1E" in kernel or len(nt) - sum(nt) == plain[re.sub("ELb[01]E", "", kernel)] + 4, (kernel, nt)
