"""The product with several vectors (cubek_amd/csrc/cq_kernels_gemv_batch.hip) overwrites the half of its shared memory that
the previous stage was read from: whatever a wave has asked of shared memory has to have come back before it arrives at
the barrier that lets the others overwrite it.  Looked up in the assembly of one of the file's objects."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_barrier_stands_behind_a_wait_for_shared_memory(tmp_path):
    asm = tmp_path / "gemv_batch.s"
    build = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-fast-math",
                            "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-DCQ_GEMV_PART=5",
                            "--cuda-device-only", "-S", os.path.join(ROOT, "cubek_amd", "csrc", "cq_kernels_gemv_batch.hip"), "-o", str(asm)],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout
    lines = [line.split(";")[0].strip() for line in asm.read_text().splitlines()]
    lines = [line for line in lines if line]
    barriers = [i for i, line in enumerate(lines) if line == "s_barrier"]
    assert len(barriers) >= 20 * 3  # five codes in four shapes, one barrier in the loop and two behind it
    for i in barriers:
        before = i - 1
        while not lines[before].startswith("s_waitcnt"):
            assert re.match(r"s_|v_", lines[before]), lines[before:i + 1]  # no access and no label between the wait and the barrier
            before -= 1
        assert "lgkmcnt(0)" in lines[before], lines[before:i + 1]
