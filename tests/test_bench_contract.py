"""bench.py's command line contract that can be checked without a GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], stdout=subprocess.PIPE,
                          stderr=subprocess.PIPE, text=True, timeout=120)
    assert proc.returncode != 0
    assert "one GPU" in proc.stderr and proc.stdout.strip() == ""


def test_world_size_from_a_launcher_is_refused_too():
    env = dict(os.environ, WORLD_SIZE="2", RANK="0")
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py")], stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                          text=True, timeout=120, env=env)
    assert proc.returncode != 0 and "one GPU" in proc.stderr


def test_bench_probe_library_loads():
    """bench.py's memory yardsticks (cubek_amd/csrc/cq_bench_probes.hip): the library is built, exports its entry
    points, and refuses bad arguments before it touches the GPU."""
    import ctypes

    import bench

    assert os.path.exists(bench.PROBES_PATH), "make -C cubek_amd/csrc builds it"
    L = ctypes.CDLL(bench.PROBES_PATH)
    L.cq_probe_run.restype = ctypes.c_int
    L.cq_probe_run.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64,
                               ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint64)]
    assert L.cq_probe_run(0, None, None, None, 100, None, None) == -1      # less than one tile
    assert L.cq_probe_run(7, None, None, None, 1 << 20, None, None) == -1  # no such probe
    L.cq_probe_shape.restype = ctypes.c_int
    L.cq_probe_shape.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64,
                                 ctypes.c_uint32, ctypes.POINTER(ctypes.c_uint64), ctypes.POINTER(ctypes.c_uint64)]
    assert L.cq_probe_shape(0, None, None, None, 100, 320, None, None) == -1       # less than one tile
    assert L.cq_probe_shape(0, None, None, None, 1 << 20, 0, None, None) == -1     # nothing on the narrow side
    assert L.cq_probe_shape(1, None, None, None, 1 << 20, 1025, None, None) == -1  # narrow side wider than the wide one
    L.cq_probe_transposed.restype = ctypes.c_int
    L.cq_probe_transposed.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p,
                                      ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32]
    assert L.cq_probe_transposed(0, 0, 0, None, None, None, None, 100, 256) == -1   # rows not in whole tiles
    assert L.cq_probe_transposed(1, 1, 1, None, None, None, None, 128, 0) == -1     # no columns


def test_the_printed_line_is_short_and_whole():
    """Everything that is measured goes to a file; the line holds the contract's fields and the roofline in brief."""
    import json

    import bench

    fractions = {f"cfg{i}": {"dynamic": 0.7654, "given": 0.7654, "dequantize": 0.7654} for i in range(1, 6)}
    roofline = dict(bound="hbm", kernel="quantize_flat_kernel (fused abs-max+scale+quantize+pack)", achieved=6536.3, peak=8000.0, unit="GB/s", frac=0.8171,
                    traffic=616710144, median_launch_ms=0.0943, per_config=fractions, min_frac_cfg3_5=0.7543, in_step={"note": "x" * 300})
    result = dict(metric="quant/dequant GB/s (bytes read+written) and % of MI355X HBM peak, 1 GPU", value=6991.5, unit="GB/s", n_gpus=1, steps=20, warmup=5,
                  ms_per_step=0.1764, higher_is_better=True, scaling="weak", vs_baseline=None, dtype="bf16", data="synthetic",
                  config=dict(workload="cfg5: " + "x" * 120, shape=[28672, 8192], block=32, value="E2M1", store="U32", param="F32",
                              algorithmic_bytes_per_step=1233125376), pct_hbm_peak=87.4, elements_per_s=2663049705215, value_note="x" * 500,
                  roofline=roofline, roofline_dequantize=roofline, first_call_ms={"quantize_dynamic": 1.8, "dequantize": 1.0, "library_bytes": 1},
                  cpu_baseline={"value": 5.29, "unit": "GB/s", "cores": 16, "what": "x" * 200}, per_config=[{"x": "y" * 1000}] * 5)
    line = bench.one_line(result)
    assert len(line) < 1800 and "\n" not in line
    got = json.loads(line)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert got[key] == result[key]
    assert got["roofline"]["frac"] == 0.8171 and got["cpu_baseline"]["value"] == 5.29
