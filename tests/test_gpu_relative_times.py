"""Calls that move the same bytes in the same way take about the same time, whatever their types: each pair below was once
two or three times apart, which no comparison of results shows.  The limits leave half as much again for noise."""
import pytest

from cubek_amd import ComputeClient, ElemType, QuantScheme, TensorHandleRef
from cubek_amd import quantize as qz
from cubek_amd import reduce as rd

pytestmark = pytest.mark.gpu


def micros(*calls):
    """The best time of each call in microseconds, the calls taking turns."""
    import torch

    best = [float("inf")] * len(calls)
    for _ in range(8):
        for i, call in enumerate(calls):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            call()
            begin.record()
            for _ in range(20):
                call()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], begin.elapsed_time(end) * 50)
    return best


def max_abs(elem, rows, cols, axis, workspace=True, outer=()):
    """One abs-max over tensors of its own, as a function without arguments."""
    import torch

    dtype = torch.float32 if elem == ElemType.F32 else torch.bfloat16
    x = torch.randn(outer + (rows, cols), device="cuda").to(dtype)
    axis += len(outer)
    out = torch.empty(tuple(1 if d == axis else n for d, n in enumerate(x.shape)), dtype=dtype, device="cuda")
    h_x, h_out, client = TensorHandleRef.from_torch(x), TensorHandleRef.from_torch(out), ComputeClient.current()
    nbytes = rd.workspace_bytes(h_x, axis, elem) if workspace else 0
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    keep = (x, out, ws)
    return lambda: (rd.max_abs(client, h_x, h_out, axis, elem, ws.data_ptr() if workspace else 0, nbytes), keep)


def test_short_rows_of_f32_as_fast_as_of_bf16():
    f32, bf16 = micros(max_abs(ElemType.F32, 85302, 328, 1), max_abs(ElemType.BF16, 85302, 656, 1))  # 82 chunks of 16 bytes each
    assert f32 < 1.5 * bf16, (f32, bf16)


def test_few_long_rows_along_the_outer_axis_as_fast_as_many_short_ones():
    few, many = micros(max_abs(ElemType.F32, 64, 65536, 0), max_abs(ElemType.F32, 2048, 2048, 0))  # 16 MiB each
    assert few < 1.5 * many, (few, many)


def test_an_outer_axis_without_a_workspace_within_a_few_times_of_one_with_it():
    """[20000, 4097]: 36 us, and without room for slices 85 in tiles over the whole axis, 2100 by the few lanes that its columns are."""
    without, sliced = micros(max_abs(ElemType.BF16, 20000, 4097, 0, workspace=False), max_abs(ElemType.BF16, 20000, 4097, 0))
    assert without < 5 * sliced, (without, sliced)


def test_many_short_axes_as_fast_as_one_of_the_same_bytes():
    """[34978, 9, 23] along 9: 54 us with a workgroup for each of its matrices."""
    many, one = micros(max_abs(ElemType.BF16, 9, 23, 0, outer=(34978,)), max_abs(ElemType.BF16, 9, 34978 * 23, 0))
    assert many < 2.5 * one, (many, one)


def one_scale(mib, streams):
    """The time of a quantize with one scale of a bf16 tensor on each stream, until all of them have ended."""
    import time

    import torch

    h, scheme, calls = TensorHandleRef.from_torch, QuantScheme.default(), []
    for s in streams:
        x = torch.empty(mib << 19, dtype=torch.bfloat16, device="cuda").normal_()
        codes = torch.empty(scheme.packed_shape(x.shape), dtype=torch.int32, device="cuda")
        scale, ws = torch.empty(1, device="cuda"), torch.empty(1024, dtype=torch.uint8, device="cuda")
        calls.append((s, h(x), h(codes), h(scale), ws, (x, codes, scale)))

    def wall():
        torch.cuda.synchronize()
        begin = time.perf_counter()
        for _ in range(10):
            for s, x, codes, scale, ws, _ in calls:
                with torch.cuda.stream(s):
                    qz.launch_dynamic(ComputeClient.current(), x, codes, scale, scheme, ElemType.BF16, ws.data_ptr(), 1024)
        torch.cuda.synchronize()
        return (time.perf_counter() - begin) / 10

    return min(wall() for _ in range(4))


def test_four_times_the_tensor_takes_about_four_times_as_long():
    """One scale for 1 GiB and for 4 GiB: 430 and 1770 us; 445 and 2800 where workgroups gave up waiting for one another."""
    import torch

    large, small = one_scale(4096, [torch.cuda.Stream()]), one_scale(1024, [torch.cuda.Stream()])
    assert large < 5 * small, (large, small)


def test_four_streams_about_as_fast_as_one():
    """64 MiB a launch: 28 us on four streams by two passes; 310 where workgroups hold compute units while they wait for others."""
    import torch

    four, one = one_scale(64, [torch.cuda.Stream() for _ in range(4)]), one_scale(64, [torch.cuda.Stream()] * 4)
    assert four < 2.5 * one, (four, one)
