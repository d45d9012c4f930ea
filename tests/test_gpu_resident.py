"""One scale for a tensor, quantized in one read of it (cq_kernels_resident.hpp), against the two calls that share no
kernel with it: compute_scales, then quantize with the given scale.  Codes and scale bit for bit."""
import ctypes
import os

import numpy as np
import pytest

from cubek_amd import ComputeClient, ElemType, QuantParam, QuantScheme, QuantStore, QuantValue, TensorHandleRef
from cubek_amd import quantize as qz

pytestmark = pytest.mark.gpu
H = TensorHandleRef.from_torch
ROUND = 512 * 256  # chunks that all workgroups read in a step each


def dtype_of(torch, elem):
    return {ElemType.F32: torch.float32, ElemType.F16: torch.float16, ElemType.BF16: torch.bfloat16}[elem]


def scheme_of(value, store=QuantStore.U32, param=QuantParam.F32):
    return QuantScheme.default().with_value(value).with_store(store).with_param(param)


class Call:
    """A tensor of `n` values and the two results: of the fused call and of the two calls."""

    def __init__(self, torch, x, elem, scheme, fill=0xFF):
        n = x.numel()
        per = scheme.num_quants()
        self.torch, self.x, self.elem, self.scheme = torch, x, elem, scheme
        kind = torch.uint8 if scheme.store == QuantStore.Native else torch.int32
        self.codes = torch.zeros(n // per + 4, dtype=kind, device="cuda")  # four more, which have to stay zero
        self.shape = scheme.packed_shape((n,))
        param = {QuantParam.F32: torch.float32, QuantParam.F16: torch.float16, QuantParam.BF16: torch.bfloat16}[scheme.param]
        self.scale = torch.full((1,), -1.0, dtype=param, device="cuda")
        self.ws = torch.full((1024,), fill, dtype=torch.uint8, device="cuda")

    def fused(self):
        qz.launch_dynamic(ComputeClient.current(), H(self.x), H(self.codes[:self.shape[0]]), H(self.scale), self.scheme, self.elem,
                          self.ws.data_ptr(), 1024)

    def check(self, what):
        torch = self.torch
        given = torch.zeros(1, dtype=self.x.dtype, device="cuda")
        codes, scale, ws = torch.zeros_like(self.codes), torch.zeros_like(self.scale), torch.empty(1024, dtype=torch.uint8, device="cuda")
        client = ComputeClient.current()
        qz.compute_scales(client, H(self.x), H(given), self.scheme, self.elem, ws.data_ptr(), 1024)
        qz.launch_ref(client, H(self.x), H(codes[:self.shape[0]]), H(given), H(scale), self.scheme, self.elem)
        torch.cuda.synchronize()
        assert torch.equal(self.scale.view(torch.uint8), scale.view(torch.uint8)), (what, self.scale, scale)
        assert torch.equal(self.codes, codes), what


def values(torch, n, elem, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(n, generator=gen, device="cuda") * 0.02).to(dtype_of(torch, elem))


# chunks: single words, a cut step, the most for one workgroup and one more, both ends of 2 and of 8 chunks per lane, and one
# more than 8 (read twice); 48 MiB, where one read begins again for codes of 8 bits
SMALL = [4, 8, 508, 512, 516, 8 * 512, 8 * 512 + 4, 33 * 512 + 8, 2 * ROUND, 2 * ROUND + 4, 8 * ROUND - 4, 8 * ROUND, 8 * ROUND + 4, 24 * ROUND]


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value,store", [(QuantValue.Q8S, QuantStore.U32), (QuantValue.Q4F, QuantStore.U32), (QuantValue.Q2S, QuantStore.U32),
                                         (QuantValue.E4M3, QuantStore.Native), (QuantValue.E2M1, QuantStore.Native)],
                         ids=lambda v: v.name)
def test_small_sizes(elem, value, store):
    """The sizes at which the kernel's way changes; elements behind the last chunk where codes are bytes."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    for i, chunks in enumerate(SMALL):
        n = chunks * per + (3 if value == QuantValue.E4M3 else 0)
        x = values(torch, n, elem, i)
        x[(0, n - 1, n // 2)[i % 3]] = -0.75
        call = Call(torch, x, elem, scheme_of(value, store, QuantParam(i % 3)), fill=(0, 0x7F, 0xFF)[i % 3])
        call.fused()
        call.check((elem.name, value.name, chunks))


def test_many_small_launches():
    """More launches than there are regions of slots, on two streams, each with its workspace; then
    captured ones, replayed on new values between launches outside the graph."""
    import torch

    scheme = scheme_of(QuantValue.Q8S)
    calls = [Call(torch, values(torch, 8 * (512 * (3 + i) + 4), ElemType.BF16, i) * (i + 1), ElemType.BF16, scheme) for i in range(100)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(2):
        for i, call in enumerate(calls):
            with torch.cuda.stream(streams[i % 2]):
                call.fused()
    torch.cuda.synchronize()
    for i, call in enumerate(calls):
        call.check(i)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(streams[0]):
        with torch.cuda.graph(graph, stream=streams[0]):
            for call in calls[:3]:
                call.fused()
    for seed in (7, 8, 9):
        for i, call in enumerate(calls[:4]):
            call.x.copy_(values(torch, call.x.numel(), ElemType.BF16, seed + i) * (seed - 6))
            call.codes.zero_()
        torch.cuda.synchronize()
        graph.replay()
        calls[3].fused()
        torch.cuda.synchronize()
        for call in calls[:4]:
            call.check(seed)


KINDS = [(QuantValue.Q8S, QuantStore.U32, 60), (QuantValue.Q8F, QuantStore.U32, 61), (QuantValue.E4M3, QuantStore.Native, 64),
         (QuantValue.E5M2, QuantStore.Native, 65), (QuantValue.Q8S, QuantStore.Native, 48 + 13), (QuantValue.Q4S, QuantStore.U32, 96),
         (QuantValue.Q4F, QuantStore.U32, 113), (QuantValue.Q2S, QuantStore.U32, 129), (QuantValue.E2M1, QuantStore.Native, 96),
         (QuantValue.E2M1_OCP, QuantStore.U32, 96)]


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value,store,mib", KINDS, ids=lambda v: getattr(v, "name", str(v)))
def test_every_kind_of_code(elem, value, store, mib):
    import torch

    per = 4 if elem == ElemType.F32 else 8
    scheme = scheme_of(value, store)
    for chunks in (mib << 16, (mib << 16) + 4 * 77):  # whole rounds where the size is one; a cut step
        call = Call(torch, values(torch, chunks * per, elem, int(value) + chunks), elem, scheme)
        call.fused()
        call.check((elem.name, value.name, store.name, chunks))


# chunks: the fewest; on both sides of what registers, registers and LDS hold; one chunk in the last step; more than is held
SIZES = [60 << 16, 47 * ROUND + 1, 48 * ROUND, 48 * ROUND + 5, 64 * ROUND - 511, 64 * ROUND, 64 * ROUND + 1, 65 * ROUND + 512, 72 * ROUND + 13, 81 * ROUND - 1]


@pytest.mark.parametrize("elem,value,store,param", [(ElemType.BF16, QuantValue.Q8S, QuantStore.U32, QuantParam.F32),
                                                    (ElemType.F16, QuantValue.E4M3, QuantStore.Native, QuantParam.F16),
                                                    (ElemType.F32, QuantValue.Q8F, QuantStore.Native, QuantParam.BF16),
                                                    (ElemType.BF16, QuantValue.Q8S, QuantStore.Native, QuantParam.F16)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_sizes_and_ends(elem, value, store, param):
    """Every number of rounds that changes the kernel's way, with elements behind the last chunk (native store), the largest
    value in the first, in the last and in a middle place, a workspace of any content."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    for i, chunks in enumerate(SIZES):
        n = chunks * per + (3 if store == QuantStore.Native else 0)
        x = values(torch, n, elem, i)
        x[(0, n - 1, n // 2)[i % 3]] = -0.75
        call = Call(torch, x, elem, scheme_of(value, store, param), fill=(0, 0x3F, 0x7F, 0xFF)[i % 4])
        call.fused()
        call.check((elem.name, chunks))
        assert float(call.scale) > 0.001


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
def test_values_that_divide(elem):
    """Zeros, an infinity, abs-maxima whose divisor is no ordinary number, NaN elements, every 16-bit pattern."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    n = ((60 << 16) + 7) * per
    dt = dtype_of(torch, elem)
    base = values(torch, n, elem, 5)
    tiny = 2.0 ** -22 if elem == ElemType.F16 else 2.0 ** -124
    variants = [torch.zeros(n, dtype=dt, device="cuda"), (base.float().sign() * tiny).to(dt), base.clone(), base.clone(), base.clone()]
    variants[2][n // 3] = float("inf")
    variants[3][::1001] = float("nan")
    variants[3][n - 1] = float("nan")
    if per == 8:
        patterns = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dt)
        finite = torch.where(patterns.float().abs() < 3.0, patterns, torch.zeros_like(patterns))
        variants[4][:65536] = finite
        variants[4][n - 65536:] = finite
    for i, x in enumerate(variants):
        for value in (QuantValue.Q8S, QuantValue.Q8F):
            call = Call(torch, x, elem, scheme_of(value))
            call.fused()
            call.check((elem.name, i, value.name))


def test_streams_and_graphs():
    """Launches on two streams at once, each with its workspace (their workgroups share the compute units, and none waits for
    one that has not started), and a captured launch replayed on new values."""
    import torch

    n = (80 << 16) * 8
    scheme = scheme_of(QuantValue.Q8S)
    calls = [Call(torch, values(torch, n + 8 * 64 * i, ElemType.BF16, i), ElemType.BF16, scheme) for i in range(4)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(3):
        for i, call in enumerate(calls):
            with torch.cuda.stream(streams[i % 2]):
                call.fused()
    torch.cuda.synchronize()
    for i, call in enumerate(calls):
        call.check(i)
    call, graph = calls[0], torch.cuda.CUDAGraph()
    with torch.cuda.stream(streams[0]):
        with torch.cuda.graph(graph, stream=streams[0]):
            call.fused()
    for seed in (7, 8, 9):
        call.x.copy_(values(torch, n, ElemType.BF16, seed) * (seed - 6))
        call.codes.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        call.check(seed)


@pytest.fixture(scope="module")
def waits():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libcq_resident_test.so"))
    lib.cq_test_resident.argtypes = [ctypes.c_int] + [ctypes.c_void_p] * 5 + [ctypes.c_uint64] * 2 + [ctypes.c_uint32] * 2
    return lib.cq_test_resident


@pytest.mark.parametrize("kind,elem,value,store", [(0, ElemType.BF16, QuantValue.Q8S, QuantStore.U32), (1, ElemType.F32, QuantValue.Q4S, QuantStore.U32),
                                                   (2, ElemType.F16, QuantValue.E4M3, QuantStore.Native)], ids=["bf16-q8", "f32-q4", "f16-e4m3"])
def test_workgroups_that_work_out_the_shares_of_others(waits, kind, elem, value, store):
    """No grace: shares that have not started when a workgroup has read its own; no patience: every share that has not arrived.  Numbered
    launches and ones with slots in the workspace, of a few, some and many steps, beyond what the chip holds, with elements
    behind the last chunk."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    for chunks in (9 * 512, 100 * 512 + 8, 2 * ROUND, 5 * ROUND + 4, 20 * ROUND + 4, 66 * ROUND + 516):
        n = chunks * per + (3 if store == QuantStore.Native else 0)
        call = Call(torch, values(torch, n, elem, chunks), elem, scheme_of(value, store))
        call.x[n - 1] = -0.75
        for grace, patience in ((0, 1024), (0, 0), (8, 1024)):
            for slots in (None, call.ws.data_ptr()):
                call.codes.zero_()
                call.scale.fill_(-1.0)
                rc = waits(kind, torch.cuda.current_stream().cuda_stream, call.x.data_ptr(), call.codes.data_ptr(), call.scale.data_ptr(), slots,
                           chunks, n, grace, patience)
                assert rc == 0
                if store == QuantStore.Native:  # the bytes behind the last chunk are another kernel's
                    tail = slice(chunks * per, n)
                    assert not call.codes[tail].any()
                    given = call.scale.to(call.x.dtype)
                    qz.launch_ref(ComputeClient.current(), H(call.x[tail]), H(call.codes[tail]), H(given), H(torch.empty_like(call.scale)), call.scheme, elem)
                call.check((chunks, grace, patience, slots is None))


def one_read(call):
    """Whether a launch leaves the workspace alone: two passes write the workgroups' abs-maxima to it."""
    call.ws.fill_(0x5A)
    call.fused()
    call.torch.cuda.synchronize()
    return bool((call.ws == 0x5A).all())


def test_sizes_of_one_read():
    """Both sides of every line between one read and two passes (their results are the same)."""
    import torch

    def reads_once(elem, value, chunks):
        per = 4 if elem == ElemType.F32 else 8
        call = Call(torch, torch.empty(chunks * per, dtype=dtype_of(torch, elem), device="cuda").normal_(), elem, scheme_of(value))
        call.fused()  # from here on the stream is one of the last two
        return one_read(call)

    mib = 1 << 16
    assert reads_once(ElemType.BF16, QuantValue.Q8S, 4) and reads_once(ElemType.BF16, QuantValue.Q8S, 16 * mib)
    assert not reads_once(ElemType.BF16, QuantValue.Q8S, 16 * mib + 4) and not reads_once(ElemType.BF16, QuantValue.Q8S, 48 * mib - 4)
    assert reads_once(ElemType.BF16, QuantValue.Q8S, 48 * mib) and reads_once(ElemType.F16, QuantValue.Q8S, 384 * mib)
    assert not reads_once(ElemType.BF16, QuantValue.Q8S, 384 * mib + 4) and reads_once(ElemType.F32, QuantValue.Q8S, 384 * mib + 4)
    assert not reads_once(ElemType.BF16, QuantValue.Q4S, 56 * mib - 4) and reads_once(ElemType.BF16, QuantValue.Q4S, 56 * mib)
    assert not reads_once(ElemType.F16, QuantValue.Q2S, 128 * mib - 4) and reads_once(ElemType.F16, QuantValue.Q2S, 128 * mib)
    assert reads_once(ElemType.BF16, QuantValue.Q4S, 768 * mib) and not reads_once(ElemType.F32, QuantValue.Q4S, 768 * mib + 8)


def test_two_passes_on_a_third_stream_and_on_part_of_the_compute_units():
    import torch

    call = Call(torch, values(torch, (48 << 16) * 8, ElemType.BF16, 1), ElemType.BF16, scheme_of(QuantValue.Q8S))
    streams = [torch.cuda.Stream() for _ in range(3)]

    def on(i):
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[i]):
            return one_read(call)

    on(0), on(1)
    assert [on(i) for i in (0, 1, 0, 1)] == [True] * 4
    assert not on(2) and on(2) and on(1) and not on(0)
    call.check("streams")

    hip = ctypes.CDLL("libamdhip64.so")
    half, stream = (ctypes.c_uint32 * 8)(*[0xffffffff] * 4 + [0] * 4), ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(stream), 8, half) == 0
    masked = torch.cuda.ExternalStream(stream.value)
    for _ in range(2):
        torch.cuda.synchronize()
        with torch.cuda.stream(masked):
            assert not one_read(call)
    call.check("mask")
    small = Call(torch, values(torch, 8 * 512 * 100, ElemType.BF16, 2), ElemType.BF16, scheme_of(QuantValue.Q8S))
    torch.cuda.synchronize()
    with torch.cuda.stream(masked):
        assert one_read(small)
    small.check("mask, small")


def test_captured_launches_on_any_stream():
    """The fourth stream's capture is one read too (its slots are the workspace's): the share of the largest value is the slot that
    holds it after a replay."""
    import torch

    call = Call(torch, values(torch, (72 << 16) * 8, ElemType.BF16, 3), ElemType.BF16, scheme_of(QuantValue.Q8S))
    call.x[8 * 512 * 37 + 5] = -0.75  # step 37: the share of workgroup 37
    graphs = []
    for _ in range(4):
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call.fused()
        graphs.append(graph)
    for graph in graphs:
        call.codes.zero_()
        call.ws.fill_(0x5A)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        slots = call.ws.view(torch.float32)
        assert slots[37].item() == 0.75 and slots.argmax().item() == 37
        call.check("captured")
