"""A tensor whose byte offsets do not fit 32 bits (bf16 [36864, 65536]: 2.4 G elements, 4.8 GB).

Every kernel family has to carry 64-bit offsets through: the flat kernels (contiguous), the row
kernels (pitched rows), the transposed kernels, the reductions.  The CPU oracle checks bands of rows
at the start, in the middle and at the very end (beyond 4 GiB); whole-tensor checks are equalities
between independent GPU paths and torch reductions."""
import numpy as np
import pytest

from cubek_amd import (ComputeClient, ElemType, QuantLevel, QuantScheme, QuantValue, TensorHandleRef)
from cubek_amd import dequantize as dq
from cubek_amd import quantize as qz
from cubek_amd import reduce as cq_reduce

pytestmark = pytest.mark.gpu
ROWS, COLS, BLOCK = 36864, 65536, 32
ELEM = ElemType.BF16


def bits_of(t):
    import torch

    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def test_offsets_beyond_32_bits(oracle):
    import torch

    client = ComputeClient.current()
    h = TensorHandleRef.from_torch
    scheme = QuantScheme.default().with_value(QuantValue.Q4S).with_level(QuantLevel.block([BLOCK]))
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    x = torch.empty((ROWS, COLS), dtype=torch.bfloat16, device="cuda")
    for r0 in range(0, ROWS, 2048):  # chunked: bounds the f32 temporary
        x[r0:r0 + 2048] = torch.randn((2048, COLS), generator=g, device="cuda").mul_(0.03).to(torch.bfloat16)
    assert x.numel() * 2 > 1 << 32

    print("contiguous: fused dynamic quantize, two-step, dequantize", flush=True)
    codes = torch.zeros((ROWS, COLS // 8), dtype=torch.int32, device="cuda")
    scales = torch.zeros((ROWS, COLS // BLOCK), dtype=torch.float32, device="cuda")
    qz.launch_dynamic(client, h(x), h(codes), h(scales), scheme, ELEM)
    in_scales = torch.zeros((ROWS, COLS // BLOCK), dtype=torch.bfloat16, device="cuda")
    qz.compute_scales(client, h(x), h(in_scales), scheme, ELEM)
    codes2 = torch.zeros_like(codes)
    scales2 = torch.zeros_like(scales)
    qz.launch_ref(client, h(x), h(codes2), h(in_scales), h(scales2), scheme, ELEM)
    y = torch.zeros_like(x)
    dq.launch_ref(client, h(codes), h(y), h(scales), scheme, ELEM)
    torch.cuda.synchronize()
    assert torch.equal(codes, codes2) and torch.equal(scales, scales2)
    del codes2, scales2

    band = 16
    refs = {}
    for r0 in (0, ROWS // 2, ROWS - band):
        xs = bits_of(x[r0:r0 + band])
        s_ref = oracle.compute_scales(xs, ELEM, (band, COLS), scheme)
        w_ref, os_ref = oracle.quantize(xs, ELEM, (band, COLS), s_ref, scheme, threads=8)
        y_ref = oracle.dequantize(w_ref, (band, COLS), os_ref, ELEM, scheme)
        refs[r0] = (w_ref, os_ref, y_ref)
        assert np.array_equal(codes[r0:r0 + band].cpu().numpy().view(np.uint32), w_ref), r0
        assert np.array_equal(scales[r0:r0 + band].cpu().numpy().reshape(-1), os_ref.reshape(-1)), r0
        assert np.array_equal(bits_of(y[r0:r0 + band]).reshape(-1), y_ref.reshape(-1)), r0

    print("reductions against torch", flush=True)
    for axis in (0, 1):
        out = torch.zeros((1, COLS) if axis == 0 else (ROWS, 1), dtype=torch.bfloat16, device="cuda")
        nbytes = cq_reduce.workspace_bytes(h(x), axis, ELEM)
        ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
        cq_reduce.max_abs(client, h(x), h(out), axis, ELEM, ws.data_ptr() if nbytes else 0, nbytes)
        torch.cuda.synchronize()
        want = torch.stack([x[r0:r0 + 4096].abs().amax(dim=axis, keepdim=True) for r0 in range(0, ROWS, 4096)])
        want = want.amax(dim=0) if axis == 0 else want.reshape(ROWS, 1)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), axis
        del out, ws, want

    print("pitched rows (row kernels)", flush=True)
    pc = COLS - 64  # the view [ROWS, COLS - 64] of the same buffer: rows keep their pitch
    hx = TensorHandleRef(h(x).handle, (ROWS, pc), (COLS, 1), 2)
    pcodes = torch.zeros((ROWS, pc // 8), dtype=torch.int32, device="cuda")
    pscales = torch.zeros((ROWS, pc // BLOCK), dtype=torch.float32, device="cuda")
    qz.launch_dynamic(client, hx, h(pcodes), h(pscales), scheme, ELEM)
    py = torch.full((ROWS, COLS), 7.0, dtype=torch.bfloat16, device="cuda")
    dq.launch_ref(client, h(pcodes), TensorHandleRef(h(py).handle, (ROWS, pc), (COLS, 1), 2), h(pscales), scheme, ELEM)
    torch.cuda.synchronize()
    assert torch.equal(pcodes, codes[:, :pc // 8]) and torch.equal(pscales, scales[:, :pc // BLOCK])
    assert torch.equal(py[:, :pc].view(torch.int16), y[:, :pc].view(torch.int16))
    assert bool((py[:, pc:] == 7.0).all())
    del pcodes, pscales, py

    print("transposed floats", flush=True)
    xt = torch.empty((COLS, ROWS), dtype=torch.bfloat16, device="cuda")
    for c0 in range(0, COLS, 8192):
        xt[c0:c0 + 8192] = x[:, c0:c0 + 8192].t()
    hxt = TensorHandleRef(h(xt).handle, (ROWS, COLS), (1, ROWS), 2)
    tcodes = torch.zeros_like(codes)
    tscales = torch.zeros_like(scales)
    qz.launch_dynamic(client, hxt, h(tcodes), h(tscales), scheme, ELEM)
    torch.cuda.synchronize()
    assert torch.equal(tcodes, codes) and torch.equal(tscales, scales)
    del tcodes, tscales
    xt.fill_(7.0)
    dq.launch_ref(client, h(codes), hxt, h(scales), scheme, ELEM)
    torch.cuda.synchronize()
    for c0 in range(0, COLS, 8192):
        assert torch.equal(xt[c0:c0 + 8192].t().contiguous().view(torch.int16),
                           y[:, c0:c0 + 8192].contiguous().view(torch.int16)), c0


@pytest.mark.parametrize("rows,cols,axis_last", [((1 << 29) + 3, 9, True), (3, ((1 << 32) + 40) // 3, False)], ids=["short_rows", "many_outputs"])
def test_more_lanes_than_a_launch_counts(rows, cols, axis_last):
    """2^29 rows that would have eight lanes each; 2^32 outputs that have a lane each (a tensor whose rows lie two elements apart)."""
    import torch

    client = ComputeClient.current()
    if axis_last:
        x = torch.zeros((rows, cols), device="cuda")
        x[-1, 4], x[5, 8] = -3.0, 2.0
        out = torch.full((rows, 1), -1.0, device="cuda")
        h_x, axis = TensorHandleRef.from_torch(x), 1
    else:
        store = torch.zeros((2 * cols * rows,), dtype=torch.bfloat16, device="cuda")
        x = store.view(1, rows, cols, 2)[..., 0]
        x[0, -1, -1], x[0, 0, 5] = -3.0, 2.0
        out = torch.full((1, rows, cols), -1.0, dtype=torch.bfloat16, device="cuda")
        h_x, axis = TensorHandleRef.from_torch(x), 0
    cq_reduce.max_abs(client, h_x, TensorHandleRef.from_torch(out), axis, ElemType.F32 if axis_last else ElemType.BF16)
    torch.cuda.synchronize()
    flat = out.view(-1)
    assert flat[-1].item() == 3.0 and flat[5].item() == 2.0
    flat[-1] = flat[5] = 0.0
    for begin in range(0, flat.numel(), 1 << 30):
        assert not flat[begin:begin + (1 << 30)].any(), begin


def test_per_element_kernels_of_more_lanes_than_a_launch_counts():
    """2^32 bytes that have a lane each: quantized from and dequantized into floats two elements apart, and copied out of rows of an
    odd pitch."""
    import torch

    from cubek_amd import QuantParam, QuantStore, _ffi, contiguous

    client, h = ComputeClient.current(), TensorHandleRef.from_torch
    rows, cols = 3, ((1 << 32) + 100) // 3
    floats = torch.zeros((rows, cols, 2), dtype=torch.bfloat16, device="cuda")[..., 0]
    ends = [(0, 5, 7), (1, 11, -9), (2, cols - 1, 3)]
    for r, c, v in ends:
        floats[r, c] = v * 0.5
    scheme = QuantScheme.default().with_value(QuantValue.Q8S).with_store(QuantStore.Native).with_param(QuantParam.F32)
    given = torch.full((1,), 0.5, dtype=torch.bfloat16, device="cuda")
    scale = torch.zeros((1,), device="cuda")
    codes = torch.full((rows, cols), 99, dtype=torch.uint8, device="cuda")
    assert _ffi.plan_kind(_ffi.OP_QUANTIZE, h(floats), h(codes), h(given), h(scale), scheme, ELEM) == "per_element"
    qz.launch_ref(client, h(floats), h(codes), h(given), h(scale), scheme, ELEM)

    def check(t, back):
        torch.cuda.synchronize()
        for r, c, v in ends:
            assert back(t[r, c].item()) == v, (r, c)
            t[r, c] = 0
        for row in t:
            for begin in range(0, cols, 1 << 28):
                assert not row[begin:begin + (1 << 28)].any(), begin
        for r, c, v in ends:
            t[r, c] = v % 256 if t.dtype == torch.uint8 else v * 0.5

    signed = lambda b: b - 256 if b > 127 else b  # noqa: E731
    check(codes, signed)
    floats.fill_(4.0)
    assert _ffi.plan_kind(_ffi.OP_DEQUANTIZE, h(floats), h(codes), h(scale), None, scheme, ELEM) == "per_element"
    dq.launch_ref(client, h(codes), h(floats), h(scale), scheme, ELEM)
    check(floats, lambda v: v * 2)
    del floats
    pitched = torch.zeros((rows, cols + 1 + cols % 2), dtype=torch.uint8, device="cuda")[:, :cols]
    pitched.copy_(codes)
    codes.fill_(99)
    contiguous.into_contiguous_packed_ref(client, h(pitched), h(codes), (rows, cols), 1)
    check(codes, signed)
