"""Blocks over the last two dimensions, quantized with the scale computed in the launch (quantize_block_tiles_kernel), against the two
calls that share no kernel with it: compute_scales, then quantize with the given scales.  Codes and scales bit for bit."""
import pytest

from cubek_amd import (ComputeClient, ElemType, QuantLevel, QuantParam, QuantScheme, QuantStore, QuantValue, TensorHandleRef, _ffi,
                       quantize)

pytestmark = pytest.mark.gpu
H = TensorHandleRef.from_torch


def types(torch):
    return {ElemType.F32: torch.float32, ElemType.F16: torch.float16, ElemType.BF16: torch.bfloat16,
            QuantParam.F32: torch.float32, QuantParam.F16: torch.float16, QuantParam.BF16: torch.bfloat16}


def compare(torch, x, scheme, elem, shift=0, pitch=0, what=None, tiles=True):
    """`shift`: words (or bytes) in front of the codes, `pitch`: behind each of their rows."""
    t = types(torch)
    packed, blocks = scheme.packed_shape(x.shape), scheme.scales_shape(x.shape)
    kind = torch.uint8 if scheme.store == QuantStore.Native else torch.int32
    n = shift + packed[-1] + pitch
    results = []
    for fused in (True, False):
        buffer = torch.full((*packed[:-1], n), 77, dtype=kind, device="cuda")
        codes = buffer[..., shift:shift + packed[-1]]
        scales = torch.zeros(blocks, dtype=t[scheme.param], device="cuda")
        client = ComputeClient.current()
        if fused:
            if tiles:
                assert _ffi.plan_kind(_ffi.OP_QUANTIZE_DYNAMIC, H(x), H(codes), None, H(scales), scheme, elem) == "blocks", what
            quantize.launch_dynamic(client, H(x), H(codes), H(scales), scheme, elem)
        else:
            given = torch.zeros(blocks, dtype=x.dtype, device="cuda")
            quantize.compute_scales(client, H(x), H(given), scheme, elem)
            quantize.launch_ref(client, H(x), H(codes), H(given), H(scales), scheme, elem)
        results.append((buffer, scales.view(torch.uint8)))
    for got, want in zip(*results):
        assert torch.equal(got, want), what


def values(torch, shape, elem, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(shape, generator=gen, device="cuda") * 0.02
    x *= torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.001, 50.0, 1.0)
    return x.to(types(torch)[elem])


KINDS = [(QuantValue.Q8S, QuantStore.U32), (QuantValue.Q8F, QuantStore.Native), (QuantValue.Q4S, QuantStore.U32), (QuantValue.Q2S, QuantStore.U32),
         (QuantValue.E4M3, QuantStore.Native), (QuantValue.E5M2, QuantStore.Native), (QuantValue.E2M1, QuantStore.Native), (QuantValue.E2M1_OCP, QuantStore.U32)]


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value,store", KINDS, ids=lambda v: v.name)
def test_blocks_and_widths(elem, value, store):
    """Every number of chunks a lane holds; rows of one tile of lanes, of a block more, of several and a cut one."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    for br, bc in ((32, 32), (64, 64), (128, 128), (16, 32), (8, 64), (128, 32), (32, 128), (4, 128)):
        scheme = QuantScheme.default().with_value(value).with_store(store).with_level(QuantLevel.block([br, bc]))
        lanes = max(16, bc // per)
        while br * lanes < 256:
            lanes *= 2
        widths = {lanes * per, lanes * per + bc, 3 * lanes * per + bc}
        for i, cols in enumerate(sorted(widths)):
            x = values(torch, (br * (1 + i), cols), elem, br + cols)
            compare(torch, x, scheme.with_param(QuantParam(i % 3)), elem, what=(br, bc, cols))


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16], ids=lambda e: e.name)
def test_large_launches_of_blocks_of_a_few_rows(elem):
    """Both sides of the size from which their tiles are wider, with a whole and a cut last tile, and without room for wider ones."""
    import torch

    per = 4 if elem == ElemType.F32 else 8
    scheme = QuantScheme.default().with_value(QuantValue.Q8S)
    for br, bc in ((8, 32), (16, 64), (8, 128), (4, 64)):
        for row_chunks in (64, 256, 224):
            rows = -(-(5 << 17) // row_chunks // br) * br
            for n in (rows - br, rows):
                x = values(torch, (n, row_chunks * per), elem, br + n)
                compare(torch, x, scheme.with_level(QuantLevel.block([br, bc])), elem, what=(br, bc, n, row_chunks))
        x = values(torch, (br * (-(-(11 << 20) // 48 // br)), 48 * per), elem, br)
        compare(torch, x, scheme.with_level(QuantLevel.block([br, 16])), elem, what=(br, 16), tiles=False)


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value", [QuantValue.Q8S, QuantValue.Q4S], ids=lambda v: v.name)
def test_layouts(elem, value):
    """A batch of matrices, pitched and permuted floats, codes that start on odd words and in rows of odd pitch."""
    import torch

    for side in (32, 64, 128):
        scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block([side, side]))
        batch = values(torch, (3, 2 * side, 5 * 128), elem, side)
        compare(torch, batch, scheme, elem, what=side)
        compare(torch, batch[:, :, 128:], scheme, elem, what=side)
        compare(torch, batch.transpose(0, 1).contiguous().transpose(0, 1), scheme, elem, what=side)
        for shift, pitch in ((1, 0), (0, 1), (1, 2), (2, 2)):
            compare(torch, batch[1], scheme, elem, shift, pitch, what=(side, shift, pitch))


@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value,store", [(QuantValue.Q8S, QuantStore.U32), (QuantValue.Q4F, QuantStore.U32), (QuantValue.E4M3, QuantStore.Native)],
                         ids=lambda v: v.name)
def test_values_that_divide(elem, value, store):
    """Blocks of zeros, with an infinity, with NaN elements, whose divisor is no ordinary number, and every 16-bit pattern."""
    import torch

    for side in (32, 128):
        scheme = QuantScheme.default().with_value(value).with_store(store).with_level(QuantLevel.block([side, side]))
        x = values(torch, (4 * side, 1024), elem, side)
        x[:side, :side] = 0.0
        x[side + 3, 5] = float("inf")
        x[2 * side:3 * side:7, ::11] = float("nan")
        x[3 * side:, :512] *= 2.0 ** -14 if elem == ElemType.F16 else 2.0 ** -120
        compare(torch, x, scheme, elem, what=side)
        if elem != ElemType.F32:
            patterns = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(x.dtype)
            finite = torch.where(patterns.float().isfinite(), patterns, torch.zeros_like(patterns))
            compare(torch, finite.view(side, -1).contiguous(), scheme, elem, what=side)
            small = torch.where(finite.float().abs() < 3.0, finite, torch.zeros_like(finite))
            compare(torch, small.view(side, -1).contiguous(), scheme, elem, what=side)
