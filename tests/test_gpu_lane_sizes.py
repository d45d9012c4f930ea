"""The lane-wise kernels by the size of a launch: one chunk per lane below small_lane_chunks() (cq_launch_rules.hpp), several from
there on.  The other tests hold small launches against the oracle; here a large launch has to give, bit for bit, what small
ones give on its parts, and small ones what the kernels over contiguous runs give."""
import pytest

from cubek_amd import (ComputeClient, ElemType, QuantLevel, QuantParam, QuantScheme, QuantStore, QuantValue, TensorHandleRef, dequantize,
                       quantize)

pytestmark = pytest.mark.gpu
H = TensorHandleRef.from_torch
LINE = 3 << 18  # chunks of 16 bytes


def types(torch):
    return {ElemType.F32: torch.float32, ElemType.F16: torch.float16, ElemType.BF16: torch.bfloat16,
            QuantParam.F32: torch.float32, QuantParam.F16: torch.float16, QuantParam.BF16: torch.bfloat16}


def call(torch, x, scheme, elem, codes, scales, given=None):
    """The codes, scales and restored values of `x`, whose buffers `codes` and `scales` may be views."""
    y = torch.zeros(x.shape, dtype=x.dtype, device="cuda")
    client = ComputeClient.current()
    if given is None:
        quantize.launch_dynamic(client, H(x), H(codes), H(scales), scheme, elem)
    else:
        quantize.compute_scales(client, H(x), H(given), scheme, elem)
        quantize.launch_ref(client, H(x), H(codes), H(given), H(scales), scheme, elem)
    dequantize.launch_ref(client, H(codes), H(y), H(scales), scheme, elem)
    return y


CASES = [(ElemType.F16, QuantValue.Q8S, QuantStore.Native, QuantParam.F16, 128, 32), (ElemType.BF16, QuantValue.Q4S, QuantStore.U32, QuantParam.F32, 80, 16),
         (ElemType.BF16, QuantValue.E4M3, QuantStore.Native, QuantParam.BF16, 96, 32), (ElemType.F32, QuantValue.Q2S, QuantStore.U32, QuantParam.F32, 128, 64),
         (ElemType.F16, QuantValue.E2M1, QuantStore.U32, QuantParam.F32, 256, 128)]


@pytest.mark.parametrize("given", [False, True], ids=["dynamic", "given"])
@pytest.mark.parametrize("elem,value,store,param,head_dim,block", CASES, ids=lambda v: getattr(v, "name", str(v)))
def test_permuted_views(elem, value, store, param, head_dim, block, given):
    """[batch, tokens, heads, head_dim] read as [batch, heads, tokens, head_dim] into a slice of a longer buffer: launches on
    both sides of the line, against one launch per batch entry (three tokens: a walk per lane; many: from the tile's first row)."""
    import torch

    t = types(torch)
    scheme = QuantScheme.default().with_value(value).with_store(store).with_param(param).with_level(QuantLevel.block([block]))
    row = head_dim * (4 if elem == ElemType.F32 else 2) // 16
    heads = 5
    for tokens, batch in ((3, LINE // (row * heads * 3) + 1), (701, LINE // (row * heads * 701) + 1), (3, 7), (67, 2), (1, 1)):
        gen = torch.Generator(device="cuda").manual_seed(tokens * 7 + batch)
        x = torch.randn((batch, tokens, heads, head_dim), generator=gen, device="cuda").to(t[elem]).permute(0, 2, 1, 3)
        kind = torch.uint8 if store == QuantStore.Native else torch.int32
        results = []
        for whole in (True, False):
            codes = torch.zeros(scheme.packed_shape((batch, heads, tokens + 5, head_dim)), dtype=kind, device="cuda")
            scales = torch.zeros(scheme.scales_shape((batch, heads, tokens + 5, head_dim)), dtype=t[param], device="cuda")
            c, s = codes[:, :, 5:], scales[:, :, 5:]
            g = torch.zeros(s.shape, dtype=t[elem], device="cuda") if given else None
            if whole:
                y = call(torch, x, scheme, elem, c, s, g)
            else:
                parts = min(batch, 8)  # up to eight launches, each below the line
                bounds = [batch * i // parts for i in range(parts + 1)]
                y = torch.cat([call(torch, x[a:b], scheme, elem, c[a:b], s[a:b], None if g is None else g[a:b]) for a, b in zip(bounds, bounds[1:])])
            results.append((codes, scales, y))
        for got, want in zip(*results):
            assert torch.equal(got, want), (tokens, batch)
        # the same values in a contiguous tensor
        codes = torch.zeros(scheme.packed_shape(x.shape), dtype=kind, device="cuda")
        scales = torch.zeros(scheme.scales_shape(x.shape), dtype=t[param], device="cuda")
        y = call(torch, x.contiguous(), scheme, elem, codes, scales, torch.zeros(scales.shape, dtype=t[elem], device="cuda") if given else None)
        assert torch.equal(codes, results[0][0][:, :, 5:]) and torch.equal(scales, results[0][1][:, :, 5:]) and torch.equal(y, results[0][2])


@pytest.mark.parametrize("given", [False, True], ids=["dynamic", "given"])
@pytest.mark.parametrize("elem", [ElemType.F32, ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
@pytest.mark.parametrize("value,block", [(QuantValue.Q8S, 24), (QuantValue.Q8S, 16), (QuantValue.Q4S, 16), (QuantValue.Q4S, 40), (QuantValue.Q2S, 16)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_contiguous_runs(elem, value, block, given):
    """Runs whose blocks have no kernel over whole tiles: around a tile of one step and the line, against halves."""
    import torch

    t = types(torch)
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block([block]))
    per = 4 if elem == ElemType.F32 else 8
    unit = block * scheme.num_quants()
    for chunks in (1, 255, 256, 257, 5 * 256 + 3, LINE - 1, LINE, LINE + 300):
        n = max(2, chunks * per // unit) * unit
        x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(chunks), device="cuda").to(t[elem])
        results = []
        for cuts in ((0, n), (0, n // unit // 2 * unit, n)):
            codes = torch.zeros(scheme.packed_shape((n,)), dtype=torch.int32, device="cuda")
            scales = torch.zeros(scheme.scales_shape((n,)), dtype=torch.float32, device="cuda")
            g = torch.zeros(scales.shape, dtype=t[elem], device="cuda") if given else None
            nq = scheme.num_quants()
            y = torch.cat([call(torch, x[a:b], scheme, elem, codes[a // nq:b // nq], scales[a // block:b // block],
                                None if g is None else g[a // block:b // block]) for a, b in zip(cuts, cuts[1:])])
            results.append((codes, scales, y))
        for got, want in zip(*results):
            assert torch.equal(got, want), chunks
