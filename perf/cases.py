"""The work that programs built on this library give it, as cases that can be timed: what each case stands for is said
at `listed()`; `draw()` gives further cases of the same kinds over the same ranges of sizes, types and options.

A case is a dict of plain values.  `prepare()` makes what the program holds before the call (tensors, handles, the
workspace), `run()` makes the calls of one pass through the public entry points of `cubek_amd`;
`exact()` says in plain torch what the results stand for.
"""
import math

import torch

from cubek_amd import (ComputeClient, ElemType, QuantLevel, QuantParam, QuantScheme, QuantStore, QuantValue,
                       TensorHandleRef, contiguous, dequantize, matvec, quantize, reduce)

_TORCH = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}
_BYTES = {"F32": 4, "F16": 2, "BF16": 2}
_BITS = {"Q8S": 8, "Q8F": 8, "E4M3": 8, "E5M2": 8, "Q4S": 4, "Q4F": 4, "E2M1": 4, "Q2S": 2, "Q2F": 2}


def listed():
    return [
        # configuration 1 of the benchmark: one scale for a small f32 tensor, where launches and latency count
        dict(name="encode_tensor_f32_small", kind="encode_tensor", rows=1024, cols=1024, elem="F32", value="Q8S",
             store="U32", dist="normal1"),
        # a decode step appends the new tokens of a batch of 16 to a quantized key cache and reads them back: the
        # smallest calls there are
        dict(name="cache_append", kind="cache", batch=16, heads=8, tokens=3, head_dim=128, elem="F16", value="Q8S",
             store="Native", param="F16", block=32),
        # configuration 2: activations with outliers, quantized and restored
        dict(name="activations_q8", kind="round_trip", rows=4096, cols=4096, elem="BF16", value="Q8S", store="U32",
             param="F32", block=32, dist="outliers"),
        # configuration 3's weight-load path: a stored 4-bit FFN weight becomes bf16 again
        dict(name="load_q4_weight", kind="load", rows=14336, cols=4096, elem="BF16", value="Q4S", store="U32",
             param="F32", block=32, dist="normal"),
        # configuration 4, by the crate's own interface: scales first, quantize with given scales, dequantize
        dict(name="given_scales_q2", kind="given", rows=8192, cols=8192, elem="F32", value="Q2S", store="U32",
             param="F32", block=64, dist="laplace"),
        # configuration 5: the largest weight, e2m1 codes, quantized and restored
        dict(name="largest_e2m1", kind="round_trip", rows=28672, cols=8192, elem="BF16", value="E2M1", store="U32",
             param="F32", block=32, dist="heavy_tail"),
        # the scheme's default level on a whole FFN weight: one scale per tensor, q8
        dict(name="encode_tensor_weight", kind="encode_tensor", rows=14336, cols=4096, elem="BF16", value="Q8S",
             store="U32", dist="normal"),
        # fp8 weights with a scale per 128 x 128 block, the native byte store
        dict(name="fp8_blocks", kind="round_trip", rows=14336, cols=4096, elem="BF16", value="E4M3", store="Native",
             param="F32", block=128, block_rows=128, dist="normal"),
        # calibration: the abs-max of every channel over a ragged batch of tokens
        dict(name="channel_maxima", kind="maxima", rows=4093, cols=11008, axis=0, elem="BF16"),
        # a weight that another program stored transposed, quantized along its rows and re-packed for a product that
        # wants the codes along the other dimension
        dict(name="transposed_weight", kind="relayout", rows=14336, cols=4096, elem="BF16", value="Q4S", block=32),
        # one token of decoding: the matrix-vector product straight from the largest 4-bit weight
        dict(name="decode_one", kind="product", rows=28672, cols=8192, vectors=1, elem="BF16", value="Q4S", store="U32",
             param="F32", block=32),
        # a decode step of a batch of 8 over an FFN weight, 4-bit codes in groups of 128 with f16 scales
        dict(name="decode_batch", kind="product", rows=14336, cols=4096, vectors=8, elem="F16", value="Q4S", store="U32",
             param="F16", block=128),
    ]


def _between(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _matrix(rng, low, high, unit, max_cols=32768):
    """Rows and columns of a matrix of about low .. high elements; columns a multiple of `unit`, odd multiples and odd
    rows as likely as others."""
    n = _between(rng, low, high)
    cols = unit * _between(rng, max(1, 256 // unit), max(1, min(max_cols, max(256, n // 2)) // unit))
    return max(1, n // cols), cols


def draw(rng):
    most = work(listed()[5])["bytes"]
    while True:
        case = _draw_one(rng)
        if work(case)["bytes"] <= most:
            return case


def _draw_one(rng):
    kind = rng.choice(["encode_tensor", "cache", "round_trip", "load", "given", "maxima", "relayout", "product"])
    elem = rng.choice(["F32", "BF16", "BF16", "F16"])
    if kind == "encode_tensor":
        store = rng.choice(["U32", "U32", "Native"])
        value = rng.choice(["Q8S", "Q8F", "Q4S"] if store == "U32" else ["Q8S", "E4M3"])
        rows, cols = _matrix(rng, 1 << 14, 1 << 27, 32 // _BITS[value] if store == "U32" else 1)
        return dict(kind=kind, rows=rows, cols=cols, elem=elem, value=value, store=store, dist="normal")
    if kind == "cache":
        elem = rng.choice(["BF16", "F16"])
        head_dim, block = rng.choice([(64, 32), (80, 16), (96, 32), (128, 32), (128, 128), (256, 64)])
        value, store = rng.choice([("Q8S", "Native"), ("Q8S", "U32"), ("Q4S", "U32"), ("E4M3", "Native")])
        return dict(kind=kind, batch=_between(rng, 1, 32), heads=rng.choice([1, 4, 5, 8, 32]), tokens=_between(rng, 1, 4096),
                    head_dim=head_dim, elem=elem, value=value, store=store, param=rng.choice(["F32", elem]), block=block)
    if kind == "maxima":
        rows, cols = _matrix(rng, 1 << 16, 1 << 27, rng.choice([1, 8, 32]))
        return dict(kind=kind, rows=rows, cols=cols, axis=rng.choice([0, 1]), elem=elem)
    if kind == "relayout":
        block = rng.choice([32, 64, 128])
        value = rng.choice(["Q4S", "E2M1", "Q8S"])
        n = _between(rng, 1 << 18, 1 << 27)
        cols = block * _between(rng, 256 // block, 16384 // block)
        return dict(kind=kind, rows=32 * max(1, n // cols // 32), cols=cols, elem=rng.choice(["BF16", "F16"]), value=value, block=block)
    if kind == "product":
        elem = rng.choice(["BF16", "BF16", "F16"])
        vectors = rng.choice([1, 1, 2, 3, 4, 5, 7, 8, 12, 16])
        value, store, block, block_rows = rng.choice([("Q4S", "U32", 32, 1), ("Q4S", "U32", 64, 1), ("Q4S", "U32", 128, 1),
                                                      ("Q8S", "U32", 32, 1), ("E2M1", "U32", 32, 1), ("E2M1", "Native", 32, 1),
                                                      ("E4M3", "Native", 128, 128)])
        cols = max(block, 32) * _between(rng, 1024 // max(block, 32), 28672 // max(block, 32))
        rows = block_rows * _between(rng, 1024 // block_rows, 28672 // block_rows)
        return dict(kind=kind, rows=rows, cols=cols, vectors=vectors, elem=elem, value=value, store=store,
                    param=rng.choice(["F32", elem]), block=block, block_rows=block_rows)
    if kind == "round_trip" and rng.random() < 0.3:  # blocks over both dimensions
        side = rng.choice([32, 64, 128])
        cols = side * _between(rng, max(1, 256 // side), 16384 // side)
        rows = side * max(1, _between(rng, 1 << 16, 1 << 27) // cols // side)
        value, store = rng.choice([("E4M3", "Native"), ("Q8S", "Native"), ("Q8S", "U32"), ("Q4S", "U32")])
        return dict(kind=kind, rows=rows, cols=cols, elem=elem, value=value, store=store, param="F32", block=side,
                    block_rows=side, dist="normal")
    value, store = rng.choice([("Q8S", "U32"), ("Q8F", "U32"), ("Q4S", "U32"), ("Q4F", "U32"), ("E2M1", "U32"), ("Q2S", "U32"),
                               ("Q8S", "Native"), ("E4M3", "Native"), ("E5M2", "Native"), ("E2M1", "Native")])
    block = rng.choice([16, 24, 32, 32, 64, 128]) if _BITS[value] > 2 else rng.choice([32, 64, 128])
    rows, cols = _matrix(rng, 1 << 14, 1 << 28, block)
    return dict(kind=kind, rows=rows, cols=cols, elem=elem, value=value, store=store, param=rng.choice(["F32", "F32", elem]),
                block=block, dist=rng.choice(["normal", "outliers", "laplace", "heavy_tail"]))


def _scheme(case):
    block, block_rows = case.get("block", 0), case.get("block_rows", 1)
    level = QuantLevel.Tensor if not block else QuantLevel.block([block_rows, block] if block_rows > 1 else [block])
    return (QuantScheme.default().with_value(QuantValue[case["value"]]).with_level(level)
            .with_store(QuantStore[case.get("store", "U32")]).with_param(QuantParam[case.get("param", "F32")]))


def _values(gen, shape, dist, dtype):
    """Seeded values of a distribution: unit normal, weights of deviation 0.02 (also with one in a thousand fifty times
    as large, or one in a hundred from Student's t with three degrees of freedom), or Laplace of scale 0.01."""
    x = torch.randn(shape, generator=gen, device="cuda")
    if dist == "normal1":
        return x.to(dtype)
    if dist == "laplace":
        u = torch.rand(shape, generator=gen, device="cuda").clamp_(min=2e-7)
        return torch.copysign(u.log_().mul_(-0.01), x).to(dtype)
    x.mul_(0.02)
    if dist == "outliers":
        x.mul_(torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.001, 50.0, 1.0))
    elif dist == "heavy_tail":
        tail = torch.rand(shape, generator=gen, device="cuda") < 0.01
        chi2 = torch.randn((3,) + tuple(shape[-1:]), generator=gen, device="cuda").square_().mean(0)  # a column's own divisor
        x = torch.where(tail, x / chi2.sqrt_().clamp_(min=0.05), x)
    return x.to(dtype)


def _stored(scheme, shape):
    """An empty stored tensor and an empty scale tensor for floats of `shape`."""
    native = scheme.store == QuantStore.Native
    codes = torch.empty(scheme.packed_shape(shape), dtype=torch.uint8 if native else torch.int32, device="cuda")
    scales = torch.empty(scheme.scales_shape(shape), dtype=_TORCH[scheme.param.name], device="cuda")
    return codes, scales


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    client = ComputeClient.current()
    h = TensorHandleRef.from_torch
    kind, elem = case["kind"], ElemType[case["elem"]]
    dtype = _TORCH[case["elem"]]
    state = dict(case=case, client=client, elem=elem)

    def keep(**tensors):
        for name, t in tensors.items():
            state[name] = t
            state["h_" + name] = h(t)

    if kind == "maxima":
        x = _values(gen, (case["rows"], case["cols"]), "outliers", dtype)
        axis = case["axis"]
        keep(x=x, maxima=torch.empty((1, case["cols"]) if axis == 0 else (case["rows"], 1), dtype=dtype, device="cuda"))
        state["workspace_bytes"] = reduce.workspace_bytes(state["h_x"], axis, elem)
        state["workspace"] = torch.empty(max(256, state["workspace_bytes"]), dtype=torch.uint8, device="cuda")
        return state

    scheme = state["scheme"] = _scheme(case)
    if kind == "cache":
        # the new tokens lie [batch, tokens, heads, head_dim]; the cache holds [batch, heads, capacity, head_dim]
        b, nh, s, d = case["batch"], case["heads"], case["tokens"], case["head_dim"]
        capacity = (s + 63) // 64 * 64
        x = _values(gen, (b, s, nh, d), "normal1", dtype)
        codes, scales = _stored(scheme, (b, nh, capacity, d))
        state["buffers"] = (x, codes, scales)
        keep(x=x.permute(0, 2, 1, 3), codes=codes[:, :, capacity - s:], scales=scales[:, :, capacity - s:],
             y=torch.empty((b, nh, s, d), dtype=dtype, device="cuda"))
        return state

    shape = (case["rows"], case["cols"])
    if kind == "relayout":  # stored [cols, rows]: the view [rows, cols] has its rows strided
        x = _values(gen, (shape[1], shape[0]), "normal", dtype).t()
    elif kind == "product":
        x = _values(gen, shape, "normal", dtype)
    else:
        x = _values(gen, shape, case["dist"], dtype)
    codes, scales = _stored(scheme, shape)
    keep(x=x, codes=codes, scales=scales)
    if kind == "encode_tensor":
        state["workspace_bytes"] = quantize.workspace_bytes(scheme, x.numel())
        state["workspace"] = torch.empty(max(256, state["workspace_bytes"]), dtype=torch.uint8, device="cuda")
    elif kind == "given":
        keep(given=torch.empty(scales.shape, dtype=dtype, device="cuda"))
    elif kind == "relayout":
        packing = state["packing"] = scheme.num_quants()
        state["h_packed_rows"] = h(codes.t())  # the codes as [cols / packing, rows], packed along their first dimension
        keep(repacked=torch.empty((shape[1], shape[0] // packing), dtype=codes.dtype, device="cuda"))
    if kind in ("load", "product"):  # the program holds the stored weight, not the floats it was made from
        quantize.launch_dynamic(client, state["h_x"], state["h_codes"], state["h_scales"], scheme, elem)
        torch.cuda.synchronize()
        del state["x"], state["h_x"]
        del x
    if kind == "product":
        v = case["vectors"]
        keep(x=_values(gen, (v, shape[1]) if v > 1 else (shape[1],), "normal1", dtype),
             y=torch.empty((v, shape[0]) if v > 1 else (shape[0],), dtype=dtype, device="cuda"))
    elif kind in ("load", "round_trip", "given"):
        keep(y=torch.empty(shape, dtype=dtype, device="cuda"))
    return state


def run(s):
    kind, client, elem = s["case"]["kind"], s["client"], s["elem"]
    if kind == "maxima":
        reduce.max_abs(client, s["h_x"], s["h_maxima"], s["case"]["axis"], elem, s["workspace"].data_ptr(), s["workspace_bytes"])
        return s["maxima"]
    scheme = s["scheme"]
    if kind == "encode_tensor":
        quantize.launch_dynamic(client, s["h_x"], s["h_codes"], s["h_scales"], scheme, elem, s["workspace"].data_ptr(),
                                s["workspace_bytes"])
        return s["codes"], s["scales"]
    if kind in ("round_trip", "cache"):
        quantize.launch_dynamic(client, s["h_x"], s["h_codes"], s["h_scales"], scheme, elem)
        dequantize.launch_ref(client, s["h_codes"], s["h_y"], s["h_scales"], scheme, elem)
        return s["codes"], s["scales"], s["y"]
    if kind == "load":
        dequantize.launch_ref(client, s["h_codes"], s["h_y"], s["h_scales"], scheme, elem)
        return s["y"]
    if kind == "given":
        quantize.compute_scales(client, s["h_x"], s["h_given"], scheme, elem)
        quantize.launch_ref(client, s["h_x"], s["h_codes"], s["h_given"], s["h_scales"], scheme, elem)
        dequantize.launch_ref(client, s["h_codes"], s["h_y"], s["h_scales"], scheme, elem)
        return s["given"], s["codes"], s["scales"], s["y"]
    if kind == "relayout":
        quantize.launch_dynamic(client, s["h_x"], s["h_codes"], s["h_scales"], scheme, elem)
        contiguous.into_contiguous_packed_ref(client, s["h_packed_rows"], s["h_repacked"], (s["case"]["cols"], s["case"]["rows"]),
                                              s["packing"])
        return s["codes"], s["scales"], s["repacked"]
    matvec.launch_ref(client, s["h_codes"], s["h_scales"], scheme, s["h_x"], s["h_y"], elem, elem)
    return s["y"]


def work(case):
    """Bytes and operations of one pass: every call reads each of its inputs once and writes each of its outputs once."""
    kind, size = case["kind"], _BYTES[case["elem"]]
    if kind == "cache":
        n = case["batch"] * case["heads"] * case["tokens"] * case["head_dim"]
    else:
        n = case["rows"] * case["cols"]
    if kind == "maxima":
        return {"bytes": n * size + (case["cols"] if case["axis"] == 0 else case["rows"]) * size, "flops": n}
    codes = n * _BITS[case["value"]] // 8
    blocks = n // (case["block"] * case.get("block_rows", 1)) if case.get("block") else 1
    scales = blocks * _BYTES[case.get("param", "F32")]
    if kind == "encode_tensor":
        return {"bytes": n * size + codes + scales, "flops": 2 * n}
    if kind in ("round_trip", "cache"):
        return {"bytes": 2 * (n * size + codes + scales), "flops": 3 * n}
    if kind == "load":
        return {"bytes": n * size + codes + scales, "flops": n}
    if kind == "given":  # three calls: floats to scales, floats and scales to codes and scales, codes and scales to floats
        return {"bytes": 3 * n * size + 2 * codes + 2 * blocks * size + 2 * scales, "flops": 3 * n}
    if kind == "relayout":
        return {"bytes": n * size + 3 * codes + scales, "flops": 2 * n}
    v = case["vectors"]
    return {"bytes": codes + scales + v * size * (case["rows"] + case["cols"]), "flops": 2 * n * v}


def tolerance(case):
    """Codes, scales, restored values, maxima and re-packed words are defined to the bit.  A product's sums are rounded once
    from f32 to the 16-bit type of y: against the same product in 64 bits the rounding alone is about 0.0017 (bf16)
    or 0.0002 (f16) of the result."""
    if case["kind"] == "product":
        return {"rel": 0.007 if case["elem"] == "BF16" else 0.0009}
    return "exact"


_RANGE = {"Q8S": (-127, 127), "Q8F": (-128, 127), "Q4S": (-7, 7), "Q4F": (-8, 7), "Q2S": (-1, 1), "Q2F": (-2, 1),
          "E2M1": (-6, 6), "E4M3": (-448, 448), "E5M2": (-57344, 57344)}


def _blocked(x, case):
    """x with every block in one dimension, the last: [scales..., values of a block]."""
    rows, cols = x.shape[-2:]
    block, block_rows = case.get("block", 0), case.get("block_rows", 1)
    if not block:
        return x.reshape(1, -1)
    lead = x.shape[:-2]
    x = x.reshape(*lead, rows // block_rows, block_rows, cols // block, block)
    return x.transpose(-2, -3).reshape(*lead, rows // block_rows, cols // block, block_rows * block)


def _whole(v, shape, case):
    """The reverse of _blocked."""
    block, block_rows = case.get("block", 0), case.get("block_rows", 1)
    if not block:
        return v.reshape(shape)
    rows, cols = shape[-2:]
    v = v.reshape(*shape[:-2], rows // block_rows, cols // block, block_rows, block)
    return v.transpose(-2, -3).reshape(shape)


def _restored(x, case):
    """The scales of a program's floats and the values its codes stand for, both in 64 bits.  The codes are whole numbers by
    a rule in the float type itself (divide, round, clamp), which is followed here in that type."""
    lo, hi = _RANGE[case["value"]]
    param = _TORCH[case.get("param", "F32")]
    v = _blocked(x, case)
    scale = 2.0 * v.abs().amax(-1, keepdim=True).double() / (hi - lo)
    stored = scale.float().to(x.dtype).to(param)
    codes = (v / stored.to(x.dtype)).round_().clamp_(lo, hi).float().nan_to_num_(0.0)
    if case.get("store") == "Native" and case["value"] in ("E4M3", "E5M2"):
        codes = codes.to(torch.float8_e4m3fn if case["value"] == "E4M3" else torch.float8_e5m2).float()
    elif case.get("store") == "Native" and case["value"] == "E2M1":
        codes = torch.where(codes.abs() == 5.0, 4.0 * codes.sign(), codes)  # 5 lies between 4 and 6: to the even code
    weights = codes.double() * stored.to(x.dtype).double()
    return scale.squeeze(-1), _whole(weights, x.shape, case)


def exact(case, seed):
    """What run() returns, in 64 bits by plain torch; None for codes, which are words of bits."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], _TORCH[case["elem"]]
    if kind == "maxima":
        x = _values(gen, (case["rows"], case["cols"]), "outliers", dtype)
        return x.abs().amax(case["axis"], keepdim=True).double()
    if kind == "cache":
        x = _values(gen, (case["batch"], case["tokens"], case["heads"], case["head_dim"]), "normal1", dtype).permute(0, 2, 1, 3)
    elif kind == "relayout":
        x = _values(gen, (case["cols"], case["rows"]), "normal", dtype).t()
    else:
        x = _values(gen, (case["rows"], case["cols"]), "normal" if kind == "product" else case["dist"], dtype)
    scale, restored = _restored(x, case)
    if kind == "encode_tensor":
        return None, scale.reshape(1)
    if kind in ("round_trip", "cache"):
        return None, scale, restored
    if kind == "load":
        return restored
    if kind == "given":
        return scale, None, scale, restored
    if kind == "relayout":
        return None, scale, None
    v = case["vectors"]
    weights = restored.to(dtype)  # a weight enters a product as the value that dequantize stores
    x = _values(gen, (v, case["cols"]) if v > 1 else (case["cols"],), "normal1", dtype).double()
    parts = [x @ weights[r:r + 4096].double().t() for r in range(0, case["rows"], 4096)]
    return torch.cat(parts, dim=-1)
