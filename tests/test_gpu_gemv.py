"""cq_gemv_quantized (y = dequantize(W) @ x from the packed weights) against the GEMV over the ORACLE's
dequantized weights, computed in float64.  Tolerance, stated once: the kernels accumulate in f32, at most
~260 sequential additions per lane followed by a 6-step tree, each rounding 2^-24 relative, so
|y - y_ref| <= 2e-5 * sum|w * x|; an output of a 16-bit type is the f32 sum rounded once (checked bit for
bit against the f32 output)."""
import numpy as np
import pytest

from cubek_amd import (ComputeClient, ElemType, QuantLevel, QuantParam, QuantScheme, QuantStore, QuantValue,
                       TensorHandleRef, _ffi, matvec)

pytestmark = pytest.mark.gpu

CASES = [
    # elem, value, block, param, rows, cols, word pitch (None: contiguous); 16-bit x of 16384 columns and more, and some of f16 and 4 bits, go to the kernel of
    # four rows a wave, the others to the streaming kernel unless noted (test_launch_rules.py says which)
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 1000, 4096, None),
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 77, 2048, None),
    (ElemType.BF16, QuantValue.E2M1, [32], QuantParam.F32, 130, 11008, None),     # last strip partly idle
    (ElemType.F16, QuantValue.Q4F, [32], QuantParam.F32, 333, 8192, None),
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 64, 4096, 520),         # pitched rows of words
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 50, 8448, None),        # four strips and an eighth
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 21, 16480, None),        # a unit behind a step
    (ElemType.BF16, QuantValue.Q4F, [32], QuantParam.F32, 1, 32768, None),        # one row
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 9, 32, None),           # one block per row
    (ElemType.BF16, QuantValue.E2M1_OCP, [32], QuantParam.F32, 37, 2048, None),   # the extension value: e2m1 nibbles in u32 words
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 11, 53248, None),       # x longer than the streaming kernel's LDS
    (ElemType.F16, QuantValue.Q8S, [64], QuantParam.F16, 5, 40000, None),         # ... 8-bit codes
    (ElemType.F16, QuantValue.Q4S, [128], QuantParam.F16, 33, 4224, None),        # four units under one f16 scale
    (ElemType.BF16, QuantValue.Q8S, [32], QuantParam.F32, 45, 2080, None),        # 8-bit codes, two units per block
    (ElemType.BF16, QuantValue.Q4F, [64], QuantParam.BF16, 19, 16448, 2060),      # bf16 scales, pitched
    (ElemType.F16, QuantValue.Q8F, [16], QuantParam.F32, 70, 1040, None),         # 8-bit codes, a scale per unit
    (ElemType.BF16, QuantValue.Q2S, [64], QuantParam.F32, 52, 4160, None),        # 2-bit codes
    (ElemType.F16, QuantValue.Q2F, [128], QuantParam.F16, 17, 8192, None),        # 2-bit codes, two units per block
    (ElemType.BF16, QuantValue.Q4S, [128], QuantParam.F16, 12, 1024, None),       # f16 scales under bf16 x
    (ElemType.F16, QuantValue.Q8S, [64], QuantParam.BF16, 31, 2112, None),        # bf16 scales under f16 x
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.BF16, 100, 1024, None),
    (ElemType.F16, QuantValue.Q8S, [64], QuantParam.F16, 50, 512, None),
    (ElemType.F32, QuantValue.Q2S, [64], QuantParam.F32, 96, 1024, None),          # x in f32: streaming again
    (ElemType.F32, QuantValue.Q4S, [32], QuantParam.F32, 75, 4160, 524),
    (ElemType.F32, QuantValue.Q8F, [16], QuantParam.F32, 31, 17008, None),         # ... rows too long for the LDS
    (ElemType.F32, QuantValue.Q4S, [32], QuantParam.BF16, 20, 1024, None),         # f32 x under bf16 scales: general kernel
    (ElemType.F32, QuantValue.Q8F, None, QuantParam.F32, 33, 260, None),          # general: 260 values are not whole units
    (ElemType.BF16, QuantValue.Q4S, [4, 16], QuantParam.F32, 64, 256, None),      # blocks narrower than a unit
    (ElemType.BF16, QuantValue.Q8S, None, QuantParam.F32, 29, 2064, None),        # streaming again: one scale per tensor
    (ElemType.F16, QuantValue.Q4F, None, QuantParam.F16, 11, 4128, None),
    (ElemType.BF16, QuantValue.Q4S, [6, 64], QuantParam.F32, 66, 4160, None),     # blocks of six rows
    (ElemType.F16, QuantValue.Q8S, [128, 128], QuantParam.F32, 256, 1024, None),  # 128 x 128 weight blocks
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 40, 1056, None),        # cols not a multiple of 64 blocks
]


def _id(c):
    elem, value, block, param, rows, cols, pitch = c
    return f"{elem.name}-{value.name}-{'x'.join(map(str, block)) if block else 'tensor'}-{param.name}-{rows}x{cols}" + \
        ("-pitched" if pitch else "")


def check_case(oracle, case, seed, native=False, vectors=1):
    import torch

    elem, value, block, param, rows, cols, pitch = case
    level = QuantLevel.Tensor if block is None else QuantLevel.block(block)
    scheme = QuantScheme.default().with_value(value).with_level(level).with_param(param)
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rng = np.random.default_rng(seed)
    w32 = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
    w32[rng.random((rows, cols)) < 0.002] *= 20
    wb = oracle.to_bits(w32, elem)
    scales = oracle.compute_scales(wb, elem, (rows, cols), scheme)
    words, out_scale = oracle.quantize(wb, elem, (rows, cols), scales, scheme)
    deq = oracle.from_bits(oracle.dequantize(words, (rows, cols), out_scale, elem, scheme), elem).astype(np.float64)
    xb = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
    x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
    want = x64 @ deq.T           # [vectors, rows]
    mag = np.abs(x64) @ np.abs(deq).T

    nq = scheme.num_quants()
    wpr = cols // nq
    pitch = pitch or wpr
    buf = np.zeros((rows, pitch), np.uint8 if native else np.uint32)  # native: stored elements are bytes
    buf[:, :wpr] = words.reshape(rows, wpr)
    d_words = torch.from_numpy(buf if native else buf.view(np.int32)).cuda()
    to16 = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda() if a.dtype == np.uint16 \
        else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d_scales, d_x = to16(out_scale), to16(xb)
    sshape = (1,) if block is None else tuple(d_scales.shape)
    h_words = TensorHandleRef(d_words.data_ptr(), (rows, wpr), (pitch, 1), 1 if native else 4)
    h_scales = TensorHandleRef(d_scales.data_ptr(), sshape, tuple(d_scales.stride()) if block else (1,),
                               d_scales.element_size())
    # one right-hand side as a vector, several as the rows of a matrix
    h_x = TensorHandleRef.from_torch(d_x) if vectors > 1 else TensorHandleRef.from_torch(d_x[0])
    client = ComputeClient.current()
    y32 = torch.full((vectors, rows), float("nan"), dtype=torch.float32, device="cuda")
    h_y = lambda t: TensorHandleRef.from_torch(t) if vectors > 1 else TensorHandleRef.from_torch(t[0])
    matvec.launch_ref(client, h_words, h_scales, scheme, h_x, h_y(y32), elem, ElemType.F32)
    torch.cuda.synchronize()
    got = y32.cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - want) <= 2e-5 * mag + 1e-30), (case, vectors, float(np.max(np.abs(got - want) / (mag + 1e-30))))
    if elem != ElemType.F32:  # the same sums, rounded once to the 16-bit type
        y16 = torch.zeros((vectors, rows), dtype=torch.int16, device="cuda")
        matvec.launch_ref(client, h_words, h_scales, scheme, h_x, h_y(y16), elem, elem)
        torch.cuda.synchronize()
        assert np.array_equal(y16.cpu().numpy().view(np.uint16).reshape(-1), oracle.to_bits(y32.cpu().numpy().reshape(-1), elem)), \
            (case, vectors)


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_gemv_matches_oracle_dequantized_weights(oracle, case):
    elem, value, block, param, rows, cols, pitch = case
    check_case(oracle, case, rows * 7 + cols)


NATIVE_CASES = [
    # the native store: e4m3 / e5m2 / i8 bytes (16 values per 16-byte unit), e2m1 pairs (32 values)
    (ElemType.BF16, QuantValue.E4M3, [32], QuantParam.F32, 77, 4128, None),
    (ElemType.F16, QuantValue.E4M3, [128, 128], QuantParam.F32, 256, 2048, None),   # 128 x 128 weight blocks
    (ElemType.BF16, QuantValue.E5M2, [16], QuantParam.BF16, 30, 2064, 2096),        # a scale per unit, pitched rows
    (ElemType.F16, QuantValue.E5M2, None, QuantParam.F16, 21, 16400, None),         # per tensor, a unit behind a step
    (ElemType.BF16, QuantValue.E2M1, [32], QuantParam.F32, 53, 8448, None),         # e2m1 pairs, a scale per unit
    (ElemType.F16, QuantValue.E2M1, [64], QuantParam.F16, 18, 1088, None),
    (ElemType.BF16, QuantValue.Q8S, [32], QuantParam.F32, 45, 2080, None),          # i8 bytes: the 8-bit fields
    (ElemType.F16, QuantValue.Q8F, [16], QuantParam.BF16, 9, 16, None),             # one unit per row
    (ElemType.F32, QuantValue.E4M3, [32], QuantParam.F32, 37, 2080, None),          # x in f32
    (ElemType.F32, QuantValue.E2M1, [64], QuantParam.F32, 12, 4160, None),
    (ElemType.BF16, QuantValue.E2M1_OCP, [32], QuantParam.F32, 41, 4160, None),     # the extension value: e2m1 pairs
]


@pytest.mark.parametrize("case", NATIVE_CASES, ids=_id)
def test_gemv_native_store_matches_oracle_dequantized_weights(oracle, case):
    elem, value, block, param, rows, cols, pitch = case
    check_case(oracle, case, rows * 11 + cols, native=True)


# 4-bit fields on blocks of 32 with f32 scales: several vectors at once go to the matrix-core kernel (a last stage cut
# short; rows not a multiple of 16; pitched rows)
MATRIX_CORE_CASES = [
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 64, 4096, None),
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 77, 4224, None),
    (ElemType.F16, QuantValue.Q4F, [32], QuantParam.F32, 333, 8192, None),
    (ElemType.BF16, QuantValue.E2M1, [32], QuantParam.F32, 130, 11008, None),
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 50, 8448, 1060),
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 21, 16512, None),
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 5, 6144, None),
    (ElemType.BF16, QuantValue.Q4F, [32], QuantParam.F32, 1, 4096, None),
]


@pytest.mark.parametrize("vectors", [2, 3, 4, 5, 9])
@pytest.mark.parametrize("case", MATRIX_CORE_CASES, ids=_id)
def test_gemv_on_the_matrix_cores(oracle, case, vectors):
    check_case(oracle, case, 3 + vectors, vectors=vectors)


# Four rows a wave (gemv_quads_kernel): rows that end inside four and workgroups with one more than others, columns that end inside a
# step of sixteen units or a unit behind one, fewer steps than waves share a row and some waves without, more than 64 times four rows to a compute
# unit, blocks over rows, every slot count of x (one, two, four; three vectors in four), x longer than two pieces a thread.  (Tolerance:
# as above; a share's sums are at most as many additions in a row.)
QUADS_CASES = [
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F16, 1, 32, None, 1, False),
    (ElemType.F16, QuantValue.Q4F, [32], QuantParam.F32, 1027, 544, None, 1, False),        # a unit behind a step
    (ElemType.F16, QuantValue.E2M1, [128], QuantParam.F32, 70, 4224, 532, 1, False),        # pitched, shares of unequal steps
    (ElemType.F16, QuantValue.Q4S, [64], QuantParam.BF16, 65541, 64, None, 1, False),       # more workgroups than compute units
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 1026, 28672, None, 1, False),
    (ElemType.BF16, QuantValue.Q8S, [6, 32], QuantParam.F32, 1026, 12800, None, 1, False),  # blocks of six rows
    (ElemType.F16, QuantValue.E4M3, [32], QuantParam.F32, 1030, 16384, None, 1, True),
    (ElemType.BF16, QuantValue.E5M2, None, QuantParam.F32, 2, 16400, None, 1, True),        # one scale
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.BF16, 7, 96, None, 2, False),
    (ElemType.F16, QuantValue.Q8S, [16], QuantParam.F16, 1031, 1296, None, 2, False),       # a scale per unit
    (ElemType.BF16, QuantValue.E2M1, [64], QuantParam.F32, 1050, 8256, None, 3, True),
    (ElemType.BF16, QuantValue.E4M3, [32, 32], QuantParam.F32, 1056, 2080, None, 4, True),
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 4444, 1056, None, 4, False),
    (ElemType.F16, QuantValue.Q4F, [32], QuantParam.F32, 9, 19424, None, 4, False),         # nearly all of the LDS
    (ElemType.F16, QuantValue.Q4F, [32], QuantParam.F32, 9, 20512, None, 4, False),         # ... and more than there is
    (ElemType.F16, QuantValue.Q4S, [64], QuantParam.F16, 1, 2112, None, 1, False),          # one row
    (ElemType.BF16, QuantValue.Q8S, [6, 32], QuantParam.F32, 1026, 16384, None, 1, False),  # blocks of six rows across groups of four
    (ElemType.BF16, QuantValue.E4M3, [128, 128], QuantParam.F32, 1152, 14464, None, 1, True),
    (ElemType.BF16, QuantValue.E2M1, [32], QuantParam.F32, 1030, 28672, None, 1, True),
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 4444, 1376, None, 4, False),       # a last group of its own round
]
# ... of these another kernel takes
NOT_QUADS = [(1, 32, 1), (1026, 12800, 1), (4444, 1056, 4), (9, 20512, 4)]


@pytest.mark.parametrize("case", QUADS_CASES, ids=lambda c: _id(c[:7]) + f"-{c[7]}")
def test_gemv_of_four_rows_a_wave(oracle, case):
    check_case(oracle, case[:7], case[4] + case[7], native=case[8], vectors=case[7])


# The streaming kernel with long rows, which it keeps where they fill its workgroups: eight waves with one piece of x, and x by segments, with a strip that
# is partly idle and a segment that is cut short.
STREAM_CASES = [
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 2309, 18400, None, 1, False),
    (ElemType.F16, QuantValue.Q8S, [32], QuantParam.F16, 3081, 16416, None, 1, False),
    (ElemType.BF16, QuantValue.E4M3, [128, 128], QuantParam.BF16, 4096, 16384, None, 1, True),
    (ElemType.BF16, QuantValue.Q4F, [64], QuantParam.BF16, 11, 90176, None, 1, False),
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 6, 84000, None, 1, False),
    (ElemType.F16, QuantValue.Q8F, [16], QuantParam.F32, 5, 82000, None, 1, False),
    (ElemType.BF16, QuantValue.E2M1, [32], QuantParam.F32, 7, 98336, None, 1, True),
    (ElemType.F16, QuantValue.Q4S, [32], QuantParam.F32, 2, 16416, 1 << 25, 1, False),      # a pitch that the others do not take
]


@pytest.mark.parametrize("case", STREAM_CASES, ids=lambda c: _id(c[:7]))
def test_gemv_of_long_rows_by_the_streaming_kernel(oracle, case):
    check_case(oracle, case[:7], case[5], native=case[8])


# Every split of a workgroup (four, two or one group of 16 rows; rows on two, four or eight waves): rows that end inside a
# group and leave a workgroup's other groups empty, columns that end inside a stage of eight units or have fewer stages
# than waves, every width of codes and type of scales, as many vectors as one launch takes and one more.  (Tolerance: as
# above; the sums go through fewer additions in a row.)
BATCH_CASES = [
    (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, 16401, 288, None, False),       # 4 x 2, a group and a bit
    (ElemType.F16, QuantValue.Q8S, [32], QuantParam.F16, 16384, 160, None, False),        # 4 x 2, two stages
    (ElemType.F16, QuantValue.Q4S, [128], QuantParam.F16, 8209, 640, None, False),        # 2 x 4
    (ElemType.BF16, QuantValue.E4M3, [32, 32], QuantParam.BF16, 8192, 96, None, True),    # 2 x 4, blocks over rows
    (ElemType.BF16, QuantValue.Q8F, [16], QuantParam.F32, 35, 1040, None, False),         # 1 x 8, a scale per unit
    (ElemType.BF16, QuantValue.E2M1, [64], QuantParam.F16, 17, 1088, None, True),         # 1 x 4 from five vectors on
    (ElemType.F16, QuantValue.Q4F, None, QuantParam.BF16, 15, 4128, None, False),         # one scale
    (ElemType.F16, QuantValue.E5M2, [16], QuantParam.F32, 16, 16, None, True),            # one unit
]


@pytest.mark.parametrize("vectors", [2, 4, 5, 16, 17])
@pytest.mark.parametrize("case", BATCH_CASES, ids=lambda c: _id(c[:7]))
def test_gemv_of_a_batch(oracle, case, vectors):
    check_case(oracle, case[:7], 40 + vectors, native=case[7], vectors=vectors)


# (rows, cols) on both sides of each line that the split of a launch over row groups and waves is drawn at: 256, 512, 768, 1024 and 1536
# groups of 16 rows, rows of 8, 12 and 48 units of 32 (4 bits) values and just more; last, long rows of parts of lines that are streamed all the same (8 bits)
SPLITS = [(17, 288), (4096, 256), (4096, 288), (1000, 384), (1000, 416), (4097, 416), (8192, 320), (8193, 320), (12288, 320), (12289, 320),
          (16384, 288), (16385, 1504), (16385, 1536), (24576, 1568), (24577, 1568), (2833, 9056)]


@pytest.mark.parametrize("vectors", [2, 5, 12, 16])
@pytest.mark.parametrize("value", [QuantValue.Q4S, QuantValue.Q8S, QuantValue.E4M3], ids=lambda v: v.name)
def test_gemv_of_a_batch_splits(value, vectors):
    """Against the float64 product of the dequantized weights (held against the oracle elsewhere); tolerance as above."""
    import torch

    from cubek_amd import dequantize, quantize

    H, client = TensorHandleRef.from_torch, ComputeClient.current()
    store = QuantStore.Native if value == QuantValue.E4M3 else QuantStore.U32
    for i, (rows, cols) in enumerate(SPLITS):
        elem, dtype = ((ElemType.BF16, torch.bfloat16), (ElemType.F16, torch.float16))[i % 2]
        scheme = QuantScheme.default().with_value(value).with_store(store).with_level(QuantLevel.block([32]))
        gen = torch.Generator(device="cuda").manual_seed(rows + vectors)
        w = (torch.randn((rows, cols), generator=gen, device="cuda") * 0.02).to(dtype)
        x = torch.randn((vectors, cols), generator=gen, device="cuda").to(dtype)
        codes = torch.empty(scheme.packed_shape(w.shape), dtype=torch.uint8 if store == QuantStore.Native else torch.int32, device="cuda")
        scales = torch.empty(scheme.scales_shape(w.shape), device="cuda")
        y = torch.full((vectors, rows), float("nan"), device="cuda")
        quantize.launch_dynamic(client, H(w), H(codes), H(scales), scheme, elem)
        dequantize.launch_ref(client, H(codes), H(w), H(scales), scheme, elem)
        matvec.launch_ref(client, H(codes), H(scales), scheme, H(x), H(y), elem, ElemType.F32)
        w64, x64 = w.double(), x.double()
        want, mag = x64 @ w64.t().contiguous(), x64.abs() @ w64.abs().t().contiguous()
        assert torch.all((y.double() - want).abs() <= 2e-5 * mag), (rows, cols)


@pytest.mark.parametrize("vectors", [2, 3, 4, 7, 8, 11])
@pytest.mark.parametrize("kind", ["q4-b32", "q8-b64-f16", "e4m3-native", "q4-general", "q4-wide", "e2m1-native-wide",
                                  "e5m2-native", "q2-in-turns"])
def test_gemv_with_several_right_hand_sides(oracle, kind, vectors):
    """x [vectors, cols] -> y [vectors, rows]: every row of y is the product with that row of x, whichever way the
    vectors are taken (up to sixteen at once on the matrix cores, in turns otherwise)."""
    import torch

    elem, value, block, param, native, rows, cols = {
        "q4-b32": (ElemType.BF16, QuantValue.Q4S, [32], QuantParam.F32, False, 70, 4160),
        "q8-b64-f16": (ElemType.F16, QuantValue.Q8S, [64], QuantParam.F16, False, 33, 2112),
        "e4m3-native": (ElemType.BF16, QuantValue.E4M3, [32], QuantParam.F32, True, 41, 1056),
        "q4-general": (ElemType.BF16, QuantValue.Q4S, [8], QuantParam.F32, False, 20, 512),   # blocks narrower than a unit
        "e5m2-native": (ElemType.F16, QuantValue.E5M2, [64], QuantParam.F32, True, 26, 2112),
        "q2-in-turns": (ElemType.BF16, QuantValue.Q2S, [64], QuantParam.F32, False, 14, 1088),   # 2-bit: one vector per launch
        "q4-wide": (ElemType.BF16, QuantValue.Q4S, [64], QuantParam.BF16, False, 19, 18560),   # five segments of x, the last short
        "e2m1-native-wide": (ElemType.F16, QuantValue.E2M1, [32], QuantParam.F32, True, 10, 10304),
    }[kind]
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block(block)).with_param(param)
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rng = np.random.default_rng(vectors * 100 + cols)
    w32 = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
    wb = oracle.to_bits(w32, elem)
    scales = oracle.compute_scales(wb, elem, (rows, cols), scheme)
    words, out_scale = oracle.quantize(wb, elem, (rows, cols), scales, scheme)
    deq = oracle.from_bits(oracle.dequantize(words, (rows, cols), out_scale, elem, scheme), elem).astype(np.float64)
    xpitch = cols + 8 * int(rng.integers(0, 3))  # rows of x on 16-byte boundaries, sometimes pitched
    xb = np.zeros((vectors, xpitch), np.uint16)
    xb[:, :cols] = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
    x64 = oracle.from_bits(xb[:, :cols].copy(), elem).astype(np.float64).reshape(vectors, cols)
    want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    wpr = cols // scheme.num_quants()
    stored = words.reshape(rows, wpr)
    d_words = torch.from_numpy(stored if native else stored.view(np.int32)).cuda()
    to16 = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda() if a.dtype == np.uint16 \
        else torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d_scales, d_x = to16(out_scale), to16(xb)
    h = TensorHandleRef.from_torch
    h_x = TensorHandleRef(d_x.data_ptr(), (vectors, cols), (xpitch, 1), 2)
    y = torch.full((vectors, rows + 3), float("nan"), dtype=torch.float32, device="cuda")
    h_y = TensorHandleRef(y.data_ptr(), (vectors, rows), (rows + 3, 1), 4)
    matvec.launch_ref(ComputeClient.current(), h(d_words), h(d_scales), scheme, h_x, h_y, elem, ElemType.F32)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    assert np.all(np.isnan(got[:, rows:]))  # nothing written between the rows of y
    assert np.all(np.abs(got[:, :rows] - want) <= 2e-5 * mag + 1e-30), float(np.max(np.abs(got[:, :rows] - want) / (mag + 1e-30)))


def test_gemv_random_configurations(oracle):
    """Sixty drawn cases (CQ_RANDOM_GEMV=N: N) of the streaming kernel's domain and its edges: every code width,
    block extents from one 16-byte unit up (also over rows), one scale per tensor, every scale type, ragged strips,
    pitched words, one to six right-hand sides, both stores, x in all three float types."""
    import os

    rng = np.random.default_rng(2024)
    values = {2: [QuantValue.Q2S, QuantValue.Q2F], 4: [QuantValue.Q4S, QuantValue.Q4F, QuantValue.E2M1],
              8: [QuantValue.Q8S, QuantValue.Q8F]}
    for i in range(int(os.environ.get("CQ_RANDOM_GEMV", "60"))):
        bits = int(rng.choice([2, 4, 8]))
        unit = 128 // bits
        elem = [ElemType.BF16, ElemType.F16, ElemType.BF16, ElemType.F32][int(rng.integers(4))]
        param = [QuantParam.F32, QuantParam.F16, QuantParam.BF16][int(rng.integers(3))]
        if elem == ElemType.F32 and rng.random() < 0.8:
            param = QuantParam.F32  # (f32 x streams under f32 scales; the rest goes to the general kernel)
        kind = int(rng.integers(4))
        units_per_block = int(2 ** rng.integers(0, 3))
        bc = unit * units_per_block
        if bc > 255:  # block extents are bytes in the scheme
            bc, units_per_block = unit, 1
        blocks = int(rng.integers(1, max(2, 6000 // bc)))
        cols = bc * blocks
        rows = int(rng.integers(1, 70))
        block = [bc]
        if kind == 0:
            block = None
        elif kind == 1:
            br = int(rng.choice([2, 3, 5]))
            rows = br * int(rng.integers(1, 20))
            block = [br, bc]
        value = values[bits][int(rng.integers(len(values[bits])))]
        wpr = cols // (32 // bits)
        pitch = None if rng.random() < 0.6 else wpr + 4 * int(rng.integers(1, 5))
        vectors = int(rng.choice([1, 1, 1, 2, 4, 5, 6]))
        # every third case in the native store, where the value has one (bytes: the pitch counts bytes)
        native = i % 3 == 2 and value in (QuantValue.Q8S, QuantValue.Q8F, QuantValue.E2M1)
        if native and elem == ElemType.F32:
            param = QuantParam.F32  # the native store only streams, and f32 x streams under f32 scales
        if native:
            pitch = None if pitch is None else (cols // (2 if value == QuantValue.E2M1 else 1)) + 16 * int(rng.integers(1, 4))
        check_case(oracle, (elem, value, block, param, rows, cols, pitch), 1000 + i, native=native, vectors=vectors)


@pytest.mark.parametrize("elem", [ElemType.BF16, ElemType.F16], ids=lambda e: e.name)
def test_gemv_scales_of_every_kind(oracle, elem):
    """Negative, zero, tiny and huge scales among ordinary ones (the streaming kernel of one vector sends their lanes down a
    plain path; several vectors at once take all of these the short way): same tolerance against the oracle's
    dequantized weights."""
    import torch

    rows, cols = 96, 4096
    scheme = QuantScheme.default().with_value(QuantValue.Q4S).with_level(QuantLevel.block([32]))
    rng = np.random.default_rng(5)
    words = rng.integers(0, 2**32, (rows, cols // 8), dtype=np.uint64).astype(np.uint32)
    scales = rng.uniform(0.001, 0.02, (rows, cols // 32)).astype(np.float32)
    odd = rng.random(scales.shape) < 0.05
    scales[odd] = rng.choice(np.array([-0.01, 0.0, -0.0, 1e-36, -3.0, 2.0 ** -110, 3000.0, -1e-30], np.float32), int(odd.sum()))
    deq = oracle.from_bits(oracle.dequantize(words, (rows, cols), scales, elem, scheme), elem).astype(np.float64)
    assert np.all(np.isfinite(deq))
    d_words = torch.from_numpy(words.view(np.int32)).cuda()
    d_scales = torch.from_numpy(scales).cuda()
    h = TensorHandleRef.from_torch
    for vectors in (1, 3):  # one right-hand side, and three at once
        xb = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
        x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
        want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
        d_x = torch.from_numpy(xb.view(np.int16)).cuda()
        y = torch.zeros((vectors, rows), dtype=torch.float32, device="cuda")
        hx, hy = (h(d_x), h(y)) if vectors > 1 else (h(d_x[0]), h(y[0]))
        matvec.launch_ref(ComputeClient.current(), h(d_words), h(d_scales), scheme, hx, hy, elem, ElemType.F32)
        torch.cuda.synchronize()
        got = y.cpu().numpy().astype(np.float64)
        assert np.all(np.abs(got - want) <= 2e-5 * mag + 1e-30), (vectors, float(np.max(np.abs(got - want) / (mag + 1e-30))))


# Several vectors at once: the short dequantization takes every scale below 2^100 in size, of either sign, zero and denormal
# ones as well; a larger one sends its wave's stage through the general code, whose operands are picked out one by one (4-bit
# f16 weights and x in another order than elsewhere, 8-bit words in pairs).  (Tolerance: as above.)
SCALE_CASES = {
    "bf16": [-0.01, 0.0, -0.0, 1e-36, -3.0, 2.0 ** -110, 3000.0, -1e-30, 1e-39, 2.0 ** 99, -(2.0 ** 99)],
    "bf16-large": [-0.01, 0.0, 2.0 ** 100, -(2.0 ** 101), 2.0 ** 110],
    "f16": [-0.01, 0.0, -0.0, 1e-36, -3.0, 1e-7, -6e-8, 400.0, 2.0 ** -110],
    "f16-edge": [4092.0, -4092.0, 4096.0, -4096.0, 8188.0, -8188.0, 6e-8, -6e-8],   # both sides of where the short way of 4 bits ends
    "f16-infinite": [1e6, 65520.0, np.inf],   # infinite once they are f16
    "bf16-infinite": [np.inf],
}


@pytest.mark.parametrize("vectors", [2, 5, 16])
@pytest.mark.parametrize("value", [QuantValue.Q4S, QuantValue.Q8S, QuantValue.E4M3, QuantValue.E2M1], ids=lambda v: v.name)
@pytest.mark.parametrize("kind", list(SCALE_CASES))
def test_gemv_of_a_batch_scales_of_every_kind(oracle, kind, value, vectors):
    """Odd scales in one block in twenty, and in a row's last one; an infinite one stands on codes of one sign against ones
    in x, so that its row sums to that infinity and every other row stays finite."""
    import torch

    elem = ElemType.F16 if kind.startswith("f16") else ElemType.BF16
    infinite = kind.endswith("infinite")
    native = value in (QuantValue.E4M3, QuantValue.E2M1)
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block([32]))
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rows, cols = 83, 1312   # 41 blocks: a last stage cut short for every width
    rng = np.random.default_rng(31 + vectors)
    bits = {QuantValue.Q8S: 8, QuantValue.E4M3: 8}.get(value, 4)
    codes = rng.integers(0, 256, (rows, cols * bits // 8), dtype=np.uint8)
    if value == QuantValue.E4M3:
        codes &= 0xBF   # no NaN, and 1.9 at most
    scales = rng.uniform(0.001, 0.02, (rows, cols // 32)).astype(np.float32)
    odd = np.array(SCALE_CASES[kind], np.float32)
    if kind == "f16-edge" and value == QuantValue.Q8S:
        odd /= 16  # 128 * 512 would not be a number of f16
    xb = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
    if infinite:
        for k, (row, block) in enumerate(((2, 0), (17, 20), (40, cols // 32 - 1), (82, 7))):
            scales[row, block] = odd[k % len(odd)]
            at = slice(block * 32 * bits // 8, (block + 1) * 32 * bits // 8)
            codes[row, at] = 0x33 if bits == 4 else 0x38
            xb[:, block * 32:(block + 1) * 32] = oracle.to_bits(np.ones(32, np.float32), elem)
    else:
        at = rng.random(scales.shape) < 0.05
        at[:, -1] |= rng.random(rows) < 0.3
        scales[at] = rng.choice(odd, int(at.sum()))
    stored = codes if native else codes.view(np.uint32)
    deq = oracle.from_bits(oracle.dequantize(stored, (rows, cols), scales, elem, scheme), elem).astype(np.float64)
    assert infinite or np.all(np.isfinite(deq))
    x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
    with np.errstate(invalid="ignore", over="ignore"):
        want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    h = TensorHandleRef.from_torch
    d_stored = torch.from_numpy(stored if native else stored.view(np.int32)).cuda()
    d_scales, d_x = torch.from_numpy(scales).cuda(), torch.from_numpy(xb.view(np.int16)).cuda()
    y = torch.zeros((vectors, rows), dtype=torch.float32, device="cuda")
    matvec.launch_ref(ComputeClient.current(), h(d_stored), h(d_scales), scheme, h(d_x), h(y), elem, ElemType.F32)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    finite = np.isfinite(want)
    assert np.array_equal(np.flatnonzero(~finite[0]), [2, 17, 40, 82] if infinite else []) and not np.any(np.isnan(want))
    assert np.array_equal(got[~finite], want[~finite])
    err = np.abs(got[finite] - want[finite])
    assert np.all(err <= 2e-5 * mag[finite] + 1e-30), float(np.max(err / (mag[finite] + 1e-30)))


# Steps of sixteen units and a last one of one or two, shared by all waves.  Values of unit deviation for x but where the weights are tiny.
@pytest.mark.parametrize("vectors", [1, 3])
@pytest.mark.parametrize("value", [QuantValue.Q4S, QuantValue.Q8S, QuantValue.E4M3, QuantValue.E2M1], ids=lambda v: v.name)
@pytest.mark.parametrize("kind", ["bf16", "bf16-large", "bf16-subnormal", "bf16-infinite", "f16", "f16-edge", "f16-subnormal", "f16-infinite"])
def test_gemv_of_four_rows_a_wave_scales_of_every_kind(oracle, kind, value, vectors):
    """Odd scales in one block in twenty and in a row's last one; all weights subnormal numbers of their type, against x large enough for sums
    above the tolerance's floor; an infinite scale on codes of one sign against ones in x."""
    import torch

    rows, cols = 70, 16416
    elem, ulp, normal = (ElemType.F16, 2.0 ** -24, 2.0 ** -14) if kind.startswith("f16") else (ElemType.BF16, 2.0 ** -133, 2.0 ** -126)
    infinite, subnormal = kind.endswith("infinite"), kind.endswith("subnormal")
    native = value in (QuantValue.E4M3, QuantValue.E2M1)
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block([32]))
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rng = np.random.default_rng(91 + vectors)
    bits = {QuantValue.Q8S: 8, QuantValue.E4M3: 8}.get(value, 4)
    codes = rng.integers(0, 256, (rows, cols * bits // 8), dtype=np.uint8)
    if value == QuantValue.E4M3:
        codes &= 0xBF   # no NaN, and 1.9 at most
    blocks = (rows, cols // 32)
    x32 = rng.normal(0, 1, (vectors, cols)).astype(np.float32)
    if subnormal:
        step = {QuantValue.Q8S: 128, QuantValue.Q4S: 8, QuantValue.E2M1: 6}.get(value, 2)  # the largest code
        scales = (rng.integers(1, int(normal / ulp / step) + 1, blocks) * ulp).astype(np.float32)
        x32 *= 100.0 if elem == ElemType.F16 else np.float32(2.0 ** 120)
    else:
        scales = rng.uniform(0.001, 0.02, blocks).astype(np.float32)
        odd = np.array(SCALE_CASES[kind], np.float32)
        if kind == "f16-edge" and value == QuantValue.Q8S:
            odd /= 16  # 128 * 512 would not be a number of f16
        at = rng.random(blocks) < 0.05
        at[:, -1] |= rng.random(rows) < 0.3
        if not infinite:
            scales[at] = rng.choice(odd, int(at.sum()))
    xb = oracle.to_bits(x32, elem).reshape(vectors, cols)
    wrong = [2, 17, 40, 69] if infinite else []
    for k, (row, block) in enumerate(zip(wrong, (0, 300, cols // 32 - 1, 7))):
        scales[row, block] = odd[k % len(odd)]
        codes[row, slice(block * 32 * bits // 8, (block + 1) * 32 * bits // 8)] = 0x33 if bits == 4 else 0x38
        xb[:, block * 32:(block + 1) * 32] = oracle.to_bits(np.ones(32, np.float32), elem)
    stored = codes if native else codes.view(np.uint32)
    deq = oracle.from_bits(oracle.dequantize(stored, (rows, cols), scales, elem, scheme), elem).astype(np.float64)
    if subnormal:
        assert np.max(np.abs(deq)) <= normal and np.mean(deq != 0) > 0.7
    x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
    with np.errstate(invalid="ignore", over="ignore"):
        want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    h = TensorHandleRef.from_torch
    d_stored = torch.from_numpy(stored if native else stored.view(np.int32)).cuda()
    d_scales, d_x = torch.from_numpy(scales).cuda(), torch.from_numpy(xb.view(np.int16)).cuda()
    y = torch.zeros((vectors, rows), dtype=torch.float32, device="cuda")
    h_x, h_y = (h(d_x), h(y)) if vectors > 1 else (h(d_x[0]), h(y[0]))
    matvec.launch_ref(ComputeClient.current(), h(d_stored), h(d_scales), scheme, h_x, h_y, elem, ElemType.F32)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    finite = np.isfinite(want)
    assert np.array_equal(np.flatnonzero(~finite[0]), wrong) and not np.any(np.isnan(want))
    assert np.array_equal(got[~finite], want[~finite])
    err = np.abs(got[finite] - want[finite])
    assert np.all(err <= 2e-5 * mag[finite] + 1e-30), float(np.max(err / (mag[finite] + 1e-30)))


def test_gemv_scales_with_strides(oracle):
    """The scales of a [rows, blocks] layout stored column by column (strides (1, rows)) and with a row pitch: the kernels of
    one vector and of several address them through both strides."""
    import torch

    rows, cols = 37, 2304
    scheme = QuantScheme.default().with_value(QuantValue.Q4S).with_level(QuantLevel.block([32]))
    rng = np.random.default_rng(11)
    words = rng.integers(0, 2**32, (rows, cols // 8), dtype=np.uint64).astype(np.uint32)
    scales = rng.uniform(0.001, 0.02, (rows, cols // 32)).astype(np.float32)
    deq = oracle.from_bits(oracle.dequantize(words, (rows, cols), scales, ElemType.BF16, scheme), ElemType.BF16).astype(np.float64)
    xb = oracle.to_bits(rng.normal(0, 1, (6, cols)).astype(np.float32), ElemType.BF16).reshape(6, cols)
    x64 = oracle.from_bits(xb, ElemType.BF16).astype(np.float64).reshape(6, cols)
    want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    d_words = torch.from_numpy(words.view(np.int32)).cuda()
    d_x = torch.from_numpy(xb.view(np.int16)).cuda()
    h = TensorHandleRef.from_torch
    nb = cols // 32
    col_major = torch.from_numpy(np.ascontiguousarray(scales.T)).cuda()           # [blocks, rows]
    pitched = torch.zeros((rows, nb + 5), dtype=torch.float32, device="cuda")
    pitched[:, :nb] = torch.from_numpy(scales).cuda()
    for name, h_scales in (("column-major", TensorHandleRef(col_major.data_ptr(), (rows, nb), (1, rows), 4)),
                           ("pitched", TensorHandleRef(pitched.data_ptr(), (rows, nb), (nb + 5, 1), 4))):
        for vectors in (1, 6):
            y = torch.full((vectors, rows), float("nan"), dtype=torch.float32, device="cuda")
            hx, hy = (h(d_x), h(y)) if vectors > 1 else (h(d_x[0]), h(y[0]))
            matvec.launch_ref(ComputeClient.current(), h(d_words), h_scales, scheme, hx, hy, ElemType.BF16, ElemType.F32)
            torch.cuda.synchronize()
            got = y.cpu().numpy().astype(np.float64)
            assert np.all(np.abs(got - want[:vectors]) <= 2e-5 * mag[:vectors] + 1e-30), (name, vectors)


@pytest.mark.parametrize("case", [
    (ElemType.F16, QuantValue.Q4S, [128], QuantParam.F16, False), (ElemType.BF16, QuantValue.Q8S, [16], QuantParam.BF16, False),
    (ElemType.F16, QuantValue.E2M1, [64], QuantParam.F32, True), (ElemType.BF16, QuantValue.E4M3, [4, 32], QuantParam.F16, True)],
    ids=lambda c: f"{c[0].name}-{c[1].name}-{c[3].name}")
def test_gemv_of_a_batch_scales_with_strides(oracle, case):
    """Several vectors: scales column by column, pitched, and every third entry of a larger tensor, in each of their types."""
    import torch

    elem, value, block, param, native = case
    rows, cols, vectors = 52, 1408, 3
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block(block)).with_param(param)
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rng = np.random.default_rng(77)
    wb = oracle.to_bits(rng.normal(0, 0.02, (rows, cols)).astype(np.float32), elem)
    words, stored_scales = oracle.quantize(wb, elem, (rows, cols), oracle.compute_scales(wb, elem, (rows, cols), scheme), scheme)
    deq = oracle.from_bits(oracle.dequantize(words, (rows, cols), stored_scales, elem, scheme), elem).astype(np.float64)
    xb = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
    x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
    want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    words = words.reshape(rows, -1)
    d_words = torch.from_numpy(words if native else words.view(np.int32)).cuda()
    d_x = torch.from_numpy(xb.view(np.int16)).cuda()
    shape = scheme.scales_shape((rows, cols))
    scales = stored_scales.reshape(shape)
    h = TensorHandleRef.from_torch
    for strides in ((1, shape[0]), (shape[1] + 3, 1), (3 * shape[1], 3)):
        room = np.zeros((shape[0] - 1) * strides[0] + (shape[1] - 1) * strides[1] + 1, scales.dtype)
        np.lib.stride_tricks.as_strided(room, shape, tuple(n * room.itemsize for n in strides))[...] = scales
        d_scales = torch.from_numpy(room.view(np.int16) if room.dtype == np.uint16 else room).cuda()
        y = torch.full((vectors, rows), float("nan"), dtype=torch.float32, device="cuda")
        matvec.launch_ref(ComputeClient.current(), h(d_words), TensorHandleRef(d_scales.data_ptr(), shape, strides, room.itemsize), scheme,
                          h(d_x), h(y), elem, ElemType.F32)
        torch.cuda.synchronize()
        got = y.cpu().numpy().astype(np.float64)
        assert np.all(np.abs(got - want) <= 2e-5 * mag + 1e-30), strides


@pytest.mark.parametrize("kind", ["e4m3-native", "q4-f32-x", "q4-bf16", "q4-bf16-four-vectors"])
def test_gemv_infinite_scale_in_a_rows_last_unit(oracle, kind):
    """Rows whose last strip is partly filled (cols / values per unit is not a multiple of 64), with an infinite scale
    on the last block of one row and +-0 codes elsewhere in it: the lanes past the row's end must contribute nothing
    (they hold the last unit again against zeros of x, and Inf * 0 is NaN).  The row with the infinite scale sums to
    +-Inf or NaN exactly where the float64 product over the oracle's dequantized weights does; every other row is
    finite and within the tolerance."""
    import torch

    native = kind == "e4m3-native"
    elem = ElemType.F32 if kind == "q4-f32-x" else ElemType.BF16
    vectors = 4 if kind.endswith("four-vectors") else 1
    value = QuantValue.E4M3 if native else QuantValue.Q4S
    scheme = QuantScheme.default().with_value(value).with_level(QuantLevel.block([32]))
    if native:
        scheme = scheme.with_store(QuantStore.Native)
    rows, cols = 6, 2080   # 65 units of 32 values (130 of 16 for the bytes): the last strip holds one or two units
    rng = np.random.default_rng(21)
    nq = scheme.num_quants()
    if native:
        stored = rng.integers(0, 120, (rows, cols), dtype=np.uint8) | (rng.integers(0, 2, (rows, cols), dtype=np.uint8) << 7)
    else:
        stored = rng.integers(0, 2**32, (rows, cols // nq), dtype=np.uint64).astype(np.uint32)
    scales = rng.uniform(0.001, 0.02, (rows, cols // 32)).astype(np.float32)
    scales[2, -1] = np.inf
    # that block's codes are all +3 (e4m3: 1.0) and x is +1 there, so row 2 sums to +Inf, not to NaN
    if native:
        stored[2, -32:] = 0x38
    else:
        stored[2, -(32 // nq):] = 0x33333333
    deq = oracle.from_bits(oracle.dequantize(stored, (rows, cols), scales, elem, scheme), elem).astype(np.float64)
    xb = oracle.to_bits(rng.normal(0, 1, (vectors, cols)).astype(np.float32), elem).reshape(vectors, cols)
    xb[:, -32:] = oracle.to_bits(np.ones(32, np.float32), elem)
    x64 = oracle.from_bits(xb, elem).astype(np.float64).reshape(vectors, cols)
    with np.errstate(invalid="ignore", over="ignore"):
        want, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
    d_stored = torch.from_numpy(stored if native else stored.view(np.int32)).cuda()
    d_scales = torch.from_numpy(scales).cuda()
    d_x = torch.from_numpy(xb.view(np.int16) if elem != ElemType.F32 else xb).cuda()
    h = TensorHandleRef.from_torch
    y = torch.zeros((vectors, rows), dtype=torch.float32, device="cuda")
    hx, hy = (h(d_x), h(y)) if vectors > 1 else (h(d_x[0]), h(y[0]))
    matvec.launch_ref(ComputeClient.current(), h(d_stored), h(d_scales), scheme, hx, hy, elem, ElemType.F32)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    finite = np.isfinite(want)
    assert np.all(want[:, 2] == np.inf) and finite[:, [0, 1, 3, 4, 5]].all()
    assert np.all(np.abs(got - want)[finite] <= (2e-5 * mag + 1e-30)[finite]), kind
    assert np.array_equal(np.isnan(got), np.isnan(want)), (kind, got[:, 2], want[:, 2])
    assert np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)]), (kind, got[:, 2], want[:, 2])


def test_gemv_without_columns_gives_zeros():
    """cols == 0: every sum is empty, y is written with zeros (one vector and three)."""
    import torch

    scheme = QuantScheme.default().with_value(QuantValue.Q4S)
    h = TensorHandleRef
    w = torch.zeros(4, dtype=torch.int32, device="cuda")
    s = torch.ones(1, dtype=torch.float32, device="cuda")
    x = torch.zeros(4, dtype=torch.bfloat16, device="cuda")
    for vectors in (1, 3):
        y = torch.full((vectors, 7), float("nan"), dtype=torch.float32, device="cuda")
        h_x = h(x.data_ptr(), (0,), (1,), 2) if vectors == 1 else h(x.data_ptr(), (vectors, 0), (0, 1), 2)
        h_y = h.from_torch(y[0]) if vectors == 1 else h.from_torch(y)
        matvec.launch_ref(ComputeClient.current(), h(w.data_ptr(), (7, 0), (0, 1), 4), h.from_torch(s), scheme, h_x, h_y,
                          ElemType.BF16, ElemType.F32)
        torch.cuda.synchronize()
        assert torch.equal(y, torch.zeros_like(y)), vectors


def test_gemv_argument_checks():
    import torch

    scheme = QuantScheme.default().with_value(QuantValue.Q4S).with_level(QuantLevel.block([32]))
    w = torch.zeros((8, 16), dtype=torch.int32, device="cuda")
    s = torch.ones((8, 4), dtype=torch.float32, device="cuda")
    x = torch.zeros(128, dtype=torch.bfloat16, device="cuda")
    y = torch.zeros(8, dtype=torch.float32, device="cuda")
    h = TensorHandleRef.from_torch
    client = ComputeClient.current()
    matvec.launch_ref(client, h(w), h(s), scheme, h(x), h(y), ElemType.BF16, ElemType.F32)

    def status(fn):
        with pytest.raises(_ffi.QuantError) as e:
            fn()
        return e.value.status

    assert status(lambda: matvec.launch_ref(client, h(w), h(s), scheme, h(x[:64]), h(y), ElemType.BF16, ElemType.F32)) \
        == _ffi.ERR_SHAPE_MISMATCH
    assert status(lambda: matvec.launch_ref(client, h(w), h(s[:, :3]), scheme, h(x), h(y), ElemType.BF16, ElemType.F32)) \
        == _ffi.ERR_SHAPE_MISMATCH
    assert status(lambda: matvec.launch_ref(client, h(w), h(s), scheme, h(x), h(y), ElemType.F32, ElemType.F32)) \
        == _ffi.ERR_SHAPE_MISMATCH  # x is not f32
    from cubek_amd import QuantStore
    assert status(lambda: matvec.launch_ref(client, h(w), h(s), scheme.with_store(QuantStore.Native), h(x), h(y),
                                            ElemType.BF16, ElemType.F32)) == _ffi.ERR_UNSUPPORTED_SCHEME
    assert status(lambda: matvec.launch_ref(client, h(w.t()), h(s), scheme, h(x), h(y), ElemType.BF16, ElemType.F32)) \
        in (_ffi.ERR_NON_CONTIGUOUS, _ffi.ERR_SHAPE_MISMATCH)
