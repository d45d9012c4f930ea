"""The package's calls (csrc/py_call.cpp) against the C ABI called with the structs that the handles and the scheme build: the same
status for every descriptor that is refused before anything touches a GPU, and the same refusals of other Python objects."""
import ctypes
import os
import subprocess

import pytest

from cubek_amd import (ElemType, QuantError, QuantLevel, QuantParam, QuantScheme, QuantStore, QuantValue, TensorHandleRef, ComputeClient,
                       _ffi, contiguous, dequantize, matvec, quantize, reduce)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
P = 1 << 20  # never read: every call here is refused
BLOCK = QuantScheme.default().with_value(QuantValue.Q4S).with_level(QuantLevel.block([32]))


def handle(shape, size=2, strides=None, ptr=P):
    if strides is None:
        strides, n = [], 1
        for s in reversed(shape):
            strides.insert(0, n)
            n *= s
    return TensorHandleRef(ptr, tuple(shape), tuple(strides), size)


SCHEMES = [QuantScheme.default(), BLOCK, BLOCK.with_level(QuantLevel.block([3])), BLOCK.with_level(QuantLevel.block([2, 1, 5, 7, 32])),
           BLOCK.with_store(QuantStore.Native), BLOCK.with_value(QuantValue.E4M3).with_store(QuantStore.Native).with_param(QuantParam.BF16),
           BLOCK.with_param(QuantParam.F16)]
# floats that do not go with codes of [4, 8] words, one for each field
FLOATS = [handle((4, 64), ptr=0), handle((4, 63)), handle((4, 64), size=4), handle((4, 2 ** 62)), handle((1,) * 8 + (64,)), handle(()),
          handle((4, 64), strides=(64,)), handle((4.0, 31)), handle((4, -1))]


@pytest.mark.parametrize("scheme", SCHEMES, ids=range(len(SCHEMES)))
@pytest.mark.parametrize("floats", FLOATS, ids=range(len(FLOATS)))
def test_the_status_is_the_one_of_the_structs(floats, scheme):
    codes, scales = handle((4, 8), size=3), handle((4, 2), size=4)
    L, c, e = _ffi.lib(), _ffi.calls(), ElemType.BF16
    s = scheme.to_c()
    f, q, p = floats.as_c(), codes.as_c(), scales.as_c()
    pairs = [(c.quantize(0, floats, codes, floats, scales, scheme, e), L.cq_quantize(0, f, q, f, p, s, 2)),
             (c.dequantize(0, codes, floats, scales, scheme, e), L.cq_dequantize(0, q, f, p, s, 2)),
             (c.compute_scales(0, floats, codes, scheme, e, 0, 0), L.cq_compute_scales(0, f, q, s, 2, 0, 0)),
             (c.quantize_dynamic(None, floats, codes, scales, scheme, e, None, 0), L.cq_quantize_dynamic(None, f, q, p, s, 2, None, 0)),
             (c.quantize_dynamic_static(0, floats, codes, scales, scheme, e), L.cq_quantize_dynamic_static(0, f, q, p, s, 2)),
             (c.gemv(0, codes, scales, scheme, floats, floats, e, e), L.cq_gemv_quantized(0, q, p, s, f, f, 2, 2)),
             (c.max_abs(0, floats, codes, 1, e, 0, 0), L.cq_reduce_max_abs(0, f, q, 1, 2, 0, 0)),
             (c.repack(0, codes, floats, [4, 64], 8), L.cq_into_contiguous_packed(0, q, f, (ctypes.c_uint64 * 2)(4, 64), 2, 8))]
    assert all(got == want != 0 for got, want in pairs), pairs


def test_objects_that_stand_for_handles_and_schemes():
    class Handle:
        def __init__(self, h):
            self.h = h

        def as_c(self):
            return self.h.as_c()

    class Scheme:
        def to_c(self):
            return BLOCK.to_c()

    for floats in FLOATS:
        codes, scales = handle((4, 8), 3), handle((4, 2), 4)
        errors = []
        for f, s in ((floats, BLOCK), (Handle(floats), Scheme())):
            with pytest.raises(QuantError) as e:
                dequantize.launch_ref(ComputeClient(), codes, f, scales, s, ElemType.BF16)
            errors.append(e.value.status)
        assert errors[0] == errors[1]


def test_other_objects_are_refused():
    h, client = handle((4, 64)), ComputeClient()
    for call in (lambda: dequantize.launch_ref(client, None, h, h, BLOCK, ElemType.F16),
                 lambda: dequantize.launch_ref(client, h, h, h, None, ElemType.F16)):
        with pytest.raises(AttributeError):
            call()
    for call in (lambda: dequantize.launch_ref(client, h, h, h, BLOCK, None),
                 lambda: dequantize.launch_ref(ComputeClient("0"), h, h, h, BLOCK, ElemType.F16),
                 lambda: quantize.launch_dynamic(client, h, h, h, BLOCK, ElemType.F16, 1.5, 0),
                 lambda: quantize.launch_dynamic(client, h, h, h, BLOCK, ElemType.F16, 0, 1024.0),
                 lambda: reduce.max_abs(client, h, h, 1.0, ElemType.F16),
                 lambda: contiguous.into_contiguous_packed_ref(client, h, h, (4.0, 64), 8),
                 lambda: matvec.launch_ref(client, h, h, BLOCK, TensorHandleRef(P, 4, 4, 2), h, ElemType.F16, ElemType.F16),
                 lambda: _ffi.calls().quantize(0, h)):
        with pytest.raises((TypeError, AttributeError)):
            call()
    with pytest.raises(IndexError):
        dequantize.launch_ref(client, handle((4,), strides=(4, 1)), h, h, BLOCK, ElemType.F16)
    # a ctypes pointer and a ctypes integer go for numbers
    got = _ffi.calls().max_abs(ctypes.c_void_p(0), h, h, ctypes.c_uint32(1), ElemType.F16, ctypes.c_void_p(0), ctypes.c_size_t(0))
    assert got == _ffi.ERR_SHAPE_MISMATCH


def test_the_module_is_named_after_the_interpreter_it_was_built_for():
    import sysconfig

    assert os.path.basename(_ffi.calls().__file__) == "_call" + sysconfig.get_config_var("EXT_SUFFIX")


def test_the_library_builds_without_python():
    made = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "cubek_amd", "csrc"), "native", "PYTHON=false"], stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, text=True)
    assert made.returncode == 0 and "libcubek_quant_hip.so" in made.stdout and "py_call.cpp" not in made.stdout
