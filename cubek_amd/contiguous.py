"""Re-packing of strided quantized tensors: ``into_contiguous_packed`` of cubecl-std as
cubek-matmul calls it on quantized operands (crates/cubek-matmul/src/base.rs:505-529).
Executed by gfx950 kernels behind the C ABI; the caller provides the output.
"""
from __future__ import annotations

from typing import Sequence

from . import _ffi
from .tensor import ComputeClient, TensorHandleRef


def into_contiguous_packed_ref(client: ComputeClient, input: TensorHandleRef, output: TensorHandleRef,
                               shape: Sequence[int], packing: int) -> None:
    """``shape`` is the logical (unpacked) shape; ``input`` holds ``packing`` values per
    stored element along its rightmost stride-1 dimension, ``output`` is contiguous with
    the last dimension of ``shape`` divided by ``packing``."""
    rc = _ffi.calls().repack(client.stream, input, output, shape, packing)
    if rc:
        _ffi.check(rc)
