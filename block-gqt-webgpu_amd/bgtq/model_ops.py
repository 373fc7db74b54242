"""The model step's kernel protocol: ModelOps / Commands of src/model/ops.ts.

ModelOps.create(device).commands() records dispatch(name, parameters,
buffers, x, y) calls and submit() runs them in order on the device's stream
and waits, as the reference's Commands does (src/model/ops.ts:21-31). The
names on the attention path are served by libbgtq.so (bgtq_model_submit):
append, encode_k, dot, compressed_dot, softmax and weighted, with the
reference's parameter arrays, binding orders and buffer layouts (as
src/model/decoder.ts:46-56 dispatches them). The model's other kernels
(embedding, matmul, norm, element, rope) raise UnsupportedError.

A buffer is a torch tensor on the GPU (device memory only: torch is the
allocator here, the arithmetic runs in the library's kernels), or, for the
config and table slots of encode_k and compressed_dot, the head's calibration
tables (a Calibration head's .config / .table, or a Tables object).
"""
from __future__ import annotations

import ctypes
import struct
import sys

from . import _lib
from ._lib import RangeError, check, lib

# Largest workgroup count per dimension a dispatch may name (the reference
# checks device.limits.maxComputeWorkgroupsPerDimension, src/model/ops.ts:26).
MAX_WORKGROUPS_PER_DIMENSION = 0x7FFFFFFF

ATTENTION_PATH = ("append", "encode_k", "dot", "compressed_dot", "softmax", "weighted")


# The C structs a submit passes, filled with struct: building a ctypes object per
# binding (37 in a SmolLM2 layer's nine dispatches) cost as much host time as
# the layer's kernels take.
_DISPATCH = struct.Struct("=Q8IQQII")  # bgtq_model_dispatch
assert _DISPATCH.size == ctypes.sizeof(_lib.ModelDispatch) and ctypes.sizeof(_lib.Binding) == 24
_NAMES = {n: ctypes.create_string_buffer(n.encode()) for n in ATTENTION_PATH}


_TENSORS: set = set()  # torch's own tensor types, once met: no attributes to look for


def _binding(b) -> tuple[int, int, int]:
    """bgtq_model_binding's words: device address, bytes, tables handle."""
    if type(b) in _TENSORS:
        if not b.is_contiguous():
            raise RangeError("Model buffers must be contiguous")
        return b.data_ptr(), b.nbytes, 0
    if b is None:
        return 0, 0, 0
    handle = getattr(b, "handle", None)
    if handle is not None and hasattr(b, "info"):  # calibration Tables
        return 0, 0, getattr(handle, "value", handle) or 0
    if not b.is_contiguous():
        raise RangeError("Model buffers must be contiguous")
    torch = sys.modules.get("torch")
    if torch is not None and type(b) in (torch.Tensor, torch.nn.Parameter):
        _TENSORS.add(type(b))
    return b.data_ptr(), b.numel() * b.element_size(), 0


class ModelOps:
    def __init__(self, device):
        self.device = device

    @classmethod
    def create(cls, device) -> "ModelOps":
        return cls(device)

    def commands(self) -> "Commands":
        return Commands(self)


class Commands:
    def __init__(self, ops: ModelOps):
        self.ops = ops
        self._dispatches: list[tuple[str, list[int], list, int, int]] = []

    def dispatch(self, name: str, parameters, buffers, x: int, y: int = 1) -> None:
        if x > MAX_WORKGROUPS_PER_DIMENSION or y > MAX_WORKGROUPS_PER_DIMENSION:
            raise RangeError("Model dispatch limit")
        params = [int(v) & 0xFFFFFFFF for v in list(parameters)[:8]]
        if len(params) < 8:
            params += [0] * (8 - len(params))
        self._dispatches.append((name, params, list(buffers), int(x), int(y)))

    def submit(self) -> None:
        """Queue every recorded dispatch in order, then wait for the device.
        A dispatch that fails its checks raises before anything is queued."""
        n = len(self._dispatches)
        words, keep = [], []
        for _, _, buffers, _, _ in self._dispatches:
            for b in buffers:
                words += _binding(b)
        binds = (ctypes.c_uint64 * max(1, len(words)))(*words)
        at = ctypes.addressof(binds)
        arr = (_lib.ModelDispatch * max(1, n))()
        for i, (name, params, buffers, x, y) in enumerate(self._dispatches):
            text = _NAMES.get(name)
            if text is None:
                text = ctypes.create_string_buffer(name.encode())
                keep.append(text)
            _DISPATCH.pack_into(arr, i * _DISPATCH.size, ctypes.addressof(text), *params, at, len(buffers), x & 0xFFFFFFFF,
                                y & 0xFFFFFFFF)
            at += 24 * len(buffers)
        self._dispatches = []
        check(lib().bgtq_model_submit(self.ops.device.handle, arr, n))
        self.ops.device.synchronize()
