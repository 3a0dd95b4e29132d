"""Kernel adapter: the callable a kernel factory returns.

Mirrors the call contract of the reference's adapter for JIT kernels
(tilelang/jit/adapter/cython/cython_wrapper.pyx:164-287, tilelang/jit/kernel.py:195-211):

* ``kernel(*inputs)``; parameters listed in ``result_idx`` are allocated here with
  ``torch.empty`` on the first input's device and returned (``out_idx`` semantics);
* before the launch: argument count, device, dtype, shape, strides, contiguity are
  checked (``skip_tensor_validation=True`` skips them); errors are ``ValueError`` with
  the reference's wording;
* tensors are passed as raw ``data_ptr()``; ``None`` becomes a NULL pointer;
* the launch goes to torch's current stream unless ``stream=`` is given; it is
  asynchronous and never synchronises;
* a non-zero return code raises ``RuntimeError("Kernel call failed: <get_last_error()>")``.
"""

from __future__ import annotations

import contextlib
import ctypes
from dataclasses import dataclass
from typing import Callable, Sequence

import torch

from . import _lib


@dataclass(frozen=True)
class KernelParam:
    name: str
    dtype: torch.dtype
    shape: tuple
    #: packed sub-byte storage: the strict dtype check accepts int8 and uint8 alike
    packed: bool = False


#: torch's private call for the current stream of a GPU; None in a build of torch that has none
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def current_stream_handle(device_type: str = "cuda", index: int | None = None) -> int:
    """Raw handle of torch's current stream (tilelang/jit/adapter/cython/cython_wrapper.pyx:178-185).  ``index``: the
    GPU that an operand lies on, which the runtime then need not be asked for."""
    if device_type == "cuda" and (index is not None or torch.cuda.is_available()):
        if _raw_stream is not None:
            return _raw_stream(torch.cuda.current_device() if index is None else index)
        return torch.cuda.current_stream(index).cuda_stream
    return 0


def _unbound(*inputs):
    """Stands for a kernel object's native call until the first call binds it.  A function, which a copy of the object
    shares: the mark is told by identity."""
    return NotImplemented


class KernelAdapter:
    def __init__(
        self,
        name: str,
        params: Sequence[KernelParam],
        result_idx: Sequence[int],
        launch: Callable[[list, int], int],
        get_last_error: Callable[[], str],
        device_type: str = "cuda",
        workspace_idx: Sequence[int] = (),
        native: tuple | None = None,
    ):
        """``native``: ``(entry point, parameter per pointer argument (None: NULL), int arguments, float argument, workspace
        bytes)`` of the C call that ``launch`` makes, where that is all that it does; a good call then goes to it without
        passing through the interpreter's checks (csrc/host_call.cpp)."""
        self.name = name
        self.params = list(params)
        n = len(self.params)
        self.result_idx = [i if i >= 0 else n + i for i in result_idx]
        # parameters the kernel uses as scratch (the reference's T.alloc_buffer globals): allocated here for every
        # call, passed to the library, never returned.  torch's caching allocator hands a freed block back to the
        # stream it was allocated under only (__call__ allocates under the stream it launches on), so calls on
        # different streams never share a scratch buffer.
        self.workspace_idx = [i if i >= 0 else n + i for i in workspace_idx]
        self._launch = launch
        self._get_last_error = get_last_error
        self.device_type = device_type
        self._native_spec = native if device_type == "cuda" else None
        # bound by the first call: a kernel object that is only looked at, or made anew, pays for none
        self._native = _unbound if self._native_spec is not None else None
        self._native_new: dict = {}

    def __getstate__(self):
        # A native call is bound to the object that it was made for and cannot be copied: a copy binds its own.
        return {**self.__dict__, "_native": _unbound if self._native_spec is not None else None, "_native_new": {}}

    def _bind(self, result_idx):
        """The native call with the parameters of ``result_idx`` allocated by it; None where there is none."""
        host = _lib.host_call() if self._native_spec is not None and _raw_stream is not None and len(result_idx) <= 1 else None
        if host is None:
            return None
        entry, slots, ints, f, ws_bytes = self._native_spec
        roles = [2 if i in self.workspace_idx else 1 if i in result_idx else 0 for i in range(len(self.params))]
        return host.bind(entry, tuple((p.dtype, int(p.packed), tuple(p.shape), role) for p, role in zip(self.params, roles)),
                         tuple(-1 if i is None else i for i in slots), tuple(ints), float(f), ws_bytes)

    # -- validation, same order and wording as the reference ------------------------------
    def _check(self, tensors: list):
        # One look per tensor settles a good call; what it does not settle goes through the five passes below, which say
        # what is wrong.  (With __call__ asking the runtime for a GPU no more: W4A16 one row through a layer 23.9 -> 17.7
        # us, MXFP4 one row 19.6 -> 12.4.)  Contiguous with no dimension of zero is every stride as expected.
        device_type = self.device_type
        for p, t in zip(self.params, tensors):
            if isinstance(t, torch.Tensor) and not (
                t.device.type == device_type
                and (t.dtype == p.dtype or (p.packed and t.dtype in (torch.int8, torch.uint8)))
                and t.shape == p.shape and 0 not in p.shape and t.is_contiguous()
            ):
                break
        else:
            return
        for p, t in zip(self.params, tensors):
            if not isinstance(t, torch.Tensor):
                continue
            if t.device.type != self.device_type:
                raise ValueError(
                    f"Buffer device mismatch for parameter {p.name}: expected {self.device_type}, got {t.device}"
                )
        for p, t in zip(self.params, tensors):
            if not isinstance(t, torch.Tensor):
                continue
            ok = t.dtype == p.dtype or (p.packed and t.dtype in (torch.int8, torch.uint8))
            if not ok:
                raise ValueError(f"Buffer dtype mismatch for parameter {p.name}: expected {p.dtype}, got {t.dtype}")
        for p, t in zip(self.params, tensors):
            if not isinstance(t, torch.Tensor):
                continue
            if t.dim() != len(p.shape):
                raise ValueError(
                    f"Static shape mismatch for parameter {p.name}: expected {len(p.shape)} dimensions, got {t.dim()}"
                )
            for i, e in enumerate(p.shape):
                if e != -1 and t.shape[i] != e:
                    raise ValueError(
                        f"Static shape mismatch for parameter {p.name}: expected {e} at index {i}, got {t.shape[i]}"
                    )
        for p, t in zip(self.params, tensors):
            if not isinstance(t, torch.Tensor):
                continue
            expected = 1
            for i in range(len(p.shape) - 1, -1, -1):
                if t.shape[i] != 1 and t.stride(i) != expected:
                    raise ValueError(
                        f"Static stride mismatch for parameter {p.name}: expected {expected} at index {i}, got {t.stride(i)}"
                    )
                expected *= t.shape[i]
        for p, t in zip(self.params, tensors):
            if isinstance(t, torch.Tensor) and not t.is_contiguous():
                raise ValueError(f"Expected parameter {p.name} to be a contiguous tensor")

    def into_new(self, out_idx: int, *inputs):
        """``kernel(*inputs, out)`` for a kernel whose output, parameter ``out_idx`` and the last one that the caller
        brings, is the caller's: allocates it on the first input's device and returns it."""
        native = self._native_new.get(out_idx)
        if native is None and out_idx not in self._native_new:
            native = self._native_new[out_idx] = self._bind([out_idx])
        if native is not None:
            out = native(*inputs)
            if out is not NotImplemented:
                return out
        p = self.params[out_idx]
        out = torch.empty(p.shape, dtype=p.dtype, device=inputs[0].device)
        self(*inputs, out)
        return out

    def __call__(self, *inputs, stream: int = -1, skip_tensor_validation: bool = False):
        native = self._native
        if native is not None and stream == -1 and not skip_tensor_validation:
            if native is _unbound:
                native = self._native = self._bind(self.result_idx)
            out = native(*inputs) if native is not None else NotImplemented
            if out is not NotImplemented:
                return out
        n_params, n_in, n_out = len(self.params) - len(self.workspace_idx), len(inputs), len(self.result_idx)
        if n_params != n_in + n_out:
            raise ValueError(
                f"Expected {n_params} inputs, got {n_in + n_out} with {n_in} inputs and {n_out} outputs"
            )
        device = None
        for t in inputs:
            if isinstance(t, torch.Tensor):
                device = t.device
                break
        if device is None:
            device = torch.device(self.device_type)
        # a tensor on the GPU says that there is one and the runtime need not be asked
        has_cuda_input = device.type == "cuda" and device.index is not None
        on_gpu = has_cuda_input or (device.type == "cuda" and torch.cuda.is_available())
        # the library launches on the CURRENT device: make the operands' device current for the length of the call
        guard = contextlib.nullcontext()
        if on_gpu and device.index is not None and device.index != torch.cuda.current_device():
            guard = torch.cuda.device(device)
        with guard:
            if has_cuda_input and _raw_stream is not None and self.device_type == "cuda":
                current = _raw_stream(device.index)  # what the function below does, without its 0.1 us
            else:
                current = current_stream_handle(self.device_type, device.index if has_cuda_input else None)
            if stream == -1:
                stream = current
            # Outputs and scratch come from torch's caching allocator, which hands a freed block back to work on
            # the stream it was allocated under only.  With an explicit stream= that is not torch's current one,
            # allocate under that stream, so that a block freed while this launch still runs cannot go to an op on
            # another stream.
            alloc_ctx = contextlib.nullcontext()
            if on_gpu and stream != current and (self.result_idx or self.workspace_idx):
                alloc_ctx = torch.cuda.stream(torch.cuda.ExternalStream(stream, device=device))
            tensors, it = [], iter(inputs)
            with alloc_ctx:
                for i, p in enumerate(self.params):
                    if i in self.workspace_idx or i in self.result_idx:
                        tensors.append(torch.empty(*p.shape, dtype=p.dtype, device=device))
                    else:
                        tensors.append(next(it))
            return self._run(tensors, stream, skip_tensor_validation, n_out)

    def _run(self, tensors, stream, skip_tensor_validation, n_out):
        ptrs = []
        for t in tensors:
            if isinstance(t, torch.Tensor):
                ptrs.append(ctypes.c_void_p(t.data_ptr()))
            elif t is None:
                ptrs.append(ctypes.c_void_p(0))
            elif isinstance(t, int):
                ptrs.append(ctypes.c_void_p(t))
            else:
                raise ValueError(f"Unsupported tensor type: {type(t)}")

        if not skip_tensor_validation:
            self._check(tensors)

        rc = self._launch(ptrs, stream)
        if rc != 0:
            raise RuntimeError(f"Kernel call failed: {self._get_last_error()}")

        if n_out == 0:
            return None
        if n_out == 1:
            return tensors[self.result_idx[0]]
        return [tensors[i] for i in self.result_idx]

    # conveniences mirroring tilelang/jit/kernel.py:494-520
    def get_profiler(self, tensor_supply_type=None):
        from .profiler import Profiler, TensorSupplyType

        return Profiler(self, tensor_supply_type or TensorSupplyType.Auto)
