"""Marshalling of path / signature arguments (pysiglib/data_handlers.py:50-189).

This package drives the GPU library only: NumPy inputs and CPU tensors are
rejected with a clear error instead of being routed to a CPU implementation.
"""
from ctypes import byref
from math import prod

import numpy as np
import torch

from ._loader import DTYPES
from .param_checks import check_array, check_dtype, own_contiguous


_NAMES = {torch.float32: "float32", torch.float64: "float64"}
_DTYPES = {name: dtype for dtype, name in _NAMES.items()}


def _pointer(tensor, dtype):
    """What the typed entry points take for the tensor's memory: ``byref`` of a view, a fifth of the cost of a ``cast``."""
    return byref(DTYPES[dtype].from_address(tensor.data_ptr()))


def _require_gpu(arr, name):
    if isinstance(arr, np.ndarray) or not arr.is_cuda:
        raise RuntimeError(
            name + " must be a torch tensor on the GPU: pysiglib_amd ships the MI355X path only and has no CPU "
            "implementation (use the reference's cpsig for host arrays).")


class PathInput:
    def __init__(self, path, time_aug, lead_lag, end_time, name="path"):
        check_array(path, name)
        self.path = own_contiguous(path)
        check_dtype(self.path, name)
        shape = tuple(self.path.shape)
        if len(shape) < 2:
            raise ValueError(name + " must have at least rank 2, got rank " + str(len(shape)) + ".")
        self.batch_shape = shape[:-2]
        self.batch_size = prod(self.batch_shape)
        self.data_length, self.data_dimension = shape[-2:]
        if self.data_dimension == 0:
            raise ValueError(name + " has 0 channels (dimension). Path dimension must be at least 1.")
        _require_gpu(self.path, name)
        self.type_ = "torch"
        self.dtype = _NAMES[self.path.dtype]
        self.device = self.path.device
        self.data_ptr = _pointer(self.path, self.dtype)
        self.time_aug, self.lead_lag, self.end_time = time_aug, lead_lag, end_time
        self.length = 2 * self.data_length - 1 if lead_lag else self.data_length
        self.dimension = (2 * self.data_dimension if lead_lag else self.data_dimension) + (1 if time_aug else 0)


class SigInput:
    """A signature-shaped input; a leading column is dropped when the input is one wider than expected."""

    def __init__(self, sig, sig_len, name):
        check_array(sig, name)
        self.sig = own_contiguous(sig)
        check_dtype(self.sig, name)
        shape = tuple(self.sig.shape)
        if len(shape) < 1:
            raise ValueError(name + " must have at least rank 1, got rank 0.")
        self.batch_shape = shape[:-1]
        self.batch_size = prod(self.batch_shape)
        length = shape[-1]
        if length == sig_len + 1:
            self.sig = own_contiguous(self.sig[..., 1:])
            length = sig_len
        if length != sig_len:
            raise ValueError(name + " is of incorrect length. Expected " + str(sig_len) + ", got " + str(length))
        _require_gpu(self.sig, name)
        self.type_ = "torch"
        self.dtype = _NAMES[self.sig.dtype]
        self.device = self.sig.device
        self.data_ptr = _pointer(self.sig, self.dtype)


def empty_like_input(data, shape):
    out = torch.empty((*data.batch_shape, *shape), dtype=_DTYPES[data.dtype], device=data.device)
    return out, _pointer(out, data.dtype)


class on_device:
    """``with on_device(dev):`` makes ``dev`` the current device for the C call; free when it already is."""

    def __init__(self, device):
        self.idx = device.index if device.index is not None else torch.cuda.current_device()
        self.prev = None

    def __enter__(self):
        cur = torch.cuda.current_device()
        if cur != self.idx:
            self.prev = cur
            torch.cuda.set_device(self.idx)
        return self

    def __exit__(self, *exc):
        if self.prev is not None:
            torch.cuda.set_device(self.prev)
        return False
