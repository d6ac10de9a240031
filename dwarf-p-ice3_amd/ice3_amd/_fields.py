"""Array plumbing shared by the drop-in components: layout checks and pointers."""
from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import _lib


def as_columns(x, layout: str, *, device, name: str) -> torch.Tensor:
    """Return a contiguous float64 CUDA tensor of shape (nlev, ncol).

    layout "columns": x is (nlev, ncol) with columns contiguous, the reference's
    Fortran (NIJT, NKT) memory (no copy when already float64 on the device).
    layout "jax": x has the JAX components' (..., nz) shape, vertical index last;
    it is transposed to (nz, ncol).
    """
    t = torch.as_tensor(x, dtype=torch.float64, device=device)
    if layout == "columns":
        if t.dim() != 2:
            raise ValueError(f"{name}: expected a (nlev, ncol) array, got {tuple(t.shape)}")
        return t.contiguous()
    if t.dim() < 2:
        raise ValueError(f"{name}: expected a (..., nz) array, got {tuple(t.shape)}")
    return t.reshape(-1, t.shape[-1]).t().contiguous()


def device_tensor(x, device) -> torch.Tensor:
    """x as a float64 tensor on the device (a tensor that is one already passes a check only)."""
    if type(x) is torch.Tensor and x.dtype is torch.float64 and x.device == device:
        return x
    return torch.as_tensor(x, dtype=torch.float64, device=device)


def columns_of(fields: dict, layout: str, *, device):
    """as_columns of every field of a call, and the names of those that are fresh copies (the
    others share the caller's memory).  "jax" fields whose memory is (..., nz) in order are
    transposed together, one launch for each shape among them."""
    out, fresh, batches = {}, set(), {}
    if layout == "columns":
        f64, tensor = torch.float64, torch.Tensor
        for k, x in fields.items():
            if type(x) is tensor and x.dtype is f64 and x.device == device and x.dim() == 2 and x.is_contiguous():
                out[k] = x
                continue
            t = device_tensor(x, device)
            out[k] = as_columns(t, layout, device=device, name=k)
            if out[k].data_ptr() != t.data_ptr():
                fresh.add(k)
        return out, fresh
    for k, x in fields.items():
        t = device_tensor(x, device)
        if t.dim() < 2:
            raise ValueError(f"{k}: expected a (..., nz) array, got {tuple(t.shape)}")
        v = t.reshape(-1, t.shape[-1])
        c = v.t()
        if not c.is_contiguous():
            # (below 2^28 either way ice3_transpose_fields' tiles, 32 by 128, fit its launch)
            if t.is_contiguous() and t.is_cuda and max(v.shape) < 2 ** 28:
                batches.setdefault(tuple(v.shape), []).append((k, v))
                out[k] = None  # keeps the order of the names
                continue
            c = c.contiguous()
        out[k] = c
        if c.data_ptr() != t.data_ptr():
            fresh.add(k)
    for (rows, cols), items in batches.items():
        for i in range(0, len(items), _lib.ICE3_MAX_CHECK_FIELDS):
            part = items[i:i + _lib.ICE3_MAX_CHECK_FIELDS]
            new = [torch.empty((cols, rows), dtype=torch.float64, device=device) for _ in part]
            arr = ctypes.c_void_p * len(part)
            with torch.cuda.device(device):
                _lib.check(_lib.load().ice3_transpose_fields(
                    len(part), arr(*[v.data_ptr() for _, v in part]), arr(*[n.data_ptr() for n in new]), rows, cols,
                    stream_ptr(device)), "ice3_transpose_fields")
            for (k, _), n in zip(part, new):
                out[k] = n
                fresh.add(k)
    return out, fresh


def column_shape(x, layout: str, name: str, *, device) -> tuple:
    """The (nlev, ncol) shape as_columns(x) would have, without making it, of a field that no kernel
    reads.  What as_columns refuses (a type, a dtype, strides or a device that it cannot convert) is
    refused here too: an array is converted as far as the host goes, anything else altogether."""
    if type(x) is not torch.Tensor or x.layout is not torch.strided or x.is_quantized or not (x.is_cuda or x.is_cpu):
        if not isinstance(x, np.ndarray):
            return tuple(as_columns(x, layout, device=device, name=name).shape)
        x = torch.as_tensor(x, dtype=torch.float64)
    shape = tuple(x.shape)
    if layout == "columns":
        if len(shape) != 2:
            raise ValueError(f"{name}: expected a (nlev, ncol) array, got {shape}")
        return shape
    if len(shape) < 2:
        raise ValueError(f"{name}: expected a (..., nz) array, got {shape}")
    n = 1
    for d in shape[:-1]:
        n *= d
    return shape[-1], n


def in_rows(fields: dict) -> bool:
    """Whether "jax" layout fields (device float64 tensors) are better taken as (ncol, nlev) rows,
    the vertical contiguous, than as (nlev, ncol) columns: True unless more of them already have
    the columns' memory order (results of a columns call are such views) than the rows'.  Looks at
    no more of them than decides it."""
    others = [t for t in fields.values() if not t.is_contiguous()]
    lead = len(fields) - 2 * len(others)  # of the rows, if all the others are in the columns' order
    if lead >= 0:
        return True
    score = len(fields) - len(others)
    for t in others:
        if t.dim() >= 2 and t.movedim(-1, 0).is_contiguous():
            score -= 1
            if score < 0:
                return False
    return True


def as_rows(t: torch.Tensor, name: str) -> torch.Tensor:
    """A "jax" layout device tensor as contiguous (ncol, nlev) rows (no copy when it is)."""
    if t.dim() < 2:
        raise ValueError(f"{name}: expected a (..., nz) array, got {tuple(t.shape)}")
    return t.reshape(-1, t.shape[-1]).contiguous()


def from_columns(t: torch.Tensor, layout: str, shape) -> torch.Tensor:
    """Inverse of as_columns for results: a (nlev, ncol) field back to ``shape``, or a
    per-column (ncol,) result to ``shape[:-1]`` (the JAX layout without its vertical axis)."""
    if layout == "columns":
        return t
    if t.dim() == 1:
        return t.reshape(tuple(shape[:-1]))
    return t.t().reshape(shape)


LAYOUTS = ("auto", "columns", "jax")


def check_layout(layout: str) -> str:
    if layout not in LAYOUTS:
        raise ValueError(f"layout must be one of {LAYOUTS}, got {layout!r}")
    return layout


def resolve_layout(layout: str, x) -> str:
    """The layout of one call: "auto" reads it from the array rank of ``x`` (a field of the
    call): three or more dimensions are the JAX components' (nx, ny, nz) /
    (ngpblks, nproma, nflevg) arrays, vertical index last; two are the Fortran
    (nlev, ncol) memory, columns contiguous."""
    if layout != "auto":
        return layout
    nd = getattr(x, "ndim", None)
    if nd is None:
        nd = torch.as_tensor(x).dim()
    return "jax" if nd >= 3 else "columns"


def ptr(t) -> ctypes.c_void_p:
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(None)


def addresses(tensors) -> list:
    """The device addresses of tensors (None: 0) as integers, which a struct of pointers takes as
    they are (without an object for each)."""
    return [t.data_ptr() if t is not None else 0 for t in tensors]


def new_fields(names, shape, device) -> dict:
    """Uninitialised float64 fields of one shape, each with memory of its own (a torch.empty_like
    takes 1.2 us, a torch.empty 1.7)."""
    names = iter(names)
    first = torch.empty(shape, dtype=torch.float64, device=device)
    out = {next(names): first}
    for k in names:
        out[k] = torch.empty_like(first)
    return out


def stream_ptr(device) -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
