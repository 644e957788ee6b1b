"""clip_grad_norm_: drop-in for torch.nn.utils.clip_grad_norm_ on the MI355X kernels.

mini-megatron names the clip value (config.py:16, MAX_GRAD_NORM = 1.0); the
standard way to apply it in its loop is ``torch.nn.utils.clip_grad_norm_``
between ``loss.backward()`` and ``optimizer.step()`` (main.py:207-209).  This
function keeps that signature and result: the global L2 norm of every gradient
as one vector (torch/nn/utils/clip_grad.py:50-117), then
``g *= min(max_norm / (norm + 1e-6), 1)`` in place (clip_grad.py:121-183).
Three launches: the float64 sum-of-squares pass, a one-workgroup finalize (norm
and coefficient, on the device) and an in-place scale pass, which leaves the
gradients alone where the coefficient is 1.  Use
``FusedAdamW(max_grad_norm=...)`` instead to fold the scale into the step.
"""
from __future__ import annotations

import threading

import numpy as np
import torch

from . import _lib
from .optimizer import _ROW_DTYPE, _Launch

_CHUNK = 4096
_cache: dict[tuple, _ClipLaunch] = {}
# what graphs hold the addresses of (_recorded_tables): a graph's end is not announced, so
# these stay, 64 bytes per gradient and 8 per 4096 elements of each recorded set of tables
_kept: list = []


class _ClipLaunch(_Launch):
    """The tables of one list of sizes on one stream, with the scratch its passes write.
    Calls on different streams may overlap and share neither.  Calls of several threads on
    one stream share both, so one of them at a time points the tables at its gradients and
    launches its passes (`lock`)."""

    __slots__ = ("stream", "lock", "partials", "coef", "recorded", "kept")

    def __init__(self, rows: np.ndarray, device: torch.device, stream: int):
        super().__init__(rows, _CHUNK, device, tables=True)
        self.stream = stream
        self.recorded = False       # a graph reads the rows, which then never change
        self.kept = None            # the rows that _kept holds
        self.lock = threading.Lock()
        self.partials = torch.zeros(_lib.MAX_NORM_BLOCKS, dtype=torch.float64, device=device)
        self.coef = torch.zeros(1, dtype=torch.float32, device=device)


def _tables(grads, device, stream: int) -> _ClipLaunch:
    """The tables for gradients of these sizes, cached per stream (so that they are allocated
    on the stream whose launches read them, and a replaced or dropped table returns to that
    stream's pool, ordered after those launches).  Cached tables may point at another call's
    gradients of the same sizes: _run moves them."""
    rows = np.zeros(len(grads), dtype=_ROW_DTYPE)
    ptrs = np.array([g.data_ptr() for g in grads], dtype=np.uint64)
    # Only the gradient pointer is read by the norm and scale kernels.
    rows["param"] = ptrs
    rows["grad"] = ptrs
    rows["numel"] = [g.numel() * (2 if torch.is_complex(g) else 1) for g in grads]
    rows["flags"] = np.where(ptrs % 16 == 0, _lib.T_VEC, 0)
    rows = rows[rows["numel"] > 0]
    key = (device, stream, rows["numel"].tobytes())
    launch = _cache.get(key)
    if launch is None and device.type == "cuda" and torch.cuda.is_current_stream_capturing():
        # another stream's tables serve (_recorded_tables); an upload cannot be recorded
        for (dev, _, numels), other in list(_cache.items()):
            if dev == device and numels == key[2]:
                return other
        raise RuntimeError("mi_adamw.clip_grad_norm_ under graph capture, but no eager call has "
                           "had gradients of these sizes; run one before capturing")
    if launch is None:
        launch = _ClipLaunch(rows, device, stream)
        if len(_cache) > 8:
            _cache.clear()
        _cache[key] = launch
    return launch


def _patch(table: torch.Tensor, n_rows: int, idx: np.ndarray, grads: np.ndarray, device) -> int:
    """New gradient addresses for the rows idx of a device table, carried there as kernel
    arguments; the library's code."""
    grads = np.ascontiguousarray(grads)
    vec = (grads % 16 == 0).astype(np.uint8)
    return _lib.load().mi_adamw_set_grads(
        table.data_ptr(), n_rows, len(idx), idx.ctypes.data, grads.ctypes.data, vec.ctypes.data,
        torch._C._cuda_getCurrentRawStream(device.index))


def _recorded_tables(launch, ptrs: bytes, device, stream: int):
    """(rows, partial sums, coefficient) for a call that a graph records.  The rows are the
    launch's where they are this stream's and say where the gradients are; they and the chunk
    table then stay as they are for good.  Otherwise the graph makes its own, a copy of the
    launch's with the addresses patched, at each replay: memory of the graph's pool, as the
    scratch is, which replays and eager calls of the stream would otherwise share."""
    if launch.kept is not launch.rows:
        _kept.append((launch.rows, launch.chunks))
        launch.kept = launch.rows
    rows = launch.rows
    if launch.stream == stream and ptrs == launch.host_rows["grad"].tobytes():
        launch.recorded = True
    else:
        rows = rows.clone()
        _lib.check(_patch(rows, launch.n_rows, np.arange(launch.n_rows, dtype=np.int32),
                          np.frombuffer(ptrs, dtype=np.uint64), device), "mi_adamw_set_grads")
    return (rows, torch.empty_like(launch.partials), torch.empty_like(launch.coef))


def _move(launch, ptrs: bytes, device) -> None:
    """The gradients lie elsewhere than the launch's table says: the table is patched in
    place (it belongs to one stream), or replaced if a graph reads it."""
    grads = np.frombuffer(ptrs, dtype=np.uint64)
    rows = launch.host_rows.copy()
    idx = np.flatnonzero(grads != rows["grad"]).astype(np.int32)
    rows["param"] = rows["grad"] = grads
    rows["flags"] = np.where(grads % 16 == 0, _lib.T_VEC, 0)
    if launch.recorded:
        launch.set_rows(rows, device)
        launch.recorded = False
        return
    code = _patch(launch.rows, launch.n_rows, idx, grads[idx], device)
    if code != _lib.OK:
        launch.host_rows["grad"] = 0    # the device table may hold part of the patch
    _lib.check(code, "mi_adamw_set_grads")
    launch.host_rows = rows


def _run(launch, ptrs: bytes, device, stream: int, max_norm: float, norm_type: float,
         error_if_nonfinite: bool) -> torch.Tensor:
    """The norm and scale passes over a launch's tables; `ptrs`: where the gradients are."""
    if torch._C._cuda_getDevice() != device.index:
        with torch.cuda.device(device):
            return _run(launch, ptrs, device, stream, max_norm, norm_type, error_if_nonfinite)
    with launch.lock:
        if torch._C._cuda_isCurrentStreamCapturing():
            rows, partials, coef = _recorded_tables(launch, ptrs, device, stream)
        else:
            if ptrs != launch.host_rows["grad"].tobytes():
                _move(launch, ptrs, device)
            rows, partials, coef = launch.rows, launch.partials, launch.coef
        lib = _lib.load()
        norm = torch.empty((), dtype=torch.float32, device=device)
        _lib.check(lib.mi_adamw_grad_norm(
            rows.data_ptr(), launch.chunks.data_ptr(), launch.n_chunks, _CHUNK,
            float(max_norm), partials.data_ptr(), norm.data_ptr(),
            coef.data_ptr(), stream), "mi_adamw_grad_norm")
        if error_if_nonfinite and bool(torch.logical_or(norm.isnan(), norm.isinf())):
            raise RuntimeError(
                f"The total norm of order {float(norm_type)} for gradients from "
                "`parameters` is non-finite, so it cannot be clipped. To disable "
                "this error and scale the gradients by the non-finite norm anyway, "
                "set `error_if_nonfinite=False`")
        _lib.check(lib.mi_adamw_scale_grads(
            rows.data_ptr(), launch.chunks.data_ptr(), launch.n_chunks, _CHUNK,
            coef.data_ptr(), stream), "mi_adamw_scale_grads")
        return norm


@torch.no_grad()
def clip_grad_norm_(parameters, max_norm: float, norm_type: float = 2.0,
                    error_if_nonfinite: bool = False, foreach: bool | None = None) -> torch.Tensor:
    """Clip the global gradient norm in place; returns the total norm (0-d tensor)."""
    parameters = [parameters] if isinstance(parameters, torch.Tensor) else list(parameters)
    if _lib._host is not None and float(norm_type) == 2.0:
        found = _lib._host.grads(parameters, torch.Tensor, torch.nn.Parameter)
        if found is not None:
            index, numels, ptrs = found
            stream = torch._C._cuda_getCurrentRawStream(index)
            device = torch.device("cuda", index)
            launch = _cache.get((device, stream, numels))
            if launch is not None:
                return _run(launch, ptrs, device, stream, max_norm, norm_type,
                            error_if_nonfinite)
    grads = [p.grad for p in parameters if p.grad is not None]
    if float(norm_type) != 2.0:
        raise NotImplementedError("mi_adamw.clip_grad_norm_ supports norm_type=2 only")
    if len(grads) == 0:
        return torch.tensor(0.0)
    device = grads[0].device
    for g in grads:
        if g.device != device or g.device.type != "cuda":
            raise RuntimeError("mi_adamw.clip_grad_norm_ needs every gradient on one ROCm GPU")
        if g.dtype not in (torch.float32, torch.complex64) or not g.is_contiguous() or g.is_sparse:
            raise NotImplementedError("mi_adamw.clip_grad_norm_ supports dense contiguous fp32 "
                                      "gradients only")
    _lib.load()
    with torch.cuda.device(device):
        stream = torch.cuda.current_stream(device).cuda_stream
        launch = _tables(grads, device, stream)
        if launch.n_chunks == 0:
            return torch.zeros((), dtype=torch.float32, device=device)
    ptrs = np.array([g.data_ptr() for g in grads if g.numel()], dtype=np.uint64).tobytes()
    return _run(launch, ptrs, device, stream, max_norm, norm_type, error_if_nonfinite)
