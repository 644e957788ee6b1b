"""clip_grad_norm_'s tables on the CPU: what a graph has recorded stays as it was and stays
alive, whatever later calls do.  The passes are stand-ins that note the table they were given
and the addresses in it, and mi_adamw_set_grads one that patches a host table."""
from __future__ import annotations

import ctypes
import gc
import types
import weakref

import numpy as np
import pytest
import torch

from mi_adamw import _lib, clip
from mi_adamw.optimizer import _ROW_DTYPE

CPU = torch.device("cpu")
SIZES = (10, 4097, 5)


class _Passes:
    """The library with its launches replaced; `seen`: (table address, gradient addresses,
    scratch addresses) of each norm pass."""

    def __init__(self):
        real = _lib.load()
        self.seen = []
        self.lib = types.SimpleNamespace(
            mi_adamw_build_chunks=real.mi_adamw_build_chunks, mi_adamw_grad_norm=self._norm,
            mi_adamw_scale_grads=self._scale, mi_adamw_set_grads=self._set)

    @staticmethod
    def rows(table):
        buf = (ctypes.c_char * (64 * len(SIZES))).from_address(table)
        return np.frombuffer(buf, dtype=_ROW_DTYPE)

    def _norm(self, table, chunks, n_chunks, chunk, max_norm, partials, norm, coef, stream):
        assert n_chunks == 4
        rows = self.rows(table)
        assert rows["numel"].tolist() == list(SIZES)
        self.seen.append((table, rows["grad"].tolist(), (partials, coef)))
        return 0

    def _scale(self, table, chunks, n_chunks, chunk, coef, stream):
        assert (table, coef) == (self.seen[-1][0], self.seen[-1][2][1])
        return 0

    def _set(self, table, n_rows, n, idx, grads, vec, stream):
        assert n_rows == len(SIZES)
        at = np.ctypeslib.as_array(ctypes.cast(idx, ctypes.POINTER(ctypes.c_int32)), (n,))
        new = np.ctypeslib.as_array(ctypes.cast(grads, ctypes.POINTER(ctypes.c_uint64)), (n,))
        self.rows(table)["grad"][at] = new
        return 0


@pytest.fixture
def passes(monkeypatch):
    p = _Passes()
    p.capturing = False
    monkeypatch.setattr(_lib, "load", lambda: p.lib)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 0, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_isCurrentStreamCapturing", lambda: p.capturing,
                        raising=False)
    clip._cache.clear()
    del clip._kept[:]
    yield p
    clip._cache.clear()
    del clip._kept[:]


def _grads():
    return [torch.zeros(n) for n in SIZES]


def _call(p, grads, stream=0, capturing=False):
    launch = clip._tables(grads, CPU, stream)
    ptrs = [g.data_ptr() for g in grads]
    p.capturing = capturing
    clip._run(launch, np.array(ptrs, dtype=np.uint64).tobytes(), CPU, stream, 1.0, 2.0, False)
    p.capturing = False
    assert p.seen[-1][1] == ptrs
    return launch


def test_recorded_tables_are_never_written_nor_freed(passes):
    a, b, c = _grads(), _grads(), _grads()
    launch = _call(passes, a)
    scratch = passes.seen[-1][2]
    _call(passes, a, capturing=True)
    table = passes.seen[-1][0]
    assert table == launch.rows.data_ptr()               # where they are: no work of the graph's
    assert not set(passes.seen[-1][2]) & set(scratch)    # scratch of its own
    kept = [weakref.ref(launch.rows), weakref.ref(launch.chunks)]
    _call(passes, b)                                     # an eager call, gradients elsewhere
    assert passes.seen[-1][0] != table
    _call(passes, c)
    clip._cache.clear()
    del launch
    gc.collect()
    assert all(r() is not None for r in kept)
    assert _Passes.rows(table)["grad"].tolist() == [g.data_ptr() for g in a]


def test_gradients_that_moved_under_capture_get_a_table_of_the_graph(passes):
    a, b = _grads(), _grads()
    launch = _call(passes, a)
    for grads, stream in ((b, 0), (a, 7), (b, 7)):       # moved, another stream, both
        clip._cache[(CPU, stream) + next(iter(clip._cache))[2:]] = launch
        n = len(clip._kept)
        _call(passes, grads, stream=stream, capturing=True)
        assert passes.seen[-1][0] != launch.rows.data_ptr()
        assert len(clip._kept) == max(n, 1)              # the source, once
    assert launch.host_rows["grad"].tolist() == [g.data_ptr() for g in a]
    assert _Passes.rows(launch.rows.data_ptr())["grad"].tolist() == [g.data_ptr() for g in a]
    _call(passes, b)                                     # still patched in place
    assert passes.seen[-1][0] == launch.rows.data_ptr()


def test_a_failed_patch_leaves_no_address_trusted(passes):
    a, b = _grads(), _grads()
    launch = _call(passes, a)
    real = passes.lib.mi_adamw_set_grads
    passes.lib.mi_adamw_set_grads = lambda *args: 1
    passes.lib.mi_adamw_strerror = lambda code: b"injected"
    with pytest.raises(_lib.MiAdamwError):
        clip._run(launch, np.array([g.data_ptr() for g in b], np.uint64).tobytes(), CPU, 0, 1.0,
                  2.0, False)
    passes.lib.mi_adamw_set_grads = real
    _Passes.rows(launch.rows.data_ptr())["grad"][1] = b[1].data_ptr()    # half of the patch
    _call(passes, a)
