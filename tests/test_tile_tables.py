"""Which sets an update gets a table of tiles for, and what is in it (CPU: no launch)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from mi_adamw import _lib
from mi_adamw.optimizer import _ROW_DTYPE, _Launch


def _launch(sizes, chunk, **kw):
    rows = np.zeros(len(sizes), dtype=_ROW_DTYPE)
    rows["numel"] = sizes
    return _Launch(rows, chunk, torch.device("cpu"), tables=True, **kw)


@pytest.mark.parametrize("sizes,chunk,tiles", [
    ([768] * 2000, 4096, True), ([768] * 300, 65536, True), ([1] * 100, 1 << 20, True),
    ([768] * 50, 4096, False), ([4096] * 2000, 4096, False),
    ([3 * 768 * 768, 768, 768 * 768] * 12, 4096, False),
    ([3 * 768 * 768, 768, 768 * 768] * 12, 65536, False),
    ([1 << 20] * 4 + [1], 1 << 20, False), ([4096 * 300 + 1] * 3, 4096, False)])
def test_which_sets_have_tiles(sizes, chunk, tiles):
    launch = _launch(sizes, chunk, update=True)
    groups = launch.n_items * (1 if tiles else chunk // _lib.TILE_ELEMS)
    exact = sum(-(-n // _lib.TILE_ELEMS) for n in sizes)
    assert (launch.item_flag == _lib.F_TILES) == tiles
    assert groups <= max(1.25 * exact, exact + 256)      # workgroups, whatever the chunk size
    if not tiles:
        assert launch.items is launch.chunks and launch.n_items == launch.n_chunks
    # the norm pass keeps its chunks: the order of its sums does not depend on this
    assert launch.n_chunks == sum(-(-n // chunk) for n in sizes)


def test_tiles_cover_every_tensor_in_order():
    sizes = [1, 1023, 1024, 1025, 4097] + [3] * 300
    launch = _launch(sizes, 4096, update=True)
    table = np.frombuffer(launch.items.numpy().tobytes(), dtype=np.int32).reshape(-1, 2)
    want = [(t, k) for t, n in enumerate(sizes) for k in range(-(-n // 1024))]
    assert table.tolist() == [list(w) for w in want] and launch.n_items == len(want)
    assert _launch(sizes, 4096).item_flag == 0           # tables that only a norm pass reads
