"""The passes' work items and grids (csrc/items.h) on the host: tests/c/items_check, built by
__graft_entry__.build()."""
from __future__ import annotations

import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "c", "items_check")


def test_items_cover_and_bounds_count_lanes():
    if not os.path.exists(BIN):
        pytest.fail(f"{BIN} is not built; run __graft_entry__.build() first")
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "items_check: ok" in r.stdout, r.stdout + r.stderr
