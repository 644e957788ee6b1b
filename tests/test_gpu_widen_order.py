"""GPU: the widen pass writes every element once and nothing else, whatever order its tiles
are taken in: plain below 256 tiles of 2048 elements, in runs per XCD within each full 256,
plain past the last; chunks of one and of several tiles, sources and destinations off their
vector boundaries.  A float32 of a bfloat16 is exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GROUP = 256 * 2048       # elements of one full group of tiles
POISON = -12345.0


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    return torch.device("cuda", 0)


@pytest.mark.parametrize("chunk", [4096, 12288])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("sizes", [(GROUP - 4096,), (GROUP - 2049,), (GROUP,), (GROUP + 1,),
                                   (GROUP - 8192, 5, 4091, 3), (3 * GROUP + 2049, 7, 2047, 1)])
def test_each_element_once(dev, sizes, chunk, offset):
    from mi_adamw import _lib
    from mi_adamw.optimizer import _ROW_DTYPE, _Launch
    gap = 8
    total = offset + sum(n + gap for n in sizes)
    gen = torch.Generator(device=dev).manual_seed(total + chunk)
    src = torch.randn(total, device=dev, generator=gen).to(torch.bfloat16)
    dst = torch.full((total,), POISON, device=dev)
    want = dst.clone()
    rows = np.zeros(len(sizes), dtype=_ROW_DTYPE)
    at = offset
    for i, n in enumerate(sizes):
        rows[i]["param"] = dst[at:].data_ptr()
        rows[i]["param_copy"] = src[at:].data_ptr()
        rows[i]["numel"] = n
        want[at:at + n] = src[at:at + n].float()
        at += n + gap
    launch = _Launch(rows, chunk, dev, tables=True)
    _lib.check(_lib.load().mi_adamw_widen_bf16(
        launch.rows.data_ptr(), launch.chunks.data_ptr(), launch.n_chunks, chunk,
        torch.cuda.current_stream(dev).cuda_stream), "mi_adamw_widen_bf16")
    assert torch.equal(dst, want)
