"""GPU: every element is stepped exactly once whatever order its tile is taken in.

Work items (1024-element tiles) are taken in runs per XCD within groups of 1024 items, in
plain order past the last full group; a chunk has chunk_elems / 1024 of them, also where
that is no power of two; a capped grid takes several per workgroup.  Sizes sit around a
group's edge.  An element left out or stepped twice differs from torch's step.
"""
from __future__ import annotations

import pytest
import torch

from _helpers import max_ulp

pytestmark = pytest.mark.gpu

GROUP = 1024 * 1024      # elements of one full group of tiles


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    return torch.device("cuda", 0)


@pytest.mark.parametrize("max_blocks", [0, 7, 1025])
@pytest.mark.parametrize("chunk", [4096, 12288, 65536])
@pytest.mark.parametrize("sizes", [(GROUP - 1,), (GROUP + 4,), (GROUP - 4096, 5, 4091, 3),
                                   (3 * GROUP + 1025, 7, 1023)])
def test_each_element_steps_once(dev, sizes, chunk, max_blocks):
    import mi_adamw
    gen = torch.Generator(device=dev).manual_seed(len(sizes) + chunk)
    values = [torch.randn(n, device=dev, generator=gen) for n in sizes]
    ours = [torch.nn.Parameter(v.clone()) for v in values]
    ref = [torch.nn.Parameter(v.clone()) for v in values]
    for q, r in zip(ours, ref):
        q.grad = torch.randn(q.numel(), device=dev, generator=gen)
        r.grad = q.grad.clone()
    opt = mi_adamw.FusedAdamW(ours, lr=1e-2, chunk_elems=chunk)
    opt.max_blocks = max_blocks
    topt = torch.optim.AdamW(ref, lr=1e-2, foreach=False)
    for _ in range(2):
        opt.step()
        topt.step()
    torch.cuda.synchronize()
    for q, r in zip(ours, ref):
        assert max_ulp(q, r) == 0
        for key in ("exp_avg", "exp_avg_sq"):
            assert max_ulp(opt.state[q][key], topt.state[r][key]) == 0
