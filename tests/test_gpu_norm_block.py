"""GPU: the clip's norm and coefficient, formed by the update itself up to 2^20 elements of
chunks and by a launch of its own above: both give the oracle's norm, and the step torch
takes with that norm, in both layouts, over replays of a recorded step too."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import max_ulp

pytestmark = pytest.mark.gpu

FOLD = 1 << 20


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    return torch.device("cuda", 0)


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("pre", [1.0, 0.125])
@pytest.mark.parametrize("sizes", [(1,), (4097, 5), (FOLD - 4096, 4096), (FOLD, 1),
                                   (FOLD + 1,)])
def test_norm_and_step_on_both_sides(dev, sizes, pre, flat):
    import mi_adamw
    from oracle import oracle as O
    gen = torch.Generator(device=dev).manual_seed(sum(sizes))
    values = [torch.randn(n, device=dev, generator=gen) for n in sizes]
    ours = [torch.nn.Parameter(v.clone()) for v in values]
    ref = [torch.nn.Parameter(v.clone()) for v in values]
    opt = mi_adamw.FusedAdamW(ours, lr=1e-2, max_grad_norm=0.5, grad_prescale=pre,
                              flat_buffer=flat)
    topt = torch.optim.AdamW(ref, lr=1e-2, foreach=False)
    for scale in (1.0, 1e-6):           # over and under the threshold
        grads = [torch.randn(n, device=dev, generator=gen) * scale for n in sizes]
        for q, r, g in zip(ours, ref, grads):
            if flat:
                q.grad.copy_(g)
            else:
                q.grad = g.clone()
            r.grad = g * pre
        opt.step()
        norm = np.float32(opt.last_grad_norm.item())
        assert norm == O.total_norm([r.grad.cpu().numpy() for r in ref])
        torch.nn.utils.clip_grads_with_norm_(ref, 0.5, opt.last_grad_norm.clone())
        topt.step()
        for q, r in zip(ours, ref):
            assert max_ulp(q, r) == 0
            assert max_ulp(opt.state[q]["exp_avg_sq"], topt.state[r]["exp_avg_sq"]) == 0


@pytest.mark.parametrize("n", [3000, FOLD + 4096])
def test_norm_of_a_recorded_step(dev, n):
    import mi_adamw
    from oracle import oracle as O
    p = torch.nn.Parameter(torch.randn(n, device=dev))
    p.grad = torch.randn(n, device=dev)
    opt = mi_adamw.FusedAdamW([p], lr=1e-2, max_grad_norm=0.5, capturable=True)
    opt.step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        opt.step()
    for k in range(3):
        p.grad.copy_(torch.randn(n, device=dev) * 10.0 ** -k)
        graph.replay()
        norm = np.float32(opt.last_grad_norm.item())
        assert norm == O.total_norm([p.grad.cpu().numpy()])
        (torch.ones(4096, device=dev) * 3).sum().item()     # other work between the replays


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sizes", [(3, 70), (5, 0, 4099), (300, 1) * 150, (FOLD, 4097)])
def test_device_step_counts_and_norm(dev, sizes, fused):
    """capturable=True: the launch before the update advances the counts (an empty tensor's,
    which has no row, apart), forms the rows and finishes the norm; more than 256 rows take
    several of its workgroups."""
    import mi_adamw
    gen = torch.Generator(device=dev).manual_seed(len(sizes))
    values = [torch.randn(n, device=dev, generator=gen) for n in sizes]
    ours = [torch.nn.Parameter(v.clone()) for v in values]
    ref = [torch.nn.Parameter(v.clone()) for v in values]
    hp = dict(lr=1e-2, capturable=True, fused=fused or None)
    opt = mi_adamw.FusedAdamW(ours, max_grad_norm=0.5, **hp)
    topt = torch.optim.AdamW(ref, foreach=None if fused else False, **hp)
    for k in range(4):
        for i, (q, r) in enumerate(zip(ours, ref)):
            g = torch.randn(q.numel(), device=dev, generator=gen)
            q.grad, r.grad = (g, g.clone()) if i or k != 2 else (None, None)
        opt.step()
        torch.nn.utils.clip_grads_with_norm_(ref, 0.5, opt.last_grad_norm.clone())
        topt.step()
        for q, r in zip(ours, ref):
            assert max_ulp(q, r) == 0
            assert float(opt.state[q]["step"]) == float(topt.state[r]["step"])
