"""GPU: gradients under the clip threshold stay as they are, bit for bit, and gradients that
are not finite still reach every other one through the coefficient, as torch's clip does."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    yield torch.device("cuda", 0)
    from mi_adamw import clip
    clip._cache.clear()      # other tests count the tables of their own sizes


def _bits(t):
    return t.view(torch.int32).cpu()


@pytest.mark.parametrize("max_norm", [1.0, 1e30, float("inf")])
@pytest.mark.parametrize("special", [[], [0.0, -0.0, 1e-45, -1e-40], [float("inf")],
                                     [float("nan")], [-float("inf"), float("nan")]])
@pytest.mark.parametrize("step", [False, True])
def test_coefficient_of_one(dev, special, max_norm, step):
    import mi_adamw
    gen = torch.Generator(device=dev).manual_seed(5)
    grads = [torch.randn(n, device=dev, generator=gen) * 1e-4 for n in (3, 1025, 4099)]
    grads[1][:len(special)] = torch.tensor(special, device=dev)
    ours, ref = ([torch.nn.Parameter(torch.ones_like(g)) for g in grads] for _ in range(2))
    for q, r, g in zip(ours, ref, grads):
        q.grad, r.grad = g.clone(), g.clone()
    if step:
        opt = mi_adamw.FusedAdamW(ours, max_grad_norm=max_norm, clip_write_grads=True)
        opt.step()
        norm = opt.last_grad_norm
    else:
        norm = mi_adamw.clip_grad_norm_(ours, max_norm)
    torch.nn.utils.clip_grads_with_norm_(ref, max_norm, norm.clone())
    for q, r in zip(ours, ref):
        both = torch.isnan(q.grad) & torch.isnan(r.grad)
        assert torch.equal(torch.isnan(q.grad), torch.isnan(r.grad))
        assert torch.equal(_bits(q.grad.masked_fill(both, 0)), _bits(r.grad.masked_fill(both, 0)))


@pytest.mark.parametrize("below", [True, False])
def test_scale_at_the_two_group_rule(dev, below):
    """Sets on both sides of the size from which a lane of the scale pass takes two groups
    (80 Mi elements, counted in 4096-element chunks), with tensors that end around its tiles
    (2048 and 4096 elements) and begin off a 16-byte boundary: g * coef, one fp32 rounding."""
    import mi_adamw
    sizes = [1, 3, 2047, 2048, 2049, 2051, 4095, 4096, 4097, 6145, 8191]
    chunks = (80 << 20) // 4096 - sum(-(-n // 4096) for n in sizes) - (1 if below else 0)
    sizes.insert(5, chunks * 4096 - 1)
    block = torch.empty(sum(sizes), device=dev)
    block.normal_(0.0, 1e-2, generator=torch.Generator(device=dev).manual_seed(9))
    was = block.clone()
    params = []
    for g in block.split(sizes):
        params.append(torch.nn.Parameter(torch.empty_like(g)))
        params[-1].grad = g
    norm = mi_adamw.clip_grad_norm_(params, 1.0)
    exact = was.double().square().sum().sqrt().item()
    assert abs(norm.item() - exact) <= 2e-7 * exact      # one fp32 rounding of a float64 sum
    coef = (1.0 / (norm + 1e-6)).clamp(max=1.0)
    assert coef.item() < 1.0
    assert torch.equal(block, was * coef)
