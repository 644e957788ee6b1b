"""GPU: clip_grad_norm_ recorded into a HIP graph.  Every replay clips the gradients that the
graph was recorded with, bit for bit as torch's clip does with the same norm, whatever eager
calls, table evictions and allocations come between the replays."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = (1000, 4097, 3, 70000)


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    yield torch.device("cuda", 0)
    from mi_adamw import clip
    clip._cache.clear()      # other tests count the tables of their own sizes


def _params(dev, seed, sizes=SIZES):
    gen = torch.Generator(device=dev).manual_seed(seed)
    out = []
    for n in sizes:
        out.append(torch.nn.Parameter(torch.zeros(n, device=dev)))
        out[-1].grad = torch.randn(n, device=dev, generator=gen) * 1e-2
    return out


def _eager_work(dev, k):
    """Calls that move, evict and overwrite whatever was freed."""
    import mi_adamw
    from mi_adamw import clip
    mi_adamw.clip_grad_norm_(_params(dev, 50 + k), 1.0)
    if k % 2:
        clip._cache.clear()
    torch.cuda.synchronize()
    for _ in range(4):
        torch.full((1 << 12,), 0x7fffffff, dtype=torch.int32, device=dev)
    for n in (64 * len(SIZES), 1 << 15):
        torch.full((n,), 255, dtype=torch.uint8, device=dev)
        torch.full((n,), 255, dtype=torch.uint8).pin_memory().to(dev, non_blocking=True)
    torch.cuda.synchronize()


@pytest.mark.parametrize("warm", ["same stream", "another stream"])
@pytest.mark.parametrize("moved", [False, True])
def test_replays_clip_what_was_recorded(dev, warm, moved):
    import mi_adamw
    from mi_adamw import clip
    clip._cache.clear()
    stream = torch.cuda.Stream()
    params = _params(dev, 1)
    source = [torch.empty_like(p) for p in params]
    with torch.cuda.stream(torch.cuda.current_stream() if warm == "another stream" else stream):
        mi_adamw.clip_grad_norm_(params, 1.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for p, s in zip(params, source):
            if moved:
                p.grad = s * 1.0            # as a recorded backward leaves them
            else:
                p.grad.copy_(s)
        norm = mi_adamw.clip_grad_norm_(params, 1.0)
    grads = [p.grad for p in params]
    for k in range(5):
        gen = torch.Generator(device=dev).manual_seed(k)
        for s in source:
            s.normal_(0.0, 1e-2, generator=gen)
        _eager_work(dev, k)
        graph.replay()
        torch.cuda.synchronize()
        exact = sum(s.double().square().sum() for s in source).sqrt().item()
        assert abs(norm.item() - exact) <= 2e-7 * exact      # one fp32 rounding
        coef = (1.0 / (norm + 1e-6)).clamp(max=1.0)
        assert coef.item() < 1.0
        for g, s in zip(grads, source):
            assert torch.equal(g, s * coef)


def test_capture_without_an_eager_call_is_refused(dev):
    import mi_adamw
    from mi_adamw import clip
    clip._cache.clear()
    params = _params(dev, 1)
    mi_adamw.clip_grad_norm_(_params(dev, 2, SIZES[:3] + (SIZES[3] + 1,)), 1.0)
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="run one before capturing"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            mi_adamw.clip_grad_norm_(params, 1.0)
    norm = mi_adamw.clip_grad_norm_(params, 1.0)
    assert 0.0 < norm.item() < float("inf")
