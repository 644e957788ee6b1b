"""GPU: clip_grad_norm_ from two threads that share a stream and a list of sizes, and so one
set of tables: each call clips its own gradients and returns their norm, wherever the other
thread's call falls between looking the tables up and launching the passes."""
from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = (1000, 4097, 3)


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    yield torch.device("cuda", 0)
    from mi_adamw import clip
    clip._cache.clear()      # other tests count the tables of their own sizes


def _params(dev, seed, std):
    gen = torch.Generator(device=dev).manual_seed(seed)
    out = []
    for n in SIZES:
        out.append(torch.nn.Parameter(torch.zeros(n, device=dev)))
        out[-1].grad = torch.randn(n, device=dev, generator=gen) * std
    return out


@pytest.mark.parametrize("cached", [False, True])
def test_a_call_between_another_calls_tables_and_passes(dev, monkeypatch, cached):
    import mi_adamw
    from mi_adamw import _lib, clip
    _lib.load()
    clip._cache.clear()
    if cached:
        mi_adamw.clip_grad_norm_(_params(dev, 1, 1e-2), 1e-3)
    mine, other = _params(dev, 2, 1e-2), _params(dev, 3, 2e-2)
    was = [[p.grad.clone() for p in ps] for ps in (mine, other)]
    real, norms = clip._tables, {}

    def interrupted(*args):
        launch = real(*args)
        monkeypatch.setattr(clip, "_tables", real)

        def call():
            norms["other"] = mi_adamw.clip_grad_norm_(other, 1e-3)
        t = threading.Thread(target=call)
        t.start()
        t.join(60)
        assert not t.is_alive()
        return launch

    monkeypatch.setattr(clip, "_tables", interrupted)
    # the native gather left out, so that the first call goes through _tables
    monkeypatch.setattr(_lib, "_host", None)
    norms["mine"] = mi_adamw.clip_grad_norm_(mine, 1e-3)
    for ps, grads, norm in ((mine, was[0], norms["mine"]), (other, was[1], norms["other"])):
        exact = sum(g.double().square().sum() for g in grads).sqrt().item()
        assert abs(norm.item() - exact) <= 2e-7 * exact      # one fp32 rounding
        coef = (1.0 / (norm + 1e-6)) * 1e-3
        for p, g in zip(ps, grads):
            assert torch.equal(p.grad, g * coef)


def test_two_threads_many_calls(dev):
    import mi_adamw
    stream = torch.cuda.current_stream()
    failures = []

    def work(seed):
        try:
            with torch.cuda.stream(stream):
                for k in range(50):
                    ps = _params(dev, 100 * seed + k, 1e-2)
                    was = [p.grad.clone() for p in ps]
                    norm = mi_adamw.clip_grad_norm_(ps, 1e-3)
                    coef = (1.0 / (norm + 1e-6)) * 1e-3
                    for p, g in zip(ps, was):
                        assert torch.equal(p.grad, g * coef)
        except BaseException as e:      # an assertion in a thread fails the test, not the thread
            failures.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
        assert not t.is_alive()
    assert not failures, failures
