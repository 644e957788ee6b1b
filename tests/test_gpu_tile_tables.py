"""GPU: an update over a table of tiles gives the bits of one over chunks, in every chain and
layout that takes it, on the general and the native path and replayed."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 768, 1023, 1024, 1025, 2049, 4095, 4097, 9000] + [5, 769] * 200


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    return torch.device("cuda", 0)


def _run(dev, opts, groups, odd):
    import mi_adamw
    gen = torch.Generator(device=dev).manual_seed(3)
    params = [torch.nn.Parameter(torch.randn(n, device=dev, generator=gen)) for n in SIZES]
    if groups == 2:
        half = len(params) // 2
        sets = [dict(params=params[:half]), dict(params=params[half:], amsgrad=True)]
    else:
        sets = params
    opt = mi_adamw.FusedAdamW(sets, lr=1e-2, **opts)

    def new_grads():
        block = torch.randn(sum(SIZES) + odd, device=dev, generator=gen) * 0.1
        for p, g in zip(params, block[odd:].split(SIZES)):
            p.grad = g

    new_grads()
    for k in range(4):
        if k == 2 and not opts.get("capturable"):
            new_grads()                          # moved: patched by the native path
        opt.step()
    if opts.get("capturable"):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            opt.step()
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
    out = [p.detach() for p in params] + [p.grad for p in params]
    for p in params:
        out += [t for _, t in sorted(opt.state[p].items())]
    if opts.get("bf16_copy"):
        out += opt.bf16_params()
    flags = [launch.item_flag for launch in opt._launch_cache.launches]
    return [t.clone() for t in out], flags, opt


@pytest.mark.parametrize("chunk", [4096, 65536])
@pytest.mark.parametrize("opts,groups", [
    (dict(max_grad_norm=1.0, clip_write_grads=True), 1), (dict(fused=True), 1),
    (dict(state_dtype=torch.bfloat16, bf16_copy=True, max_grad_norm=1.0), 1),
    (dict(amsgrad=True), 1), (dict(max_grad_norm=1.0), 2),
    (dict(capturable=True, max_grad_norm=1.0), 1),
    (dict(capturable=True, fused=True), 1)])
def test_tiles_give_the_bits_of_chunks(dev, monkeypatch, opts, groups, chunk):
    from mi_adamw import _lib, optimizer
    from mi_adamw.probe import time_probe
    for odd in (0, 1):
        got, flags, opt = _run(dev, dict(opts, chunk_elems=chunk), groups, odd)
        assert set(flags) == {_lib.F_TILES}
        cache = opt._launch_cache
        assert cache.norm_launch is cache.launches[0] or cache.norm_launch.item_flag == 0
        if groups == 1:
            assert time_probe(opt, launches=2) > 0.0     # the twin of this launch
        with monkeypatch.context() as m:
            m.setattr(optimizer, "_TILE_RULE", float("inf"))
            want, flags, _ = _run(dev, dict(opts, chunk_elems=chunk), groups, odd)
        assert set(flags) == {0}
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and torch.equal(a, b)
