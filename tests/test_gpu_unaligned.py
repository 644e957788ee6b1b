"""GPU: tensors at any element boundary (bucketed gradients, odd-sized neighbours).

The kernels read and write groups of four elements wherever a tensor begins, so each
stream here starts at an offset of its own inside a buffer whose other elements must stay
as they were.  Sizes sit at the edges of a group (4), a norm and an update tile (1024) and
a chunk (4096).  The same element chain runs at every alignment, so results are compared
bit for bit: fp32 with torch, bf16 moments with the oracle's bf16-state model.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import max_ulp, same_bits

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 4, 5, 1023, 1024, 1027, 4095, 4096, 4097, 9001]
MARK = -7.0     # exact in bf16


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a ROCm GPU")
    yield torch.device("cuda", 0)
    from mi_adamw import clip
    clip._cache.clear()      # other tests count the tables of their own sizes


def _guarded(values: torch.Tensor, offset: int):
    """`values` as a view at element `offset` of a buffer of marks, and the buffer."""
    buf = torch.full((values.numel() + offset + 5,), MARK, dtype=values.dtype,
                     device=values.device)
    view = buf[offset:offset + values.numel()]
    view.copy_(values)
    return view, buf


def _untouched(bufs, n: int, offsets) -> bool:
    return all(bool((b[:o] == MARK).all()) and bool((b[o + n:] == MARK).all())
               for b, o in zip(bufs, offsets))


def _values(n: int, dev, seed: int):
    gen = torch.Generator(device=dev).manual_seed(seed)
    p, g, m, v = (torch.randn(n, device=dev, generator=gen) for _ in range(4))
    return p * 0.02, g * 1e-2, m * 1e-3, (v * 1e-6).abs()


@pytest.mark.parametrize("offsets", [(0, 1, 0, 0), (3, 2, 1, 3), (1, 0, 2, 1)])
@pytest.mark.parametrize("state", [torch.float32, torch.bfloat16])
def test_step_at_any_element_boundary(dev, state, offsets):
    import mi_adamw
    from oracle import oracle as O
    hp = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
    params, bufs, before = [], [], []
    for k, n in enumerate(SIZES):
        p, g, m, v = _values(n, dev, 100 + k)
        m, v = m.to(state), v.to(state)
        views, bs = zip(*(_guarded(t, o) for t, o in zip((p, g, m, v), offsets)))
        q = torch.nn.Parameter(views[0])
        q.grad = views[1]
        params.append((q, views[2], views[3]))
        bufs.append(bs)
        before.append((p, g, m, v))
    opt = mi_adamw.FusedAdamW([q for q, _, _ in params], state_dtype=state, bf16_copy=True,
                              max_grad_norm=0.5, clip_write_grads=True, **hp)
    for q, m, v in params:
        opt.state[q] = {"step": torch.tensor(9.0), "exp_avg": m, "exp_avg_sq": v}
    opt.step()
    torch.cuda.synchronize()
    coef = O.clip_coef(np.float32(opt.last_grad_norm.item()), 0.5)
    assert np.float32(opt.last_grad_norm.item()) == O.total_norm(
        [g.cpu().numpy() for _, g, _, _ in before])
    for (q, m, v), bs, (p0, g0, m0, v0) in zip(params, bufs, before):
        n = q.numel()
        assert _untouched(bs, n, offsets), n
        assert same_bits(opt.bf16_param(q), q.detach().to(torch.bfloat16)), n
        g = (g0 * torch.tensor(float(coef), device=dev))
        assert max_ulp(q.grad, g) == 0, n
        if state == torch.float32:
            ref = torch.nn.Parameter(p0.clone())
            ref.grad = g
            topt = torch.optim.AdamW([ref], foreach=False, **hp)
            topt.state[ref] = {"step": torch.tensor(9.0), "exp_avg": m0.clone(),
                               "exp_avg_sq": v0.clone()}
            topt.step()
            st = topt.state[ref]
            assert max_ulp(q, ref) == 0, n
            assert max_ulp(m, st["exp_avg"]) == 0 and max_ulp(v, st["exp_avg_sq"]) == 0, n
        else:
            bits = [t.view(torch.int16).cpu().numpy().view("uint16").copy() for t in (m0, v0)]
            p = p0.cpu().numpy().copy()
            O.adamw_step_bf16state(p, g0.cpu().numpy().copy(), *bits, step=10.0,
                                   grad_scale=coef, **hp)
            assert O.max_ulp(p, q.detach().cpu().numpy())[0] == 0, n
            for t, b in zip((m, v), bits):
                assert np.array_equal(t.view(torch.int16).cpu().numpy().view("uint16"), b), n


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_clip_at_any_element_boundary(dev, offset):
    import mi_adamw
    from oracle import oracle as O
    grads = [_values(n, dev, 200 + k)[1] for k, n in enumerate(SIZES)]
    placed = [_guarded(g, offset) for g in grads]
    params = [torch.nn.Parameter(torch.empty_like(g)) for g in grads]
    for q, (view, _) in zip(params, placed):
        q.grad = view
    norm = mi_adamw.clip_grad_norm_(params, 0.25)
    torch.cuda.synchronize()
    assert np.float32(norm.item()) == O.total_norm([g.cpu().numpy() for g in grads])
    coef = torch.tensor(float(O.clip_coef(np.float32(norm.item()), 0.25)), device=dev)
    for q, g, (_, buf) in zip(params, grads, placed):
        assert max_ulp(q.grad, g * coef) == 0
        assert _untouched([buf], g.numel(), [offset])
