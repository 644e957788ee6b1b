"""The work that programs have mi_adamw do, as cases that a measurement can prepare, run and check.

A case names a parameter set (a GPT of mini-megatron's family by its sizes) and how a program
steps it: ``kind`` is the public entry point,

  step    FusedAdamW.step() after a backward, tables or flat buffers
  graph   the same step (capturable=True) recorded once into a HIP graph and replayed
  zero    one ZeRO-1 rank's step: ZeroRangeStep.begin / grad_sumsq / finalize / update
  clip    clip_grad_norm_() on its own, ahead of some other optimizer
  train   a bf16-autocast training iteration of linear layers on the optimizer's bf16 copies:
          zero_grad, forward under bf16_weights, backward, step

Values follow the repository's workloads: weights N(0, 0.02), LayerNorm weights 1 and biases 0,
gradients N(0, grad_std), exp_avg N(0, 1e-3), exp_avg_sq |N(0, 1e-6)|, step count 1000 before
the pass; lr 3e-4, betas (0.9, 0.95), eps 1e-8, weight decay 0.1.

Tensors of the tables layout are views of one block per stream, each at a multiple of 512 bytes
(where torch's caching allocator would put a tensor of its own), so that a pass returns a few
whole blocks instead of hundreds of tensors.  With ``bucket`` the gradients lie as
DistributedDataParallel's gradient_as_bucket_view leaves them: end to end in reverse order,
each wherever the one before it ends.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mini-megatron_amd"))

import mi_adamw  # noqa: E402
from mi_adamw.workloads import GPT_125M, GPT_1P3B, GPT_350M, GPTShape, init_kind  # noqa: E402

LR, BETA1, BETA2, EPS, DECAY = 3e-4, 0.9, 0.95, 1e-8, 0.1
STEP = 1000            # every parameter's step count before the pass
MAX_NORM = 1.0
ALIGN = 128            # fp32 elements: 512 bytes
FLAT_ALIGN = 32        # fp32 elements: the flat layout's 128 bytes

DEFAULTS = dict(kind="step", layout="tables", state="fp32", copy=False, clip=True, chain="default",
                amsgrad=False, groups=1, bucket=False, moving=False, grad_std=1e-2, world=1)


def _case(name, shape, **options):
    c = dict(DEFAULTS, layers=shape.layers, hidden=shape.hidden, ffn=shape.ffn, vocab=shape.vocab,
             positions=shape.positions)
    c.update(options)
    return dict(c, name=name) if name else c


def _shape(layers, hidden, ffn, vocab, positions):
    return GPTShape("", layers=layers, hidden=hidden, heads=1, ffn=ffn, vocab=vocab,
                    positions=positions)


def listed():
    return [
        # the model of the training tests (19 tensors, 0.1M parameters) in the reference's loop:
        # what a call costs when there is next to nothing to update
        _case("tiny-clip", _shape(2, 64, 256, 64, 8)),
        # a small GPT (5M) whose whole iteration a program captured: launches and their gaps
        _case("small-graph", _shape(4, 256, 1024, 4096, 512), kind="graph"),
        # a small GPT (17M) in flat buffers, with the bf16 weights its forward runs on
        _case("mini-flat-copy-clip", _shape(6, 384, 1536, 8192, 512), layout="flat", copy=True),
        # odd widths, gradients as DDP's bucket views: no tensor ends, and few gradients begin,
        # on a 16-byte boundary
        _case("ragged-bucket-clip", _shape(6, 511, 2045, 10007, 257), bucket=True),
        # mini-megatron's default model in its loop: zero_grad() frees the gradients, backward
        # allocates them elsewhere
        _case("gpt125m-clip", GPT_125M, moving=True),
        # the same under --fused (torch's fused=True arithmetic), without the clip
        _case("gpt125m-fused", GPT_125M, chain="fused", clip=False),
        # gradient clipping in front of another optimizer, above and below the threshold
        _case("clip-gpt125m", GPT_125M, kind="clip"),
        _case("clip-mini-quiet", _shape(6, 384, 1536, 8192, 512), kind="clip", grad_std=1e-4),
        # one of 8 ZeRO-1 ranks at its real share of the 350M set, fp32 with the bf16 copy
        _case("gpt350m-zero8", GPT_350M, kind="zero", layout="flat", copy=True, world=8),
        # a pipeline stage of the 1.3B set (6 of 24 layers), per-tensor, bf16 moments and copy
        _case("gpt1.3b-stage-bf16", _shape(6, 2048, 8192, 0, 0), state="bf16", copy=True),
        # the largest: the whole 1.3B set in flat buffers, bf16 moments and copy
        _case("gpt1.3b-flat-bf16", GPT_1P3B, layout="flat", state="bf16", copy=True),
        # a training iteration whose linears run on the bf16 copies: the casts' backward and
        # the step beside a forward and backward of 4 x 512 tokens
        _case("train-bf16-weights", _shape(4, 768, 3072, 0, 0), kind="train", copy=True,
              positions=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        kind = rng.choice(["step"] * 9 + ["clip"] * 3 + ["graph"] * 2 + ["zero"] * 2 + ["train"])
        hidden = _log_int(rng, 32, 2048)
        if rng.random() < 0.6:
            hidden = max(32, hidden // 32 * 32)      # most models; the rest stay odd
        shape = _shape(rng.randint(1, 24), hidden, hidden * rng.choice([2, 3, 4]) +
                       (hidden % 2) * rng.randint(0, 7), _log_int(rng, 64, 50257),
                       _log_int(rng, 8, 2048))
        c = _case(None, shape, kind=kind, grad_std=rng.choice([1e-2, 1e-2, 1e-5]))
        if kind == "train":
            c.update(layers=rng.randint(1, 6), hidden=rng.choice([256, 512, 768, 1024]), vocab=0,
                     positions=rng.choice([512, 1024, 2048]), copy=True, grad_std=1e-2)
            c.update(ffn=4 * c["hidden"])
            return c
        if kind == "clip":
            c.update(bucket=rng.random() < 0.4)
        if kind in ("step", "graph"):
            c.update(clip=rng.random() < 0.7, state=rng.choice(["fp32", "fp32", "bf16"]),
                     chain=rng.choice(["default", "default", "fused"]))
        if kind == "graph":
            c.update(layers=rng.randint(1, 12), hidden=min(hidden, 768),
                     ffn=min(shape.ffn, 3072))
        if kind == "step":
            c.update(layout=rng.choice(["tables", "tables", "flat"]), copy=rng.random() < 0.4,
                     amsgrad=rng.random() < 0.12, groups=rng.choice([1, 1, 2]))
            if c["layout"] == "tables":
                c.update(bucket=rng.random() < 0.3, moving=rng.random() < 0.3)
                if c["copy"]:
                    c.update(layers=min(c["layers"], 6))
        if kind == "zero":
            c.update(layout="flat", copy=rng.random() < 0.6, state=rng.choice(["fp32", "bf16"]),
                     world=rng.choice([2, 3, 4, 8]))
        if work(c)["bytes"] <= most:
            return c


# ------------------------------------------------------------------ the parameter set

def _tensors(c):
    """(name, shape, numel) of every tensor in registration order."""
    if c["kind"] == "train":
        h, f = c["hidden"], c["ffn"]
        out = [(f"mlp.{i}", s) for i in range(c["layers"]) for s in ((f, h), (h, f))]
    else:
        out = [(n, s) for n, s in _shape(c["layers"], c["hidden"], c["ffn"], c["vocab"],
                                         c["positions"]).tensors() if math.prod(s)]
    return [(n, s, math.prod(s)) for n, s in out]


def _numel(c):
    return sum(n for _, _, n in _tensors(c))


def _group_of(c, name):
    """With two groups: matrices decay, LayerNorm weights and biases do not."""
    return 1 if c["groups"] == 2 and init_kind(name) != "normal" else 0


def _order(c):
    """Indices of the tensors in param_groups order."""
    t = _tensors(c)
    return sorted(range(len(t)), key=lambda i: (_group_of(c, t[i][0]), i))


def _offsets(c, align):
    """Where each tensor begins in a block, and the block's length."""
    t, at, off = _tensors(c), {}, 0
    for i in _order(c):
        at[i] = off
        off += -(-t[i][2] // align) * align
    return at, off


def _grad_offsets(c):
    if not c["bucket"]:
        return _offsets(c, ALIGN)
    t, at, off = _tensors(c), {}, 0
    for i in reversed(_order(c)):
        at[i] = off
        off += t[i][2]
    return at, off


def _views(block, at, tensors):
    return [block[at[i]:at[i] + n].view(s) for i, (_, s, n) in enumerate(tensors)]


def _inputs(c, seed):
    """Blocks of p, g, m, v (and g2, vmax where the case has them), made from the seed alone."""
    dev = torch.device("cuda", 0)
    rng = torch.Generator(device=dev).manual_seed(seed)
    t = _tensors(c)
    at, total = _offsets(c, FLAT_ALIGN if c["layout"] == "flat" else ALIGN)
    gat, gtotal = _grad_offsets(c)
    sdt = torch.bfloat16 if c["state"] == "bf16" else torch.float32
    out = {}
    if c["kind"] != "clip":
        p = torch.zeros(total, device=dev)
        for (name, _, n), x in zip(t, _views(p, at, t)):
            kind = init_kind(name)
            if kind == "normal":
                x.normal_(0.0, 0.02, generator=rng)
            elif kind == "ones":
                x.fill_(1.0)
        out["p"] = p
        for key in ("m", "v") + (("x",) if c["amsgrad"] else ()):
            b = torch.zeros(total, device=dev)
            for x in _views(b, at, t):
                if key == "m":
                    x.normal_(0.0, 1e-3, generator=rng)
                else:
                    x.normal_(0.0, 1e-6, generator=rng).abs_()
            out[key] = b.to(sdt)
    for key in ("g", "g2") if c["moving"] else ("g",):
        b = torch.zeros(gtotal, device=dev)
        for x in _views(b, gat, t):
            x.normal_(0.0, c["grad_std"], generator=rng)
        out[key] = b
    return out, at, gat


def _whole(t):
    """The whole memory block that tensor t is a view of."""
    return torch.empty(0, dtype=t.dtype, device=t.device).set_(t.untyped_storage())


# ------------------------------------------------------------------ prepare and run

def _optimizer(c, params, **more):
    named = list(zip(_tensors(c), params))
    groups = [dict(params=[p for (n, _, _), p in named if _group_of(c, n) == k],
                   weight_decay=0.0 if k else DECAY) for k in range(c["groups"])]
    return mi_adamw.FusedAdamW(
        [g for g in groups if g["params"]], lr=LR, betas=(BETA1, BETA2), eps=EPS,
        weight_decay=DECAY, amsgrad=c["amsgrad"], fused=c["chain"] == "fused" or None,
        max_grad_norm=MAX_NORM if c["clip"] else None,
        state_dtype=torch.bfloat16 if c["state"] == "bf16" else torch.float32,
        bf16_copy=c["copy"], flat_buffer=c["layout"] == "flat", **more)


def prepare(case, seed):
    c = case
    if c["kind"] == "train":
        return _prepare_train(c, seed)
    t = _tensors(c)
    blocks, at, gat = _inputs(c, seed)
    if c["kind"] == "clip":
        gs = _views(blocks["g"], gat, t)
        params = [torch.nn.Parameter(torch.empty_like(g)) for g in gs]
        for p, g in zip(params, gs):
            p.grad = g
        return {"case": c, "params": params, "out": {"g": blocks["g"]}}
    params = [torch.nn.Parameter(x) for x in _views(blocks["p"], at, t)]
    for p, g in zip(params, _views(blocks["g"], gat, t)):
        p.grad = g
    more = {}
    if c["kind"] == "graph":
        more["capturable"] = True
    if c["kind"] == "zero":
        more["grad_prescale"] = mi_adamw.dp_prescale(c["world"])
    opt = _optimizer(c, params, **more)
    keys = [("exp_avg", "m"), ("exp_avg_sq", "v")] + ([("max_exp_avg_sq", "x")] if c["amsgrad"]
                                                      else [])
    state = {key: _views(blocks[b], at, t) for key, b in keys}
    if c["layout"] == "flat":
        for i, p in enumerate(params):
            opt.set_state(p, STEP, *[state[key][i] for key, _ in keys])
        out = {"p": _whole(params[0])}
        out.update({b: _whole(opt.state[params[0]][key]) for key, b in keys})
        if c["copy"]:
            out["copy"] = _whole(opt.bf16_param(params[0]))
    else:
        # a checkpoint's tensors put into the state, as a loader leaves them
        for i, p in enumerate(params):
            opt.state[p] = {key: state[key][i] for key, _ in keys}
            opt.state[p]["step"] = torch.tensor(float(STEP))
        out = {b: blocks[b] for b in ("p", "m", "v", "x") if b in blocks}
        if c["copy"]:
            out["copy"] = opt.bf16_params()
    s = {"case": c, "params": params, "opt": opt, "out": out}
    if c["moving"]:
        s["grads"] = [_views(blocks[k], gat, t) for k in ("g", "g2")]
        s["turn"] = 0
    if c["kind"] == "zero":
        s["rank"] = mi_adamw.ZeroRangeStep(opt, c["world"])
    if c["kind"] == "graph":
        _record(s, blocks, state)
    return s


def _record(s, blocks, state):
    """One eager step builds the tables, then the step is recorded; the values go back to
    what they were."""
    opt, params = s["opt"], s["params"]
    saved = {k: blocks[k].clone() for k in ("p", "m", "v")}
    opt.step()
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        opt.step()
    for k, b in saved.items():
        blocks[k].copy_(b)
    for p in params:
        opt.state[p]["step"].fill_(float(STEP))


def run(state):
    c = state["case"]
    if c["kind"] == "train":
        return _run_train(state)
    if c["kind"] == "clip":
        norm = mi_adamw.clip_grad_norm_(state["params"], MAX_NORM)
        return {"norm": norm, **state["out"]}
    opt = state["opt"]
    if c["kind"] == "graph":
        state["graph"].replay()
    elif c["kind"] == "zero":
        rank = state["rank"]
        hypers = rank.begin()
        # across GPUs the ranks' sums are all-reduced here
        norm, coef = rank.finalize(rank.grad_sumsq(0))
        rank.update(0, hypers, coef)
        return {"norm": norm, **state["out"]}
    else:
        if c["moving"]:
            for p, g in zip(state["params"], state["grads"][state["turn"]]):
                p.grad = g
            state["turn"] ^= 1
        opt.step()
    if c["clip"]:
        return {"norm": opt.last_grad_norm, **state["out"]}
    return dict(state["out"])


# ------------------------------------------------------------------ the training iteration

class _Stack(torch.nn.Module):
    def __init__(self, weights):
        super().__init__()
        self.linears = torch.nn.ModuleList()
        for w in weights:
            lin = torch.nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
            lin.weight = torch.nn.Parameter(w)
            self.linears.append(lin)

    def forward(self, x):
        for up, down in zip(self.linears[::2], self.linears[1::2]):
            x = x + down(torch.nn.functional.gelu(up(x)))
        return x


def _train_inputs(c, seed):
    dev = torch.device("cuda", 0)
    rng = torch.Generator(device=dev).manual_seed(seed)
    ws = [torch.randn(s, generator=rng, device=dev) * 0.02 for _, s, _ in _tensors(c)]
    x, y = (torch.randn(c["positions"], c["hidden"], generator=rng, device=dev)
            for _ in range(2))
    return ws, x, y


def _loss(out, y):
    return (out - y).square().sum() / y.shape[0]


def _prepare_train(c, seed):
    ws, x, y = _train_inputs(c, seed)
    model = _Stack(ws)
    opt = _optimizer(c, list(model.parameters()))
    return {"case": c, "model": model, "opt": opt, "x": x, "y": y}


def _run_train(s):
    model, opt = s["model"], s["opt"]
    opt.zero_grad()
    with torch.autocast("cuda", dtype=torch.bfloat16), mi_adamw.bf16_weights(opt, model):
        out = model(s["x"])
    _loss(out.float(), s["y"]).backward()
    opt.step()
    params = list(model.parameters())
    return {"logits": out.detach(), "norm": opt.last_grad_norm,
            "w": [p.detach() for p in params], "grad": [p.grad for p in params],
            "m": [opt.state[p]["exp_avg"] for p in params]}


# ------------------------------------------------------------------ what a pass needs

def _owned(c):
    """[lo, hi) of the flat block that the case's rank owns: rank 0's of equal slices cut at
    the flat layout's alignment."""
    total = _offsets(c, FLAT_ALIGN)[1]
    return 0, min(total, total // FLAT_ALIGN // c["world"] * FLAT_ALIGN)


def work(case):
    c = case
    n = _numel(c)
    if c["kind"] == "clip":
        # every gradient read; written only where the norm is over the threshold
        over = c["grad_std"] * math.sqrt(n) > MAX_NORM
        return {"bytes": n * (8 if over else 4), "flops": 3 * n}
    s = 2 if c["state"] == "bf16" else 4
    per = 4 + 8 + 4 * s + (2 if c["copy"] else 0) + (2 * s if c["amsgrad"] else 0)
    if c["kind"] == "zero":
        n = _owned(c)[1]
    w = {"bytes": n * per, "flops": 15 * n}
    if c["kind"] == "train":
        # the step, the widened gradients (2 read, 4 written) and each product's operands
        w["bytes"] += n * (6 + 3 * 2) + 10 * 2 * c["positions"] * c["layers"] * (
            c["hidden"] + c["ffn"])
        w["flops"] += 6 * n * c["positions"]
    return w


def tolerance(case):
    """About four times the largest error against exact(): in fp32 6e-8 (the values' own
    rounding); a bf16 moment or copy is its own rounding, 1.7e-3; in the training iteration the
    bf16 products show, 4.3e-3 in its logits, gradients and moments."""
    c = case
    if c["kind"] == "train":
        return {"rel": 1.8e-2, "max": 0.2}
    if c["state"] == "bf16" or c["copy"]:
        return {"rel": 6.8e-3, "max": 1.6e-2}
    return {"rel": 2.5e-7, "max": 2.5e-6}


# ------------------------------------------------------------------ in 64 bits

def _adamw64(p, g, m, v, x, decay):
    p = p * (1.0 - LR * decay)
    m = m + (1.0 - BETA1) * (g - m)
    v = BETA2 * v + (1.0 - BETA2) * g * g
    d = v if x is None else torch.maximum(x, v)
    t = STEP + 1
    den = d.sqrt() / math.sqrt(1.0 - BETA2 ** t) + EPS
    return p - LR / (1.0 - BETA1 ** t) * m / den, m, v, d


def _coef64(norm):
    return torch.clamp(MAX_NORM / (norm + 1e-6), max=1.0)


def _norm64(xs):
    return torch.stack([x.double().square().sum() for x in xs]).sum().sqrt()


def exact(case, seed):
    c = case
    if c["kind"] == "train":
        return _exact_train(c, seed)
    t = _tensors(c)
    blocks, at, gat = _inputs(c, seed)
    gs = _views(blocks["g"], gat, t)
    if c["kind"] == "clip":
        norm = _norm64(gs)
        return {"norm": norm, "g": blocks["g"].double() * _coef64(norm)}
    pre = 1.0 / c["world"] if c["kind"] == "zero" else 1.0
    lo, hi = _owned(c) if c["kind"] == "zero" else (0, blocks["p"].numel())
    own = [(max(lo - at[i], 0), min(max(hi - at[i], 0), n)) for i, (_, _, n) in enumerate(t)]
    norm = _norm64([g.reshape(-1)[a:b] * pre for g, (a, b) in zip(gs, own)])
    scale = pre * (_coef64(norm) if c["clip"] else 1.0)
    keys = [k for k in ("p", "m", "v", "x") if k in blocks]
    out = {k: blocks[k].double() for k in keys}
    copies = [None] * len(t)
    for i, (name, shape, _) in enumerate(t):
        a, b = own[i]
        if b <= a:
            continue
        at_, to = at[i] + a, at[i] + b
        new = _adamw64(out["p"][at_:to], gs[i].reshape(-1)[a:b].double() * scale,
                       out["m"][at_:to], out["v"][at_:to],
                       out["x"][at_:to] if "x" in out else None,
                       0.0 if _group_of(c, name) else DECAY)
        for k, value in zip(("p", "m", "v", "x"), new):
            if k in out:
                out[k][at_:to] = value
        copies[i] = out["p"][at_:to].view(shape) if c["layout"] == "tables" else None
    if c["copy"]:
        out["copy"] = out["p"] if c["layout"] == "flat" else [copies[i] for i in _order(c)]
    if c["clip"]:
        out["norm"] = norm
    return out


def _exact_train(c, seed):
    ws, x, y = _train_inputs(c, seed)
    ws = [w.double().requires_grad_() for w in ws]
    out = x.double()
    for up, down in zip(ws[::2], ws[1::2]):
        out = out + torch.nn.functional.gelu(out @ up.t()) @ down.t()
    _loss(out, y.double()).backward()
    norm = _norm64([w.grad for w in ws])
    coef = _coef64(norm)
    new_w, new_m = [], []
    with torch.no_grad():
        for w in ws:
            m = (1.0 - BETA1) * w.grad * coef
            v = (1.0 - BETA2) * (w.grad * coef).square()
            den = v.sqrt() / math.sqrt(1.0 - BETA2) + EPS
            new_w.append(w * (1.0 - LR * DECAY) - LR / (1.0 - BETA1) * m / den)
            new_m.append(m)
    return {"logits": out.detach(), "norm": norm, "w": new_w, "grad": [w.grad for w in ws],
            "m": new_m}
