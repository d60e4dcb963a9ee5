"""The work that a trainer has this package do, as measurable cases.

Each case goes through the package's public entry points the way a stage of
a pipeline-parallel trainer calls them: the optimizer step over its parameter
shard, the gradient clip, the sharded "pieces" unit update, the fp8 codec of
a stage boundary in both directions, the boundary's autograd function, the
scaled-fp8 wire and the tied table's row fold.  `listed()` fixes one size of
each; `draw()` spreads the sizes over the ranges they stand for, ragged ones
among them.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from elysium_wan_amd import boundary as _boundary
from elysium_wan_amd import fp8, optim, pieces, planes
from elysium_wan_amd.accumulate import TiedRowFold

DEV = "cuda"
LR, BETAS, EPS = 3e-4, (0.9, 0.95), 1e-8
STEP0 = 100  # the step a resumed optimizer has reached
FP8 = {"e4m3": (torch.float8_e4m3fn, 8), "e5m2": (torch.float8_e5m2, 15)}
DT = {"f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "bf16": 2}
# tensors laid out one by one start on 256-byte boundaries, as the optimizer's
# own moment slices do; packed ones follow each other without padding
ALIGN = 64


def listed():
    return [
        # a tiny GPT stage (d = 768, 3 blocks and the final norm, 21.3M
        # parameters in 38 tensors, fp32 gradients): a step short enough that
        # launches and host work count
        dict(name="step_tiny", kind="step", d=768, blocks=3, tail=True, gdt="f32", order="host", wd=0.1, clip=1.0, fold=False, packed=False),
        # one of two stages of a 2.8B model (d = 2560, 16 blocks, 1.26B
        # parameters, bf16 gradients): the ordinary large step
        dict(name="step_stage", kind="step", d=2560, blocks=16, tail=False, gdt="bf16", order="host", wd=0.1, clip=1.0, fold=False, packed=False),
        # a ragged shard, 1,000 norm and bias vectors among 100 matrices, with
        # torch's AdamW and the last microbatch folded inside the update
        dict(name="step_ragged_fold", kind="step", d=6144, blocks=0, tail=False, vecs=1000, mats=100, matrows=512, gdt="bf16", order="torch", wd=0.0, clip=0.0, fold=True, packed=False),
        # one block's pieces on one of three peers, packed back to back (the
        # pieces' lengths are no multiple of a vector): the microbatches' fold,
        # the unit's step and the bf16 casts
        dict(name="pieces_unit", kind="pieces", d=2560, peers=3, mbs=4),
        # the gradient clip by itself, as a loop with another optimizer calls it
        dict(name="clip_mid", kind="clip", d=1600, blocks=4, gdt="f32", packed=False),
        # the smallest codec call: a tiny stage's activation [4, 1024, 768]
        # scaled per tensor, sent and received
        dict(name="codec_tiny_tensor", kind="codec", rows=4096, cols=768, dt="bf16", fmt="e4m3", per_tensor=True, out="bf16"),
        # the boundary of the 2.8B model, forward and backward
        dict(name="boundary_stage", kind="boundary", rows=16384, cols=2560, dt="bf16", fmt="e4m3"),
        # a boundary [8, 2047, 1601] of an odd width, sent and received per row
        dict(name="codec_odd_rows", kind="codec", rows=16376, cols=1601, dt="bf16", fmt="e5m2", per_tensor=False, out="bf16"),
        # an fp32 recipe's boundary at the width of the 25.1B model (d = 6144)
        dict(name="boundary_wide_f32", kind="boundary", rows=4096, cols=6144, dt="f32", fmt="e4m3"),
        # the largest codec call: a 1 GiB activation [16, 4096, 8192] scaled
        # per tensor, sent and received
        dict(name="codec_large_tensor", kind="codec", rows=65536, cols=8192, dt="bf16", fmt="e5m2", per_tensor=True, out="bf16"),
        # the scaled-fp8 wire, encoded and decoded with the host's compressor
        dict(name="wire_scaled", kind="wire", rows=512, cols=1600, dt="bf16", fmt="e4m3"),
        # the tied table's gradient over four microbatches (32,768 rows of the
        # 2.8B model's width, 4,096 rows touched by each)
        dict(name="tied_table", kind="tied", rows=32768, d=2560, mbs=4, touched=4096, dt="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A row width: a model's (a multiple of 64) half of the time, any else."""
    w = _log(rng, lo, hi)
    return max(64, w // 64 * 64) if rng.random() < 0.5 else w


def draw(rng):
    kind = rng.choice(["step", "step", "step", "pieces", "clip", "codec", "codec", "codec", "codec", "boundary", "boundary", "wire", "tied"])
    if kind == "step":
        gdt, order = rng.choice(["f32", "bf16"]), rng.choice(["host", "torch"])
        opts = dict(gdt=gdt, order=order, wd=rng.choice([0.0, 0.1]), clip=rng.choice([0.0, 1.0]), fold=rng.random() < 0.3, packed=rng.random() < 0.4)
        if rng.random() < 0.3:
            return dict(kind=kind, d=_width(rng, 256, 6144), blocks=0, tail=False, vecs=_log(rng, 50, 1000), mats=_log(rng, 5, 100), matrows=_log(rng, 64, 512), **opts)
        return dict(kind=kind, d=_width(rng, 64, 2048), blocks=rng.randint(1, 8), tail=rng.random() < 0.5, **opts)
    if kind == "pieces":
        return dict(kind=kind, d=_width(rng, 256, 3072), peers=rng.randint(2, 7), mbs=rng.randint(2, 6))
    if kind == "clip":
        return dict(kind=kind, d=_width(rng, 64, 2048), blocks=rng.randint(1, 8), gdt=rng.choice(["f32", "bf16"]), packed=rng.random() < 0.4)
    if kind in ("codec", "boundary"):
        n, cols = _log(rng, 1 << 14, 1 << 27), _width(rng, 64, 20480)
        case = dict(kind=kind, rows=max(1, n // cols), cols=cols, dt=rng.choice(["f32", "bf16", "bf16"]), fmt=rng.choice(["e4m3", "e5m2"]))
        if kind == "codec":
            case.update(per_tensor=rng.random() < 0.4, out=rng.choice(["f32", "bf16", "bf16"]))
        return case
    if kind == "wire":
        return dict(kind=kind, rows=_log(rng, 16, 1024), cols=_width(rng, 64, 2048), dt=rng.choice(["f32", "bf16"]), fmt=rng.choice(["e4m3", "e5m2"]))
    rows = _log(rng, 1024, 32768)
    return dict(kind=kind, rows=rows, d=_width(rng, 64, 2560), mbs=rng.randint(2, 4), touched=max(1, rows // rng.choice([8, 16, 32])), dt=rng.choice(["f32", "bf16"]))


# ------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _block(d):
    """One GPT block's tensors: two norms, qkv, projection and the MLP."""
    return [(d,), (d,), (3 * d, d), (3 * d,), (d, d), (d,), (d,), (d,), (4 * d, d), (4 * d,), (d, 4 * d), (d,)]


def _shapes(c):
    if c.get("blocks"):
        return _block(c["d"]) * c["blocks"] + ([(c["d"],), (c["d"],)] if c.get("tail") else [])
    per = c["vecs"] // c["mats"]
    out = []
    for i in range(c["mats"]):
        out += [(c["d"],)] * per + [(c["matrows"], c["d"])]
    return out + [(c["d"],)] * (c["vecs"] - per * c["mats"])


def _piece_shapes(c):
    return [(-(-math.prod(s) // c["peers"]),) for s in _block(c["d"])]


def _offsets(shapes, packed):
    offs, total = [], 0
    for s in shapes:
        offs.append(total)
        n = math.prod(s)
        total += n if packed else -(-n // ALIGN) * ALIGN
    return offs, total


def _views(flat, shapes, offs):
    return [flat[o : o + math.prod(s)].view(s) for s, o in zip(shapes, offs)]


def _normal(gen, n, scale, dtype=torch.float32):
    return torch.randn(n, generator=gen, device=DEV).mul_(scale).to(dtype)


def _step_inputs(c, seed, shapes, packed, fold):
    """Flat p, g, m, v (and the fold's accumulator): parameters N(0, 0.02),
    gradients N(0, 1e-3), the moments of a run that has gone on for a while."""
    g = _gen(seed)
    offs, total = _offsets(shapes, packed)
    moffs, mtotal = _offsets(shapes, False)
    x = dict(offs=offs, total=total, moffs=moffs, mtotal=mtotal)
    x["p"] = _normal(g, total, 0.02)
    x["g"] = _normal(g, total, 1e-3, DT[c.get("gdt", "bf16")])
    x["m"] = _normal(g, mtotal, 3e-4)
    x["v"] = _normal(g, mtotal, 1e-3).square_()
    x["acc"] = _normal(g, total, 1e-3) if fold else None
    return x


def _resume(opt, shapes, x):
    """The optimizer as a resumed run has it: moments and step loaded."""
    ms, vs = _views(x["m"], shapes, x["moffs"]), _views(x["v"], shapes, x["moffs"])
    group = {k: v for k, v in opt.param_groups[0].items() if k != "params"}
    opt.load_state_dict({
        "state": {i: {"step": torch.tensor(float(STEP0)), "exp_avg": m, "exp_avg_sq": v} for i, (m, v) in enumerate(zip(ms, vs))},
        "param_groups": [{**group, "params": list(range(len(shapes)))}],
    })


def _whole(t):
    """The whole flat buffer that a moment is a view of."""
    return torch.empty(0, dtype=t.dtype, device=t.device).set_(t.untyped_storage())


def _activation(c, seed, stream=0):
    """N(0, 1) with 0.1 % of the values 50 times larger, rows of different
    scales: a boundary tensor."""
    g = _gen(seed * 2 + stream)
    rows, cols = c["rows"], c["cols"]
    out = torch.empty(rows, cols, dtype=DT[c["dt"]], device=DEV)
    scale = torch.exp2(torch.randint(-3, 4, (rows, 1), generator=g, device=DEV).float())
    chunk = max(1, (1 << 26) // cols)
    for r in range(0, rows, chunk):
        e = min(rows, r + chunk)
        x = torch.randn(e - r, cols, generator=g, device=DEV)
        big = torch.rand(e - r, cols, generator=g, device=DEV) < 1e-3
        out[r:e] = torch.where(big, x * 50, x) * scale[r:e]
    return out


def prepare(c, seed):
    kind = c["kind"]
    if kind == "step":
        shapes = _shapes(c)
        x = _step_inputs(c, seed, shapes, c["packed"], c["fold"])
        params = [p.requires_grad_(True) for p in _views(x["p"], shapes, x["offs"])]
        copies = torch.zeros(x["total"], dtype=torch.bfloat16, device=DEV)
        opt = optim.FusedAdamW(params, lr=LR, betas=BETAS, eps=EPS, weight_decay=c["wd"], order=c["order"], max_norm=c["clip"] or None,
                               working_copy=_views(copies, shapes, x["offs"]))
        _resume(opt, shapes, x)
        st = opt.state[0]
        return dict(kind=kind, opt=opt, grads=_views(x["g"], shapes, x["offs"]), acc=_views(x["acc"], shapes, x["offs"]) if c["fold"] else None,
                    out=[x["p"], _whole(st["exp_avg"]), _whole(st["exp_avg_sq"]), copies])
    if kind == "pieces":
        shapes = _piece_shapes(c)
        x = _step_inputs(c, seed, shapes, True, False)
        params = [p.requires_grad_(True) for p in _views(x["p"], shapes, x["offs"])]
        opt = pieces.adamw(params, LR)
        _resume(opt, shapes, x)
        st = opt.state[0]
        mbs = [_views(g, shapes, x["offs"]) for g in _microbatches(c, seed, x["total"])]
        return dict(kind=kind, opt=opt, params=params, mbs=mbs, out=[x["p"], _whole(st["exp_avg"]), _whole(st["exp_avg_sq"])])
    if kind == "clip":
        shapes = _shapes(c)
        offs, total = _offsets(shapes, c["packed"])
        flat = _normal(_gen(seed), total, 1e-3, DT[c["gdt"]])
        params = [torch.zeros_like(g) for g in _views(flat, shapes, offs)]
        for p, g in zip(params, _views(flat, shapes, offs)):
            p.grad = g
        return dict(kind=kind, params=params, out=flat)
    if kind == "codec":
        return dict(kind=kind, x=_activation(c, seed), fmt=c["fmt"], per_tensor=c["per_tensor"], out=DT[c["out"]])
    if kind == "boundary":
        return dict(kind=kind, x=_activation(c, seed).requires_grad_(True), g=_activation(c, seed, 1).mul_(1e-5), dtype=FP8[c["fmt"]][0])
    if kind == "wire":
        # the send buffer holds the longest payload its planes can compress to
        return dict(kind=kind, t=_boundary.narrow(_activation(c, seed), FP8[c["fmt"]][0], True), fmt=c["fmt"],
                    send=np.zeros(2 * c["rows"] * (c["cols"] + 1) + 4096, dtype=np.uint8))
    hs, ids, es = _tied_inputs(c, seed)
    return dict(kind=kind, rows=c["rows"], hs=hs, ids=ids, es=es)


def _microbatches(c, seed, total):
    g = _gen(seed + 7919)
    return [_normal(g, total, 1e-3, torch.bfloat16) for _ in range(c["mbs"])]


def _tied_inputs(c, seed):
    g = _gen(seed)
    dt = DT[c["dt"]]
    hs = [torch.randn(c["rows"], c["d"], generator=g, device=DEV).mul_(1e-3).to(dt) for _ in range(c["mbs"])]
    ids = [torch.randperm(c["rows"], generator=g, device=DEV)[: c["touched"]].sort().values.cpu() for _ in range(c["mbs"])]
    es = [torch.randn(c["touched"], c["d"], generator=g, device=DEV).mul_(1e-3).to(dt) for _ in range(c["mbs"])]
    return hs, ids, es


# -------------------------------------------------------------------- a pass


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["opt"].step(grads=s["grads"], acc=s["acc"])
        norm = s["opt"].grad_norm()
        return s["out"] + ([norm] if norm is not None else [])
    if kind == "pieces":
        sums = [pieces.fold(mb[i] for mb in s["mbs"]) for i in range(len(s["params"]))]
        pieces.step_unit(s["opt"], s["params"], sums)
        return s["out"] + sums + [pieces.cast_piece(p, torch.bfloat16) for p in s["params"]]
    if kind == "clip":
        return [optim.clip_grad_norm_(s["params"], 1.0), s["out"]]
    if kind == "codec":
        q, k = fp8.quantize(s["x"], s["fmt"], per_tensor=s["per_tensor"])
        return [q.view(torch.uint8), k, fp8.dequantize(q, k, s["out"])]
    if kind == "boundary":
        y = _boundary.boundary(s["x"], s["dtype"], True)
        return [y, torch.autograd.grad(y, s["x"], s["g"])[0]]
    if kind == "wire":
        payload, shape = planes.encode_scaled_fp8(s["t"], s["fmt"])
        s["send"][: len(payload)] = np.frombuffer(payload, dtype=np.uint8)
        return [len(payload), s["send"], planes.decode(payload, shape)]
    n = len(s["hs"])
    fold = TiedRowFold(s["rows"], range(n))
    for mb in range(n):
        fold.add_head(mb, s["hs"][mb], s["ids"][mb])
        if mb:
            fold.add_embed(mb - 1, s["es"][mb - 1])
    fold.add_embed(n - 1, s["es"][n - 1])
    return [fold.result()]


# ------------------------------------------------------- what a pass amounts to


def work(c):
    kind = c["kind"]
    if kind == "step":
        n = sum(math.prod(s) for s in _shapes(c))
        return dict(bytes=n * (26 + SIZE[c["gdt"]] + (4 if c["fold"] else 0)), flops=n * (16 + (3 if c["clip"] else 0)))
    if kind == "pieces":
        n = sum(math.prod(s) for s in _piece_shapes(c))
        # the parts in, the sums out, p, m and v both ways, the casts out
        return dict(bytes=n * (2 * c["mbs"] + 4 + 24 + 2), flops=n * (14 + c["mbs"]))
    if kind == "clip":
        n = sum(math.prod(s) for s in _shapes(c))
        return dict(bytes=2 * n * SIZE[c["gdt"]], flops=3 * n)
    if kind == "codec":
        n = c["rows"] * c["cols"]
        # x in, the codes out; the codes in, the result out
        return dict(bytes=n * (SIZE[c["dt"]] + 2 + SIZE[c["out"]]), flops=4 * n)
    if kind == "boundary":
        n = c["rows"] * c["cols"]
        return dict(bytes=4 * n * SIZE[c["dt"]], flops=8 * n)
    if kind == "wire":
        n = c["rows"] * c["cols"]
        return dict(bytes=n * (SIZE[c["dt"]] + 1 + 4), flops=6 * n)
    n = c["rows"] * c["d"]
    return dict(bytes=(n * (c["mbs"] + 1) + c["mbs"] * c["touched"] * c["d"]) * SIZE[c["dt"]], flops=2 * n * c["mbs"])


def tolerance(c):
    # The codec, the boundary and the wire give the bytes of their definition;
    # so do the folds, whose order is fixed.
    if c["kind"] in ("codec", "boundary", "wire", "tied"):
        return "exact"
    # fp32 updates in another order of roundings: 1e-7 in p, m and v; a bf16
    # copy whose fp32 value moved by that much may round the other way (one
    # unit of 2^-8 of its value, for about one in 50,000 of them).
    return {"rel": 6e-5, "max": 1.6e-2}


# ------------------------------------------------------------- in 64 bits


def _adamw64(p, g, m, v, wd):
    t = STEP0 + 1
    b1, b2 = BETAS
    m = b1 * m + (1 - b1) * g
    v = b2 * v + (1 - b2) * g * g
    u = (m / (1 - b1**t)) / ((v / (1 - b2**t)).sqrt() + EPS)
    return p * (1 - LR * wd) - LR * u, m, v


def _exact_step(c, seed):
    shapes = _shapes(c)
    x = _step_inputs(c, seed, shapes, c["packed"], c["fold"])
    n = [math.prod(s) for s in shapes]

    def grad(i):
        o = x["offs"][i]
        g = x["g"][o : o + n[i]].double()
        return g + x["acc"][o : o + n[i]].double() if c["fold"] else g

    coef, norm = 1.0, None
    if c["clip"]:
        norm = sum(grad(i).square().sum() for i in range(len(n))).sqrt()
        coef = (c["clip"] / (norm + 1e-6)).clamp(max=1.0)
    P, C = x["p"].double(), torch.zeros(x["total"], dtype=torch.float64, device=DEV)
    M, V = (torch.zeros(x["mtotal"], dtype=torch.float64, device=DEV) for _ in range(2))
    for i in range(len(n)):
        o, mo = slice(x["offs"][i], x["offs"][i] + n[i]), slice(x["moffs"][i], x["moffs"][i] + n[i])
        P[o], M[mo], V[mo] = _adamw64(P[o], grad(i) * coef, x["m"][mo].double(), x["v"][mo].double(), c["wd"])
        C[o] = P[o]
    return [P, M, V, C] + ([norm] if c["clip"] else [])


def _exact_pieces(c, seed):
    shapes = _piece_shapes(c)
    x = _step_inputs(c, seed, shapes, True, False)
    mbs = _microbatches(c, seed, x["total"])
    G = torch.zeros(x["total"], dtype=torch.float64, device=DEV)
    for g in mbs:
        G += g.double()
    P = x["p"].double()
    M, V = (torch.zeros(x["mtotal"], dtype=torch.float64, device=DEV) for _ in range(2))
    cuts = []
    for s, a, b in zip(shapes, x["offs"], x["moffs"]):
        o, mo = slice(a, a + s[0]), slice(b, b + s[0])
        P[o], M[mo], V[mo] = _adamw64(P[o], G[o], x["m"][mo].double(), x["v"][mo].double(), 0.0)
        cuts.append(o)
    return [P, M, V] + [G[o] for o in cuts] + [P[o] for o in cuts]


def _narrow64(x, fmt, per_tensor=False):
    """x scaled by a power of two per row (or over the tensor), rounded to the
    fp8 format and scaled back, in 64 bits."""
    dt, e = FP8[fmt]
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    chunk = max(1, (1 << 26) // x.shape[1])
    parts = range(0, x.shape[0], chunk)
    top = max(x[r : r + chunk].abs().max() for r in parts) if per_tensor else None
    for r in parts:
        y = x[r : r + chunk].double()
        a = top.double().reshape(1, 1) if per_tensor else y.abs().amax(dim=1, keepdim=True)
        k = torch.where(a > 0, torch.frexp(a).exponent - e, 0).double()
        out[r : r + chunk] = (y * torch.exp2(-k)).float().to(dt).double() * torch.exp2(k)
    return out


def exact(c, seed):
    kind = c["kind"]
    if kind == "step":
        return _exact_step(c, seed)
    if kind == "pieces":
        return _exact_pieces(c, seed)
    if kind == "clip":
        shapes = _shapes(c)
        offs, total = _offsets(shapes, c["packed"])
        flat = _normal(_gen(seed), total, 1e-3, DT[c["gdt"]]).double()
        held = torch.zeros(total, dtype=torch.bool, device=DEV)
        for s, o in zip(shapes, offs):
            held[o : o + math.prod(s)] = True
        norm = (flat * held).square().sum().sqrt()
        return [norm, torch.where(held, flat * (1.0 / (norm + 1e-6)).clamp(max=1.0), flat)]
    if kind == "codec":
        return [None, None, _narrow64(_activation(c, seed), c["fmt"], c["per_tensor"])]
    if kind == "boundary":
        return [_narrow64(_activation(c, seed), c["fmt"]), _narrow64(_activation(c, seed, 1).mul_(1e-5), c["fmt"])]
    if kind == "wire":
        return [None, None, _narrow64(_activation(c, seed), c["fmt"])]
    hs, ids, es = _tied_inputs(c, seed)
    acc = torch.zeros(c["rows"], c["d"], dtype=torch.float64, device=DEV)
    for h, i, e in zip(hs, ids, es):
        acc += h.double()
        acc[i.to(DEV)] += e.double()
    return [acc]
