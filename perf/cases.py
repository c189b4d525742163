"""The work this library is used for, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare`` makes what a program holds
before the call (fields on the GPU, a batch's problem table, a network),
``run`` makes one pass through the public entry points and returns its
outputs, ``work`` counts the bytes and operations the pass cannot do without
and ``exact`` gives the same outputs from plain torch in 64 bits.

Kinds of case:

* ``sweep``    iterations of the star stencil on one grid (AUTO variant), as
               the command line program and every solver loop run them;
               with ``residual`` the FP64 norm that a solver checks between
               runs of sweeps;
* ``mixed``    the same with 16-bit storage and FP32 defect correction;
* ``batched``  many uneven grids advanced together;
* ``layer``    one 3x3x3 convolution layer of the warm-start network, forward
               and backward, as a training step runs it;
* ``train``    loss and gradients of one batch of the network (the optimizer
               step is left to the caller so that passes stay comparable).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import thesis_amd as st
from thesis_amd import nn, warmstart

DEV = "cuda" if torch.cuda.is_available() else "cpu"
TORCH = {"f32": torch.float32, "f64": torch.float64}
STORE = {"f32": st.F32, "f64": st.F64, "bf16": st.BF16, "f16": st.F16}


def _sweep(dims, nx, ny, nz, radius, iterations, dtype="f32", op="jacobi", shells="equal", residual=False):
    return dict(kind="sweep", dims=dims, nx=nx, ny=ny, nz=nz, radius=radius, iterations=iterations,
                dtype=dtype, op=op, shells=shells, residual=residual)


def listed():
    return [
        # the smallest call: the 5-point Jacobi iteration of a 256 x 256 plate, bound by launches
        dict(_sweep(2, 256, 256, 1, 1, 64), name="plane_256"),
        # one step of the 128^3 Laplace solver: 200 sweeps, then the residual that decides whether to go on
        dict(_sweep(3, 128, 128, 128, 1, 200, residual=True), name="solve_128"),
        # the program's default run: 256^3, 64 sweeps of the THESIS operator, only the first buffer's shell set
        dict(_sweep(3, 256, 256, 256, 1, 64, op="thesis", shells="first"), name="default_256"),
        # the headline sweep: 512^3, 7-point, 100 sweeps
        dict(_sweep(3, 512, 512, 512, 1, 100), name="cube_512"),
        # a grid that is no multiple of anything, 13-point
        dict(_sweep(3, 333, 251, 207, 2, 20), name="ragged_r2"),
        # high order in double precision: 25-point, 384^3
        dict(_sweep(3, 384, 384, 384, 4, 20, dtype="f64"), name="cube_384_r4_f64"),
        # the same stencil with BF16 storage and a defect correction every 10 sweeps
        dict(kind="mixed", nx=384, ny=384, nz=384, radius=4, iterations=40, restart=10, dtype="bf16",
             name="mixed_384_r4"),
        # a wide star (49-point), from the upper half of the radii the program is run with
        dict(_sweep(3, 512, 512, 512, 8, 10), name="cube_512_r8"),
        # a large plane with a 17-point star
        dict(_sweep(2, 8192, 8192, 1, 4, 16), name="plane_8192_r4"),
        # 512 uneven problems (edges 16..128, radius 1 or 2) advanced 50 sweeps together
        dict(kind="batched", count=512, lo=16, hi=128, iterations=50, mode="graph", name="batch_512"),
        # the widest layer of the network's decoder, forward and backward, batch of 8 at 64^3
        dict(kind="layer", n=8, d=64, h=64, w=64, ci=48, co=16, name="layer_48_16"),
        # loss and gradients of a training batch: 8 samples at 64^3, 64 smoothing sweeps in the loss
        dict(kind="train", batch=8, n=64, smooth=64, name="train_64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sweep3"] * 10 + ["sweep2"] * 3 + ["mixed"] * 2 + ["batched"] * 2 + ["layer"] * 2 + ["train"])
    if kind in ("sweep3", "sweep2"):
        radius = rng.choice([1, 1, 1, 2, 2, 3, 4, 4, 6, 8, 12, 16])
        dtype = rng.choice(["f32", "f32", "f32", "f64"])
        op, shells = rng.choice([("jacobi", "equal"), ("jacobi", "equal"), ("thesis", "first")])
        lo = max(40, 4 * radius)
        if kind == "sweep3":
            nx, ny, nz = (_log(rng, lo, 512) for _ in range(3))
            if rng.random() < 0.4:  # cubes of whole cache lines, as solvers like them
                nx = ny = nz = max(lo, nx // 32 * 32)
        else:
            nx, ny, nz = _log(rng, 64, 8192), _log(rng, 64, 8192), 1
            if rng.random() < 0.4:
                nx = ny = max(64, nx // 64 * 64)
        # up to 64 sweeps, fewer on the large and wide ones (a third of the headline sweep's work)
        budget = 4.5e9 / (nx * ny * nz * (1 + radius) * (2 if dtype == "f64" else 1))
        iters = max(2, min(_log(rng, 4, 64), int(budget)))
        return _sweep(2 if kind == "sweep2" else 3, nx, ny, nz, radius, iters, dtype, op, shells,
                      residual=rng.random() < 0.2)
    if kind == "mixed":
        radius = rng.choice([1, 2, 3, 4])
        nx, ny, nz = (_log(rng, 48, 384) for _ in range(3))
        if rng.random() < 0.5:
            nx = ny = nz = max(64, nx // 64 * 64)
        return dict(kind="mixed", nx=nx, ny=ny, nz=nz, radius=radius, iterations=_log(rng, 10, 40),
                    restart=rng.choice([5, 10, 20]), dtype=rng.choice(["bf16", "f16"]))
    if kind == "batched":
        return dict(kind="batched", count=_log(rng, 8, 512), lo=16, hi=rng.choice([48, 96, 128]),
                    iterations=_log(rng, 5, 50), mode=rng.choice(["graph", "persistent"]))
    if kind == "layer":
        ci, co = rng.choice([(8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (48, 16)])
        top = 64 if ci * co <= 1024 else 32
        d, h, w = (2 * _log(rng, 4, top // 2) for _ in range(3))
        return dict(kind="layer", n=rng.randint(1, 8), d=d, h=h, w=w, ci=ci, co=co)
    return dict(kind="train", batch=rng.randint(1, 8), n=rng.choice([16, 24, 32, 40, 48, 64]),
                smooth=rng.choice([0, 16, 32, 64]))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _shell_field(shape, r, g, dtype):
    """Uniform [0, 1) Dirichlet values on the r-thick shell, zero inside."""
    u = torch.rand(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)
    u[tuple(slice(r, n - r) for n in shape)] = 0
    return u


def _shape(case):
    return (case["ny"], case["nx"]) if case.get("dims") == 2 else (case["nz"], case["ny"], case["nx"])


def _sweep_fields(case, seed):
    dtype = TORCH[case["dtype"]]
    u1 = _shell_field(_shape(case), case["radius"], _gen(seed), dtype)
    return u1, (u1.clone() if case["shells"] == "equal" else torch.zeros_like(u1))


def _batch_shapes(case, seed):
    """Edges log-uniform on [lo, hi], each axis its own, radius 1 or 2; the shapes belong to the case."""
    rng = np.random.default_rng(case["count"] * 1009 + case["hi"])
    lo, hi, n = case["lo"], case["hi"], case["count"]
    edges = np.rint(lo * (hi / lo) ** rng.random((n, 3))).astype(int)
    return [(*(int(e) for e in edges[i]), int(rng.integers(1, 3))) for i in range(n)]


def _batch_fields(case, seed):
    shapes = _batch_shapes(case, seed)
    total = sum(nx * ny * nz for nx, ny, nz, _ in shapes)
    u = torch.rand(total, generator=_gen(seed), device=DEV)
    at, views = 0, []
    for nx, ny, nz, r in shapes:
        v = u[at:at + nx * ny * nz].view(nz, ny, nx)
        v[r:nz - r, r:ny - r, r:nx - r] = 0
        views.append(v)
        at += nx * ny * nz
    return shapes, u, views


def _layer_inputs(case, seed):
    g = _gen(seed)
    shape, ci, co = (case["n"], case["d"], case["h"], case["w"]), case["ci"], case["co"]
    x = torch.relu(torch.randn((*shape, ci), generator=g, device=DEV)).bfloat16()
    w = torch.zeros((co, (27 * ci + 31) // 32 * 32), device=DEV, dtype=torch.bfloat16)
    w[:, :27 * ci] = (torch.randn((co, 27 * ci), generator=g, device=DEV) * math.sqrt(2.0 / (27 * ci))).bfloat16()
    b = torch.randn(co, generator=g, device=DEV) * 0.1
    gy = torch.randn((*shape, co), generator=g, device=DEV) * 1e-3
    return shape, x, w, b, gy


NET = [("e1a", 8, 16), ("e1b", 16, 16), ("e2a", 16, 32), ("e2b", 32, 32), ("bta", 32, 64), ("btb", 64, 64),
       ("d2a", 96, 32), ("d2b", 32, 32), ("d1a", 48, 16), ("d1b", 16, 16)]


def _net_weights(seed):
    rng = np.random.default_rng(seed)
    sd = {}
    for name, ci, co in NET:
        sd[name + ".w"] = (rng.standard_normal((co, 27 * ci)) * math.sqrt(2.0 / (27 * ci))).astype(np.float32)
        sd[name + ".b"] = (rng.standard_normal(co) * 0.01).astype(np.float32)
    sd["head.w"] = (rng.standard_normal(16) * 0.1).astype(np.float32)
    sd["head.b"] = (rng.standard_normal(1) * 0.01).astype(np.float32)
    return sd


def _solved_fields(case, seed):
    """Laplace fields whose faces are sums of eight sine modes: the closed form of what a training set holds."""
    n, rng = case["n"], np.random.default_rng(seed)
    s = torch.linspace(0, 1, n, dtype=torch.float64, device=DEV)
    out = torch.zeros((case["batch"], n, n, n), dtype=torch.float64, device=DEV)
    for b in range(case["batch"]):
        for axis in range(3):
            for far in (0, 1):
                for _ in range(8):
                    a, p, q = rng.standard_normal(), int(rng.integers(1, 5)), int(rng.integers(1, 5))
                    k = math.pi * math.hypot(p, q)
                    prof = torch.sinh(k * (s if far else 1 - s)) / math.sinh(k)
                    f = [torch.sin(math.pi * p * s), torch.sin(math.pi * q * s)]
                    f.insert(axis, prof)
                    out[b] += a * f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]
    return out.float()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sweep":
        u1, u2 = _sweep_fields(case, seed)
        p = st.StencilParams.make(nx=case["nx"], ny=case["ny"], nz=case["nz"], dimensions=case["dims"],
                                  radius=case["radius"], iterations=case["iterations"], dtype=STORE[case["dtype"]],
                                  op=st.OP_JACOBI if case["op"] == "jacobi" else st.OP_THESIS,
                                  variant="auto", heuristic=1)
        # the THESIS operator is no contraction (its fields grow up to twofold
        # a sweep), so each pass is a run of its own, from the initial field
        start = u1.clone() if case["op"] == "thesis" else None
        return dict(kind=kind, p=p, u=[u1, u2], start=start, residual=case["residual"])
    if kind == "mixed":
        x = _shell_field(_shape(case), case["radius"], _gen(seed), torch.float32)
        p = st.StencilParams.make(nx=case["nx"], ny=case["ny"], nz=case["nz"], radius=case["radius"],
                                  iterations=case["iterations"], restart=case["restart"], op=st.OP_JACOBI,
                                  dtype=STORE[case["dtype"]], variant="auto", heuristic=1)
        return dict(kind=kind, p=p, x=x, u=torch.empty_like(x),
                    e=[torch.empty(x.shape, dtype=torch.int16, device=DEV) for _ in range(3)])
    if kind == "batched":
        shapes, u1, v1 = _batch_fields(case, seed)
        u2 = u1.clone()
        probs = (st.Problem * len(shapes))()
        at = 0
        for i, (nx, ny, nz, r) in enumerate(shapes):
            probs[i] = st.Problem(nx, ny, nz, r, case["iterations"], st.OP_JACOBI, 0.0,
                                  u1.data_ptr() + 4 * at, u2.data_ptr() + 4 * at)
            at += nx * ny * nz
        even = case["iterations"] % 2 == 0
        return dict(kind=kind, probs=probs, u1=u1, u2=u2, result=u1 if even else u2, stream=st.Stream(),
                    mode=st.BATCH_GRAPH if case["mode"] == "graph" else st.BATCH_PERSISTENT)
    if kind == "layer":
        shape, x, w, b, gy = _layer_inputs(case, seed)
        ci, co = case["ci"], case["co"]
        wt = torch.empty((ci, nn.kpad(co)), device=DEV, dtype=torch.bfloat16)
        nn.wt_transpose(w.data_ptr(), wt.data_ptr(), ci, co)
        return dict(kind=kind, shape=shape, ci=ci, co=co, x=x, w=w, wt=wt, b=b, gy=gy,
                    out=torch.empty((*shape, co), device=DEV, dtype=torch.bfloat16),
                    g16=torch.empty((*shape, co), device=DEV, dtype=torch.bfloat16),
                    gx=torch.empty((*shape, ci), device=DEV),
                    gw=torch.empty((co, nn.kpad(ci)), device=DEV), gb=torch.empty(co, device=DEV))
    net = warmstart.UNet(case["batch"], case["n"])
    net.load_state_dict(_net_weights(seed))
    net.u.upload(_solved_fields(case, seed).cpu().numpy(), net.s)
    net.s.sync()
    return dict(kind=kind, net=net, smooth=case["smooth"], grads=_views(net))


class _DeviceView:
    def __init__(self, d):
        self.d = d
        self.__cuda_array_interface__ = dict(shape=d.shape, typestr=d.dtype.str, data=(d.ptr.value, False), version=2)


def _views(net):
    """torch views of the network's prediction, losses and gradients (its own buffers)."""
    t = lambda d: torch.as_tensor(_DeviceView(d), device=DEV)
    out = dict(pred=t(net.pred), loss=t(net.loss), sloss=t(net.sloss))
    for name, d in net.params.items():
        out[name + ".w"], out[name + ".b"] = t(d["gw"]), t(d["gb"])
    return out


# ---------------------------------------------------------------- one pass

SMOOTH_WEIGHT = 100.0


def run(state):
    kind = state["kind"]
    if kind == "sweep":
        u1, u2 = state["u"]
        if state["start"] is not None:
            u1.copy_(state["start"])
            u2.zero_()
        in_u2, _ = st.dispatch_kernels(state["p"], u1.data_ptr(), u2.data_ptr())
        res = u2 if in_u2 else u1
        if state["residual"]:
            return dict(field=res, norm=st.residual_norm(state["p"], res.data_ptr()))
        return res
    if kind == "mixed":
        x, u, (e1, e2, d) = state["x"], state["u"], state["e"]
        st.dispatch_mixed(state["p"], x.data_ptr(), e1.data_ptr(), e2.data_ptr(), d.data_ptr(), u.data_ptr())
        state["x"], state["u"] = u, x  # a further call goes on from the result
        return u
    if kind == "batched":
        st.dispatch_batched(state["probs"], (), state["mode"], state["stream"])
        return state["result"]
    if kind == "layer":
        s, ci, co = state["shape"], state["ci"], state["co"]
        x, out, g16, gx, gw, gb = (state[k] for k in ("x", "out", "g16", "gx", "gw", "gb"))
        pos = s[0] * s[1] * s[2] * s[3]
        nn.conv3(x.data_ptr(), state["w"].data_ptr(), state["b"].data_ptr(), out.data_ptr(), None, s, ci, co, relu=True)
        gw.zero_()
        gb.zero_()
        nn.relu_bwd(state["gy"].data_ptr(), out.data_ptr(), g16.data_ptr(), pos * co)
        nn.conv3_wgrad(x.data_ptr(), g16.data_ptr(), gw.data_ptr(), s, ci, co)
        nn.bias_grad(g16.data_ptr(), gb.data_ptr(), pos, co)
        nn.conv3(g16.data_ptr(), state["wt"].data_ptr(), None, None, gx.data_ptr(), s, co, ci)
        return dict(out=out, gw=gw, gb=gb, gx=gx)
    net = state["net"]
    net.forward(target=net.u)
    if state["smooth"]:
        net.add_smoothed_error_loss(net.u, state["smooth"], SMOOTH_WEIGHT)
    net.backward()
    if not state["smooth"]:
        return {k: v for k, v in state["grads"].items() if k != "sloss"}
    return state["grads"]


# ---------------------------------------------------------------- what a pass cannot do without

def _inner(ns, r):
    return math.prod(n - 2 * r for n in ns)


def work(case):
    kind = case["kind"]
    if kind == "sweep":
        ns, r, es = _shape(case), case["radius"], 8 if case["dtype"] == "f64" else 4
        ops = 2 * len(ns) * r + (1 if case["op"] == "jacobi" else 2)
        extra = ops + 3 if case["residual"] else 0
        return dict(bytes=2.0 * es * math.prod(ns), flops=float(_inner(ns, r)) * (case["iterations"] * ops + extra))
    if kind == "mixed":
        ns, r = _shape(case), case["radius"]
        return dict(bytes=8.0 * math.prod(ns), flops=float(_inner(ns, r)) * case["iterations"] * (6 * r + 2))
    if kind == "batched":
        shapes = _batch_shapes(case, 0)
        return dict(bytes=8.0 * sum(nx * ny * nz for nx, ny, nz, _ in shapes),
                    flops=float(sum(_inner(s[:3], s[3]) * (6 * s[3] + 1) for s in shapes)) * case["iterations"])
    if kind == "layer":
        pos, ci, co = case["n"] * case["d"] * case["h"] * case["w"], case["ci"], case["co"]
        return dict(bytes=float(pos * (2 * ci + 2 * co + 4 * co + 4 * ci) + 27 * ci * co * (2 + 2 + 4) + 8 * co),
                    flops=3.0 * 2 * 27 * ci * co * pos)
    n, b = case["n"], case["batch"]
    pos = [b * n ** 3, b * (n // 2) ** 3, b * (n // 4) ** 3]
    level = dict(e1a=0, e1b=0, e2a=1, e2b=1, bta=2, btb=2, d2a=1, d2b=1, d1a=0, d1b=0)
    macs = sum(27 * ci * co * pos[level[name]] * (2 if name == "e1a" else 3) for name, ci, co in NET)
    weights = sum(27 * ci * co + co for _, ci, co in NET) + 17
    return dict(bytes=8.0 * pos[0] + 8.0 * weights, flops=2.0 * macs + 2.0 * case["smooth"] * 7 * b * (n - 2) ** 3)


# ---------------------------------------------------------------- the same in 64 bits

def _star_sum(u, r):
    """Sum of the 2*D*r axis neighbours at the interior cells."""
    nd, acc = u.dim(), None
    for ax in range(nd):
        for d in range(1, r + 1):
            for sgn in (-d, d):
                idx = [slice(r, n - r) for n in u.shape]
                idx[ax] = slice(r + sgn, u.shape[ax] - r + sgn)
                v = u[tuple(idx)]
                acc = v.clone() if acc is None else acc.add_(v)
    return acc


def _iterate(a, b, r, iters, op):
    """iters sweeps ping-ponging between a and b; the result."""
    inner = tuple(slice(r, n - r) for n in a.shape)
    w = 1.0 / (2 * a.dim() * r)
    for _ in range(iters):
        s = _star_sum(a, r).mul_(w)
        b[inner] = s if op == "jacobi" else s - a[inner]
        a, b = b, a
    return a


def _taps(x, ci):
    """The 27 shifted views of a zero-padded channels-last tensor, as (positions, ci) matrices."""
    d, h, w = x.shape[1:4]
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    for t in range(27):
        z, y, q = t // 9, t // 3 % 3, t % 3
        yield t, xp[:, z:z + d, y:y + h, q:q + w].reshape(-1, ci)


class _Conv(torch.autograd.Function):
    """3x3x3 convolution, zero padding 1, weights (co, 27*ci) with k = tap*ci + channel."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        ci = x.shape[-1]
        out = torch.zeros((x[..., 0].numel(), w.shape[0]), dtype=x.dtype, device=x.device)
        for t, v in _taps(x, ci):
            out.addmm_(v, w[:, t * ci:(t + 1) * ci].t().contiguous())
        return out.view(*x.shape[:-1], w.shape[0])

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        ci, co = x.shape[-1], w.shape[0]
        gf = g.reshape(-1, co)
        gw = torch.cat([gf.t().contiguous() @ v for _, v in _taps(x, ci)], 1)
        gx = torch.zeros((gf.shape[0], ci), dtype=x.dtype, device=x.device)
        for t, v in _taps(g, co):
            k = 26 - t
            gx.addmm_(v, w[:, k * ci:(k + 1) * ci].contiguous())
        return gx.view(x.shape), gw


def _features(u):
    """Transfinite blend of the faces, shell value, coordinates, distance to the nearest face."""
    n = u.shape[-1]
    s = torch.arange(n, dtype=u.dtype, device=u.device) / (n - 1)
    sx, sy, sz = s.view(1, 1, 1, n), s.view(1, 1, n, 1), s.view(1, n, 1, 1)
    blend = ((1 - sx) * u[..., :1] + sx * u[..., -1:] + (1 - sy) * u[:, :, :1] + sy * u[:, :, -1:]
             + (1 - sz) * u[:, :1] + sz * u[:, -1:]) / 3
    shell = torch.ones_like(u, dtype=torch.bool)
    shell[:, 1:-1, 1:-1, 1:-1] = False
    zero = torch.zeros_like(u)
    dist = 2 * torch.minimum(torch.minimum(torch.minimum(sx, 1 - sx), torch.minimum(sy, 1 - sy)),
                             torch.minimum(sz, 1 - sz))
    feat = torch.stack([blend, torch.where(shell, u, zero), sx + zero, sy + zero, sz + zero, dist + zero, zero, zero], -1)
    return feat, torch.where(shell, u, blend), shell


def _exact_train(case, seed):
    u = _solved_fields(case, seed).double()
    sd = {k: torch.from_numpy(v).double().to(DEV).requires_grad_() for k, v in _net_weights(seed).items()}
    feat, base, shell = _features(u)
    conv = lambda name, x: torch.relu(_Conv.apply(x, sd[name + ".w"]) + sd[name + ".b"])

    def pool(x):
        b, d, h, w, c = x.shape
        return x.view(b, d // 2, 2, h // 2, 2, w // 2, 2, c).mean((2, 4, 6))

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    e1 = conv("e1b", conv("e1a", feat))
    e2 = conv("e2b", conv("e2a", pool(e1)))
    bt = conv("btb", conv("bta", pool(e2)))
    d2 = conv("d2b", conv("d2a", torch.cat([up(bt), e2], -1)))
    d1 = conv("d1b", conv("d1a", torch.cat([up(d2), e1], -1)))
    y = (d1 * sd["head.w"]).sum(-1) + sd["head.b"]
    pred = torch.where(shell, base, base + y)
    count = case["batch"] * (case["n"] - 2) ** 3
    loss = (pred - u).square().sum()
    total, out = loss / count, dict(pred=pred.detach().reshape(-1), loss=loss.detach().reshape(1))
    if case["smooth"]:
        e = pred - u
        for _ in range(case["smooth"]):
            s = sum(e[:, 1 + i:e.shape[1] - 1 + i, 1 + j:e.shape[2] - 1 + j, 1 + k:e.shape[3] - 1 + k]
                    for i, j, k in ((0, 0, -1), (0, 0, 1), (0, -1, 0), (0, 1, 0), (-1, 0, 0), (1, 0, 0))) / 6
            e = torch.nn.functional.pad(s, (1, 1, 1, 1, 1, 1))
        sl = e.square().sum()
        total = total + SMOOTH_WEIGHT / count * sl
        out["sloss"] = sl.detach().reshape(1)
    total.backward()
    for name, ci, co in NET:
        gw = torch.zeros((co, (27 * ci + 31) // 32 * 32), dtype=torch.float64, device=DEV)
        gw[:, :27 * ci] = sd[name + ".w"].grad
        out[name + ".w"], out[name + ".b"] = gw, sd[name + ".b"].grad
    out["head.w"], out["head.b"] = sd["head.w"].grad, sd["head.b"].grad
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "sweep":
        u1, u2 = (u.double() for u in _sweep_fields(case, seed))
        res = _iterate(u1, u2, case["radius"], case["iterations"], case["op"])
        if not case["residual"]:
            return res
        r = case["radius"]
        inner = res[tuple(slice(r, n - r) for n in res.shape)]
        norm = (_star_sum(res, r).mul_(1.0 / (2 * res.dim() * r)) - inner).square().sum().sqrt()
        return dict(field=res, norm=float(norm))
    if kind == "mixed":
        x = _shell_field(_shape(case), case["radius"], _gen(seed), torch.float32).double()
        return _iterate(x, x.clone(), case["radius"], case["iterations"], "jacobi")
    if kind == "batched":
        shapes, u, views = _batch_fields(case, seed)
        out = torch.empty(u.shape, dtype=torch.float64, device=DEV)
        at = 0
        for (_, _, _, r), v in zip(shapes, views):
            a = v.double()
            out[at:at + a.numel()] = _iterate(a, a.clone(), r, case["iterations"], "jacobi").reshape(-1)
            at += a.numel()
        return out
    if kind == "layer":
        shape, x, w, b, gy = _layer_inputs(case, seed)
        ci, co = case["ci"], case["co"]
        xd = x.double().requires_grad_()
        wd = w[:, :27 * ci].double().requires_grad_()
        bd = b.double().requires_grad_()
        out = torch.relu(_Conv.apply(xd, wd) + bd)
        out.backward(gy.double())
        gw = torch.zeros(w.shape, dtype=torch.float64, device=DEV)
        gw[:, :27 * ci] = wd.grad
        return dict(out=out.detach(), gw=gw, gb=bd.grad, gx=xd.grad)
    return _exact_train(case, seed)
