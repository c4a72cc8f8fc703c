"""The work whose speed counts: listed cases, a generator of more cases of the same ranges, and how
to prepare, run, size and check each one. Every pass goes through the package's public entry points
(kernels of the ParallelStencil language, the Stokes2D solvers, the adjoint inversion, the network).

Kinds of work:
  diffusion   one 3-D heat diffusion step, FP64, on-the-fly fluxes (plain, memopt, fastmath memopt)
  diffgrad    reverse-mode derivative launch of that step (@parallel ∇=...)
  acoustic    one 3-D acoustic step (compute_V!, compute_P!), FP64, FP32 or BFloat16 storage
  inversion   misfit and gradient of the 2-D acoustic inversion (forward, recompute, adjoint)
  stokes      one block of pseudo-transient Stokes2D iterations and its residual check
  stokesbatch the same for many samples per launch
  conv        one 3x3 convolution layer of the network, forward and backward
  unet        network inference on one or more samples
  train       one training step of the network (forward, loss, backward, Adam)
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "parallelstencil.jl_amd"))

import parallelstencil as ps  # noqa: E402
from parallelstencil import acoustic_adjoint as AA  # noqa: E402
from parallelstencil import stokes_fused as SF  # noqa: E402
from parallelstencil import unet as U  # noqa: E402
from parallelstencil import workloads as W  # noqa: E402
from parallelstencil._lib import check, lib  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------------------------- cases
def listed():
    return [
        # the first thing a user runs (and the launch-bound end of a convergence study): one blocking
        # @parallel call on a 32^3 grid
        dict(name="diffusion_32_plain", kind="diffusion", nx=32, ny=32, nz=32, variant="plain"),
        # an ordinary grid with odd extents, plain kernel, blocking call
        dict(name="diffusion_253x190x127_plain", kind="diffusion", nx=253, ny=190, nz=127, variant="plain"),
        # the headline size: time loop of prepared memopt launches with fastmath
        dict(name="diffusion_512_fastmath", kind="diffusion", nx=512, ny=512, nz=512, variant="fastmath"),
        # sensitivity of a diffusion step: reverse-mode derivative of the memopt kernel
        dict(name="diffgrad_256", kind="diffgrad", nx=256, ny=256, nz=256),
        # wave propagation at the miniapp's benchmark size, single precision
        dict(name="acoustic_384_f32", kind="acoustic", nx=384, ny=384, nz=384, dtype="Float32"),
        # wave propagation in BFloat16 storage on a ragged grid
        dict(name="acoustic_383x255x319_bf16", kind="acoustic", nx=383, ny=255, nz=319, dtype="BFloat16"),
        # one gradient evaluation of the acoustic inversion, as an optimiser calls it
        dict(name="inversion_1024x64", kind="inversion", nx=1024, ny=1024, nt=64),
        # the resolution at which the learned warm start serves the Stokes solver
        dict(name="stokes_511", kind="stokes", nx=511, ny=511, nout=200),
        # training-data generation: 64 samples per launch at the training resolution
        dict(name="stokesbatch_127x64", kind="stokesbatch", nx=127, ny=127, S=64, nout=200),
        # a full-resolution layer of the network in training
        dict(name="conv_32_32_8x128", kind="conv", B=8, H=128, W=128, cin=32, cout=32),
        # inference for one 511^2 sample
        dict(name="unet_1x512", kind="unet", B=1, H=512, W=512, base=32),
        # a training step at the training resolution
        dict(name="train_8x128", kind="train", B=8, H=128, W=128, base=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["diffusion", "diffusion", "diffgrad", "acoustic", "acoustic", "inversion", "stokes", "stokesbatch", "conv", "conv",
                       "unet", "train"])
    if kind in ("diffusion", "diffgrad", "acoustic"):
        # 3-D grids of 24 to 512 (256 for the derivative) cells per side, no two sides tied
        top = {"diffusion": 512, "diffgrad": 256, "acoustic": 384}[kind]
        c = dict(kind=kind, nx=_log(rng, 24, top), ny=_log(rng, 24, top), nz=_log(rng, 24, top))
        if kind == "diffusion":
            c["variant"] = rng.choice(["plain", "memopt", "fastmath"])
        if kind == "acoustic":
            c["dtype"] = rng.choice(["Float64", "Float32", "BFloat16"])
        return c
    if kind == "inversion":
        return dict(kind=kind, nx=_log(rng, 192, 1024), ny=_log(rng, 192, 1024), nt=rng.randint(24, 64))
    if kind == "stokes":
        return dict(kind=kind, nx=_log(rng, 31, 511), ny=_log(rng, 31, 511), nout=200)
    if kind == "stokesbatch":
        n = _log(rng, 31, 255)
        return dict(kind=kind, nx=n, ny=n, S=max(1, min(64, int(rng.uniform(0.3, 1.0) * 64 * 127 * 127 / (n * n)))), nout=200)
    if kind == "conv":
        # layers of the network's levels: more channels at lower resolution; odd image sizes and,
        # as in the first layer and in networks of other widths, other channel counts
        H = _log(rng, 9, 160)
        cin, cout = (rng.choice([2, 3, 24, 32, 40, 48, 64, 96, 128, 192, 256]) for _ in range(2))
        Wd = max(8, int(H * rng.uniform(0.6, 1.5)))
        B = max(1, min(8, int(131072 * 32 * 32 * 2 / (H * Wd * cin * cout))))
        return dict(kind=kind, B=B, H=H, W=Wd, cin=cin, cout=cout)
    if kind == "unet":
        H, Wd = 8 * _log(rng, 4, 64), 8 * _log(rng, 4, 64)
        return dict(kind=kind, B=max(1, min(rng.choice([1, 1, 2, 8]), 512 * 512 // (H * Wd))), H=H, W=Wd, base=rng.choice([16, 24, 32]))
    H, Wd = 8 * _log(rng, 4, 16), 8 * _log(rng, 4, 16)
    return dict(kind="train", B=rng.randint(1, 8), H=H, W=Wd, base=rng.choice([16, 24, 32]))


# ---------------------------------------------------------------------------------- device memory
class _Mem:
    """Device memory of `owner` (which the tensor made of it keeps alive)."""

    def __init__(self, owner, ptr, shape, strides, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, strides=strides, typestr=typestr, data=(ptr, False), version=2)


_TYPES = {"Float64": ("<f8", torch.float64, 8), "Float32": ("<f4", torch.float32, 4), "BFloat16": ("<i2", torch.bfloat16, 2)}


def _field(A):
    """The field's own memory as a tensor [z][y][x] (or [y][x]), without a copy."""
    ts, dt, sz = _TYPES[A.eltype]
    st = (sz, int(A.f.pitch) * sz, int(A.f.plane) * sz)[:A.ndim]
    t = torch.as_tensor(_Mem(A, A.ptr, A.shape[::-1], st[::-1], ts), device=DEV)
    return t.view(dt) if t.dtype != dt else t


def _buf(b):
    """A network buffer's own memory as a tensor, without a copy."""
    n = b.n
    t = torch.as_tensor(_Mem(b, b.p.value, (n,), (2 if b.dtype == "bf16" else 4,), "<i2" if b.dtype == "bf16" else "<f4"), device=DEV)
    return (t.view(torch.bfloat16) if b.dtype == "bf16" else t).view(b.shape)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _module(numbertype, ndims):
    m = f"perf.{numbertype}.{ndims}"
    if not ps.is_initialized(module=m):
        ps.init_parallel_stencil(ps.AMDGPU, numbertype, ndims, module=m)
    return m


# ---------------------------------------------------------------------------------- inputs
def _bumps(g, shape, spacing, lx):
    """Three Gaussian bumps on the cells [z][y][x] of a box, random centres, heights and widths."""
    nz, ny, nx = shape
    ax = [torch.arange(n, device=DEV, dtype=torch.float64) * spacing for n in (nz, ny, nx)]
    out = torch.zeros(shape, device=DEV, dtype=torch.float64)
    for _ in range(3):
        c, w, h = _rand(g, 3).tolist(), 0.1 * lx * (0.5 + _rand(g, 1).item()), 0.5 + _rand(g, 1).item()
        e = [torch.exp(-((a - ci * a[-1]) / w) ** 2) for a, ci in zip(ax, c)]
        out += h * e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
    return out


def _diffusion_inputs(case, seed):
    g = _gen(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    dx = 10.0 / max(shape)
    T = 100.0 * _bumps(g, shape, dx, 10.0)
    Cp = 1.0 + _rand(g, *shape)
    return T, Cp, (1.0, dx * dx / 8.1, dx, dx, dx)


def _acoustic_inputs(case, seed):
    g = _gen(seed)
    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    dx = 40.0 / (max(nx, ny, nz) - 1)
    P = _bumps(g, (nz, ny, nx), dx, 40.0)
    Vx, Vy, Vz = (0.2 * _bumps(g, s, dx, 40.0) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)))
    dt = torch.float64 if case["dtype"] == "Float64" else torch.float32 if case["dtype"] == "Float32" else torch.bfloat16
    return [A.to(dt) for A in (P, Vx, Vy, Vz)], (dx / 6.1, 1.0, 1.0, dx)


def _inversion_inputs(case, seed):
    s = AA.Setup(case["nx"], case["ny"], case["nt"], seed=int(seed) + 1, nrec=min(64, case["nx"] // 4), sigma=case["nx"] / 20.0)
    return s, np.asfortranarray(1.0 + 0.5 * (s.K - 1.0))


def _seed64(seed, k):
    return (1000 * int(seed) + k + 1) % (1 << 62)


def _stokes_material(case, seed, k=0):
    return W.stokes2d_inclusions(case["nx"], case["ny"], _seed64(seed, k), log10_contrast=0.8)


def _net_inputs(case, seed):
    """log10 viscosity and body force of B inclusion samples, [B][H][W][2]."""
    X = np.empty((case["B"], case["H"], case["W"], 2), np.float32)
    for b in range(case["B"]):
        Mus, Rog = W.stokes2d_inclusions(case["W"], case["H"], _seed64(seed, b), log10_contrast=2.0)
        X[b, :, :, 0], X[b, :, :, 1] = np.log10(Mus).T, Rog.T
    return X


def _net_targets(case, seed):
    """Smooth normalised target fields and their mask (the padded rows and columns do not count)."""
    g = _gen(seed)
    B, H, Wd = case["B"], case["H"], case["W"]
    y, x = torch.arange(H, device=DEV, dtype=torch.float64) / H, torch.arange(Wd, device=DEV, dtype=torch.float64) / Wd
    T = torch.zeros(B, H, Wd, 3, device=DEV, dtype=torch.float64)
    for _ in range(3):
        k, ph, a = 1 + 3 * _rand(g, B, 1, 1, 3, 2), 6.28 * _rand(g, B, 1, 1, 3, 2), _rand(g, B, 1, 1, 3)
        T += a * torch.sin(6.28 * k[..., 0] * x[None, None, :, None] + ph[..., 0]) * torch.cos(6.28 * k[..., 1] * y[None, :, None, None] + ph[..., 1])
    Mk = torch.ones_like(T)
    Mk[:, H - 7:], Mk[:, :, Wd - 7:] = 0, 0
    return T.float(), Mk.float()


# ---------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    ps.ensure_device()
    s = globals()["_prepare_" + case["kind"]](case, int(seed))
    s["kind"] = case["kind"]
    torch.cuda.synchronize()
    return s


def _prepare_diffusion(case, seed):
    mod = _module(ps.Float64, 3)
    kw = {"plain": dict(memopt=False), "memopt": dict(memopt=True), "fastmath": dict(memopt=True, fastmath=True)}[case["variant"]]
    k = W.define_diffusion3d(kw.pop("memopt"), mod, **kw)
    T0, Cp0, sc = _diffusion_inputs(case, seed)
    T, T2, Cp = (ps.zeros(case["nx"], case["ny"], case["nz"], eltype=ps.Float64) for _ in range(3))
    tT, tT2, tC = _field(T), _field(T2), _field(Cp)
    tT.copy_(T0), tT2.copy_(T0), tC.copy_(Cp0)
    k.precompile_launch(T2, T, Cp, *sc)
    s = dict(k=k, T=T, T2=T2, Cp=Cp, tT=tT, tT2=tT2, sc=sc)
    if case["variant"] == "fastmath":  # a time loop of prepared launches, T and T2 in turn
        s["loop"] = [k.launcher(T2, T, Cp, *sc), k.launcher(T, T2, Cp, *sc)]
    return s


def _prepare_diffgrad(case, seed):
    k = W.define_diffusion3d(True, _module(ps.Float64, 3))
    T0, Cp0, sc = _diffusion_inputs(case, seed)
    g = _gen(seed + 7919)
    T, T2, Cp, Tb, T2b = (ps.zeros(case["nx"], case["ny"], case["nz"], eltype=ps.Float64) for _ in range(5))
    tT2b, tTb = _field(T2b), _field(Tb)
    _field(T).copy_(T0), _field(T2).copy_(T0), _field(Cp).copy_(Cp0)
    seedT = _rand(g, *tT2b.shape) - 0.5
    tT2b.copy_(seedT)
    return dict(k=k, a=(T2, T, Cp) + sc, T=T, T2=T2, Tb=Tb, T2b=T2b, tTb=tTb, tT2b=tT2b)


def _prepare_acoustic(case, seed):
    nt = ps.Float64 if case["dtype"] == "Float64" else ps.Float32
    mod = _module(nt, 3)
    kV, kP = W.define_acoustic3d(mod)
    (P0, *V0), (dt, rho, k, dx) = _acoustic_inputs(case, seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    P, Vx, Vy, Vz = (ps.zeros(*d, eltype=case["dtype"]) for d in ((nx, ny, nz), (nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)))
    out = [_field(A) for A in (P, Vx, Vy, Vz)]
    for t, h in zip(out, [P0] + V0):
        t.copy_(h)
    kV.precompile_launch(Vx, Vy, Vz, P, dt, rho, dx, dx, dx)
    kP.precompile_launch(P, Vx, Vy, Vz, dt, k, dx, dx, dx)
    return dict(V=kV.launcher(Vx, Vy, Vz, P, dt, rho, dx, dx, dx), P=kP.launcher(P, Vx, Vy, Vz, dt, k, dx, dx, dx), out=out)


def _prepare_inversion(case, seed):
    s, K0 = _inversion_inputs(case, seed)
    inv = AA.Acoustic2DInversion(_module(ps.Float32, 2), s)
    inv.set_observed(inv.forward(s.K))
    return dict(inv=inv, K0=K0)


def _prepare_stokes(case, seed):
    sv = SF.Stokes2DFused(_module(ps.Float64, 2), case["nx"], case["ny"], nout=case["nout"], eta_ts="maxV")
    sv.iterate_block()  # the solver of a running program: its graph exists, the sample is new
    sv.set_material(*_stokes_material(case, seed))
    sv.reset()
    names = ("Vx", "Vy", "Pt", "dVxdt", "dVydt", "txx", "tyy", "txy", "Rx", "Ry", "divV")
    return dict(sv=sv, out={n: _field(getattr(sv, n)) for n in names})


def _prepare_stokesbatch(case, seed):
    sv = SF.Stokes2DBatch(_module(ps.Float64, 3), case["nx"], case["ny"], case["S"], nout=case["nout"], eta_ts="maxV")
    sv.iterate_block()
    ms = [_stokes_material(case, seed, k) for k in range(case["S"])]
    sv.set_material(np.asfortranarray(np.stack([m[0] for m in ms], -1)), np.asfortranarray(np.stack([m[1] for m in ms], -1)))
    sv.reset()
    names = ("Vx", "Vy", "Pt", "dVxdt", "dVydt", "txx", "tyy", "txy", "Rx", "Ry", "divV")
    return dict(sv=sv, out={n: _field(getattr(sv, n)) for n in names})


def _prepare_conv(case, seed):
    B, H, Wd, cin, cout = (case[n] for n in ("B", "H", "W", "cin", "cout"))
    layer = U.Conv(cin, cout, np.random.default_rng(seed), k=3, relu=True)
    x, dy = U.Buf((B, H, Wd, cin)), U.Buf((B, H, Wd, cout))
    layer.forward(x, B, H, Wd)  # the layer of a running program: its buffers exist, the inputs are new
    layer.backward(dy)
    torch.cuda.synchronize()
    x0, dy0, b0 = _conv_inputs(case, seed)
    _buf(x).copy_(x0), _buf(dy).copy_(dy0), _buf(layer.b).copy_(b0)
    return dict(layer=layer, x=x, dy=dy, g=(B, H, Wd))


def _conv_inputs(case, seed):
    g = _gen(seed)
    B, H, Wd = case["B"], case["H"], case["W"]
    r = lambda *s: torch.randn(*s, generator=g, device=DEV, dtype=torch.float32)  # noqa: E731
    return (torch.relu(r(B, H, Wd, case["cin"])).bfloat16(), (r(B, H, Wd, case["cout"]) * 1e-3).bfloat16(), 0.1 * r(case["cout"]))


def _prepare_unet(case, seed):
    net = U.UNet(base=case["base"], cin=2, seed=seed)
    B, H, Wd = case["B"], case["H"], case["W"]
    x = U.Buf((B, H, Wd, 2))
    net.forward(x, B, H, Wd)  # the network of a running program: its buffers exist, the samples are new
    torch.cuda.synchronize()
    x.upload(_net_inputs(case, seed))
    return dict(net=net, x=x, g=(B, H, Wd))


def _prepare_train(case, seed):
    s = _prepare_unet(case, seed)
    T, Mk = _net_targets(case, seed)
    sh = (case["B"], case["H"], case["W"], 3)
    s.update(t=U.Buf(sh, "f32"), m=U.Buf(sh, "f32"), dout=U.Buf(sh), loss=U.Buf((1,), "f32"), scale=1.0 / float(Mk.sum().item()))
    _buf(s["t"]).copy_(T), _buf(s["m"]).copy_(Mk)
    s["net"].backward(s["dout"])
    return s


# ---------------------------------------------------------------------------------- run
def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_diffusion(s):
    if "loop" in s:
        s["loop"][0]()
        s["loop"].reverse()
    else:
        s["k"](s["T2"], s["T"], s["Cp"], *s["sc"])
        s["T"], s["T2"] = s["T2"], s["T"]
    s["tT"], s["tT2"] = s["tT2"], s["tT"]
    return s["tT"]


def _run_diffgrad(s):
    s["k"](*s["a"], grad=[(s["T2"], s["T2b"]), (s["T"], s["Tb"])], ad_mode=ps.AD.Reverse)
    # a chain of steps feeds the adjoint of T to the step before it, whose seed it is
    s["T2b"], s["Tb"], s["tT2b"], s["tTb"] = s["Tb"], s["T2b"], s["tTb"], s["tT2b"]
    return s["tT2b"], s["tTb"]


def _run_acoustic(s):
    s["V"]()
    s["P"]()
    return s["out"]


def _run_inversion(s):
    return s["inv"].gradient(s["K0"])


def _run_stokes(s):
    s["sv"].iterate_block()
    return s["out"], s["sv"].error()


def _run_stokesbatch(s):
    s["sv"].iterate_block()
    return s["out"], s["sv"].errors()


def _run_conv(s):
    layer = s["layer"]
    y = layer.forward(s["x"], *s["g"])
    layer.gw.zero()
    layer.gb.zero()
    dx = layer.backward(s["dy"])
    return tuple(_buf(b) for b in (y, dx, layer.gw, layer.gb))


def _run_unet(s):
    return _buf(s["net"].forward(s["x"], *s["g"]))


def _run_train(s):
    net = s["net"]
    y = net.forward(s["x"], *s["g"])
    s["loss"].zero()
    check(lib.ps_nn_mse(y.p, s["t"].p, s["m"].p, y.n, s["scale"], s["dout"].p, s["loss"].p, None))
    net.zero_grad()
    net.backward(s["dout"])
    net.adam(1e-5)  # late in the decay of the schedule
    L = net.layers()
    return dict(pred=_buf(y), loss=_buf(s["loss"]), gw=[_buf(l.gw) for l in L], gb=[_buf(l.gb) for l in L], w=[_buf(l.w) for l in L])


# ---------------------------------------------------------------------------------- work
def _convs(base, cout=3, cin=2):
    """(cin, cout, kernel size, level) of the network's layers."""
    c = [base, 2 * base, 4 * base, 8 * base]
    L = []
    for l in range(4):
        L += [(cin if l == 0 else c[l - 1], c[l], 3, l), (c[l], c[l], 3, l)]
    for l in (2, 1, 0):
        L += [(c[l + 1] + c[l], c[l], 3, l), (c[l], c[l], 3, l)]
    return L + [(c[0], cout, 1, 0)]


def work(case):
    kind = case["kind"]
    if kind in ("diffusion", "diffgrad", "acoustic"):
        n = case["nx"] * case["ny"] * case["nz"]
        if kind == "diffusion":  # T, Cp read, T2 written
            return dict(bytes=3 * 8 * n, flops=22 * n)
        if kind == "diffgrad":  # seed and Cp read, seed cleared, the adjoint of T read and written
            return dict(bytes=5 * 8 * n, flops=30 * n)
        return dict(bytes=8 * {"Float64": 8, "Float32": 4, "BFloat16": 2}[case["dtype"]] * n, flops=24 * n)  # P, Vx, Vy, Vz read and written
    if kind == "inversion":
        n, nt = case["nx"] * case["ny"], case["nt"]
        return dict(bytes=2 * 8 * n, flops=(2 * 14 + 22) * n * nt)  # K in, the gradient out; two forward passes and the adjoint
    if kind in ("stokes", "stokesbatch"):
        n = case["nx"] * case["ny"] * case.get("S", 1)
        # state (3 + 2 arrays), steps (3), viscosity and force (2) in; state and residual fields (11) out
        return dict(bytes=(10 + 11) * 8 * n, flops=55 * n * case["nout"])
    if kind == "conv":
        p, ci, co = case["B"] * case["H"] * case["W"], case["cin"], case["cout"]
        # x, dy, weights in; y, dx, weight and bias gradients out
        return dict(bytes=2 * p * 2 * (ci + co) + 9 * ci * co * (2 + 4) + 8 * co, flops=3 * 2 * 9 * ci * co * p)
    p = case["B"] * case["H"] * case["W"]
    L = _convs(case["base"])
    fl = sum(2 * k * k * ci * co * (p >> (2 * l)) for ci, co, k, l in L)
    nw = sum(k * k * ci * co + co for ci, co, k, l in L)
    if kind == "unet":
        return dict(bytes=p * 2 * (2 + 3) + 2 * nw, flops=fl)
    # inputs, targets, masks in; weights, moments in and out, gradients out
    return dict(bytes=p * (2 * 2 + 3 * 4 * 2 + 2 * 3) + nw * (6 * 4 + 4), flops=3 * fl - 2 * 9 * 2 * case["base"] * p)


# ---------------------------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    if kind in ("diffusion", "diffgrad"):
        return {"rel": 1e-12, "max": 1e-11}
    if kind == "acoustic":
        return {"Float64": {"rel": 1e-12, "max": 1e-11}, "Float32": {"rel": 2e-7, "max": 2e-6}, "BFloat16": {"rel": 5e-3, "max": 5e-2}}[case["dtype"]]
    if kind == "inversion":  # FP32 traces against observed ones: their difference carries the rounding
        return {"rel": 1e-5, "max": 5e-4}
    if kind in ("stokes", "stokesbatch"):  # 200 iterations in FP64
        return {"rel": 1e-10, "max": 1e-8}
    if kind == "conv":
        return {"rel": 5e-3, "max": 5e-2}
    if kind == "unet":  # BF16 activations through 15 layers
        return {"rel": 2e-2, "max": 0.5}
    return {"rel": 3e-2, "max": 0.9}  # and back through them


# ---------------------------------------------------------------------------------- exact
def exact(case, seed):
    r = globals()["_exact_" + case["kind"]](case, int(seed))
    torch.cuda.synchronize()
    return r


def _d(A, dim):
    """Difference of neighbours along `dim` (0 x, 1 y, 2 z of a tensor whose last axis is x)."""
    ax = A.dim() - 1 - dim
    n = A.shape[ax]
    return A.narrow(ax, 1, n - 1) - A.narrow(ax, 0, n - 1)


def _exact_diffusion(case, seed):
    T, Cp, (lam, dt, dx, dy, dz) = _diffusion_inputs(case, seed)
    c = slice(1, -1)
    div = (_d(-lam * _d(T[c, c, :], 0) / dx, 0) / dx + _d(-lam * _d(T[c, :, c], 1) / dy, 1) / dy + _d(-lam * _d(T[:, c, c], 2) / dz, 2) / dz)
    T2 = T.clone()
    T2[c, c, c] = T[c, c, c] - dt / Cp[c, c, c] * div
    return T2


def _exact_diffgrad(case, seed):
    T, Cp, (lam, dt, dx, dy, dz) = _diffusion_inputs(case, seed)
    s = _rand(_gen(seed + 7919), *T.shape) - 0.5
    c = slice(1, -1)
    w = torch.zeros_like(T)
    w[c, c, c] = s[c, c, c] * dt / Cp[c, c, c] * lam
    out = torch.zeros_like(T)
    out[c, c, c] = s[c, c, c]
    for ax, h in ((2, dx), (1, dy), (0, dz)):  # transpose of the 3-point second difference along each axis
        n = T.shape[ax]
        out -= 2.0 * w / (h * h)
        out.narrow(ax, 0, n - 1).add_(w.narrow(ax, 1, n - 1) / (h * h))
        out.narrow(ax, 1, n - 1).add_(w.narrow(ax, 0, n - 1) / (h * h))
    s[c, c, c] = 0.0
    return out, s


def _exact_acoustic(case, seed):
    A, (dt, rho, k, dx) = _acoustic_inputs(case, seed)
    P, Vx, Vy, Vz = (a.double() for a in A)
    c = slice(1, -1)
    Vx[c, c, c] -= dt / rho * _d(P[c, c, :], 0) / dx
    Vy[c, c, c] -= dt / rho * _d(P[c, :, c], 1) / dx
    Vz[c, c, c] -= dt / rho * _d(P[:, c, c], 2) / dx
    P = P - dt * k * (_d(Vx, 0) / dx + _d(Vy, 1) / dx + _d(Vz, 2) / dx)
    return [P, Vx, Vy, Vz]


def _exact_inversion(case, seed):
    s, K0 = _inversion_inputs(case, seed)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.float64).T)).to(DEV)  # noqa: E731
    c = slice(1, -1)
    dt, rho, dx, dy = s.dt, s.rho, s.dx, s.dy
    rx = torch.arange(s.nrec, device=DEV) * s.rdx + s.rx0 - 1
    ry, sx, sy = s.ry - 1, s.isx - 1, s.isy - 1

    def forward(K, keep):
        P = torch.zeros(s.ny, s.nx, device=DEV, dtype=torch.float64)
        Vx, Vy = torch.zeros(s.ny, s.nx + 1, device=DEV, dtype=torch.float64), torch.zeros(s.ny + 1, s.nx, device=DEV, dtype=torch.float64)
        D, V = [], []
        for n in range(s.nt):
            Vx[c, c] -= dt / rho * _d(P[c, :], 0) / dx
            Vy[c, c] -= dt / rho * _d(P[:, c], 1) / dy
            div = _d(Vx, 0) / dx + _d(Vy, 1) / dy
            P = P - dt * K * div
            P[sy, sx] += float(s.src[n])
            D.append(P[ry, rx].clone())
            if keep:
                V.append(div)
        return torch.stack(D), V

    Dobs, _ = forward(dev(s.K), False)
    K = dev(K0)
    D, V = forward(K, True)
    r = D - Dobs
    lP = torch.zeros(s.ny, s.nx, device=DEV, dtype=torch.float64)
    lVx, lVy = torch.zeros(s.ny, s.nx + 1, device=DEV, dtype=torch.float64), torch.zeros(s.ny + 1, s.nx, device=DEV, dtype=torch.float64)
    g = torch.zeros_like(lP)
    for n in reversed(range(s.nt)):
        lP[ry, rx] += r[n]
        g -= dt * lP * V[n]
        Wk = K * lP
        lVx[c, c] += dt * _d(Wk[c, :], 0) / dx
        lVy[c, c] += dt * _d(Wk[:, c], 1) / dy
        lP = lP + dt / rho * (_d(lVx, 0) / dx + _d(lVy, 1) / dy)
    return 0.5 * float((r * r).sum()), g.T.contiguous().cpu().numpy()


def _exact_stokes_fields(case, Mus, Rog):
    """`nout` pseudo-transient iterations from rest of [S][y][x] samples."""
    nx, ny = case["nx"], case["ny"]
    lead = Mus.shape[:-2]
    dx, dy = 10.0 / (nx - 1), 10.0 / (ny - 1)
    m2, mx = min(dx, dy) ** 2, max(nx, ny)
    dampX, dampY = 1.0 - 4.0 / nx, 1.0 - 4.0 / ny
    c = slice(1, -1)
    big = F.max_pool2d(Mus.reshape(-1, 1, ny, nx), 3, 1, 1).reshape(Mus.shape)
    av = lambda A, ax: 0.5 * (A.narrow(ax, 0, A.shape[ax] - 1) + A.narrow(ax, 1, A.shape[ax] - 1))  # noqa: E731
    tx, ty, tp = m2 / av(big[..., c, :], -1) / 4.1, m2 / av(big[..., :, c], -2) / 4.1, 0.25 * 4.1 * Mus / mx
    mun = av(av(Mus, -1), -2)
    z = lambda a, b: torch.zeros(*lead, b, a, device=DEV, dtype=torch.float64)  # noqa: E731
    Pt, Vx, Vy, ax_, ay_ = z(nx, ny), z(nx + 1, ny), z(nx, ny + 1), z(nx - 1, ny - 2), z(nx - 2, ny - 1)
    for _ in range(case["nout"]):
        ex, ey = _d(Vx, 0) / dx, _d(Vy, 1) / dy
        div = ex + ey
        Pt = Pt - tp * div
        txx, tyy = 2.0 * Mus * (ex - div / 3.0), 2.0 * Mus * (ey - div / 3.0)
        txy = mun * (_d(Vx[..., :, c], 1) / dy + _d(Vy[..., c, :], 0) / dx)
        Rx = _d(txx[..., c, :], 0) / dx + _d(txy, 1) / dy - _d(Pt[..., c, :], 0) / dx
        Ry = _d(tyy[..., :, c], 1) / dy + _d(txy, 0) / dx - _d(Pt[..., :, c], 1) / dy + av(Rog[..., :, c], -2)
        ax_, ay_ = dampX * ax_ + Rx, dampY * ay_ + Ry
        Vx[..., c, c] += tx * ax_
        Vy[..., c, c] += ty * ay_
        Vx[..., 0, :], Vx[..., -1, :] = Vx[..., 1, :], Vx[..., -2, :]
        Vy[..., :, 0], Vy[..., :, -1] = Vy[..., :, 1], Vy[..., :, -2]
    m = lambda A: A.abs().mean(dim=(-2, -1))  # noqa: E731
    err = torch.maximum(torch.maximum(m(Rx), m(Ry)), m(div))
    return dict(Vx=Vx, Vy=Vy, Pt=Pt, dVxdt=ax_, dVydt=ay_, txx=txx, tyy=tyy, txy=txy, Rx=Rx, Ry=Ry, divV=div), err


def _exact_stokes(case, seed):
    Mus, Rog = (torch.from_numpy(np.ascontiguousarray(a.T)).to(DEV) for a in _stokes_material(case, seed))
    f, err = _exact_stokes_fields(case, Mus, Rog)
    return f, float(err)


def _exact_stokesbatch(case, seed):
    ms = [_stokes_material(case, seed, k) for k in range(case["S"])]
    Mus, Rog = (torch.from_numpy(np.ascontiguousarray(np.stack([m[i].T for m in ms]))).to(DEV) for i in (0, 1))
    f, err = _exact_stokes_fields(case, Mus, Rog)
    return f, err.cpu().numpy()


def _conv3(x, w, b):
    """3x3 convolution of [B][H][W][C] with weights [9*Cin][Cout], in 64 bits: nine shifted products."""
    B, H, Wd, C = x.shape
    p = F.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(B, H, Wd, -1)
    for t in range(9):
        y = y + p[:, t // 3:t // 3 + H, t % 3:t % 3 + Wd].reshape(-1, C).matmul(w[t * C:(t + 1) * C]).view(B, H, Wd, -1)
    return y


def _exact_conv(case, seed):
    std = math.sqrt(2.0 / (9 * case["cin"]))
    w0 = (np.random.default_rng(seed).standard_normal((9 * case["cin"], case["cout"])) * std).astype(np.float32)
    x0, dy0, b0 = _conv_inputs(case, seed)
    x = x0.double().requires_grad_()
    w = torch.from_numpy(w0).to(DEV).bfloat16().double().requires_grad_()
    b = b0.double().requires_grad_()
    y = torch.relu(_conv3(x, w, b))
    dx, gw, gb = torch.autograd.grad(y, (x, w, b), dy0.double())
    return y.detach(), dx, gw, gb


def _net_params(case, seed):
    rng = np.random.default_rng(seed)
    base, P = case["base"], {}
    c = [base, 2 * base, 4 * base, 8 * base]
    order = [("e", l, i) for l in range(4) for i in range(2)] + [("d", l, i) for l in range(3) for i in range(2)] + [("h", 0, 0)]
    for n in order:  # the order in which the network draws its weights
        kind, l, i = n
        ci = (2 if l == 0 else c[l - 1]) if kind == "e" else c[l + 1] + c[l] if kind == "d" else c[0]
        ci, co, k = (c[l] if i else ci), (c[l] if kind != "h" else 3), (1 if kind == "h" else 3)
        w = (rng.standard_normal((k * k * ci, co)) * math.sqrt(2.0 / (k * k * ci))).astype(np.float32)
        P[n] = (torch.from_numpy(w).to(DEV).bfloat16().double().requires_grad_(), torch.zeros(co, device=DEV, dtype=torch.float64, requires_grad=True))
    return P, order


def _net(P, x):
    conv = lambda n, h: torch.relu(_conv3(h, *P[n]))  # noqa: E731
    skips, h = [], x
    for l in range(4):
        h = conv(("e", l, 1), conv(("e", l, 0), h))
        if l < 3:
            skips.append(h)
            h = (h[:, ::2, ::2] + h[:, 1::2, ::2] + h[:, ::2, 1::2] + h[:, 1::2, 1::2]) * 0.25
    for l in (2, 1, 0):
        h = torch.cat([h.repeat_interleave(2, 1).repeat_interleave(2, 2), skips[l]], -1)
        h = conv(("d", l, 1), conv(("d", l, 0), h))
    w, b = P[("h", 0, 0)]
    return h.matmul(w) + b


def _exact_unet(case, seed):
    P, _ = _net_params(case, seed)
    with torch.no_grad():
        return _net(P, torch.from_numpy(_net_inputs(case, seed)).to(DEV).bfloat16().double())


def _exact_train(case, seed):
    P, order = _net_params(case, seed)
    T, Mk = _net_targets(case, seed)
    y = _net(P, torch.from_numpy(_net_inputs(case, seed)).to(DEV).bfloat16().double())
    scale = 1.0 / float(Mk.sum().item())
    loss = scale * (Mk.double() * (y - T.double()) ** 2).sum()
    g = torch.autograd.grad(loss, [t for n in order for t in P[n]])
    # the updated weights follow the sign of every single gradient value: no value in 64 bits to hold them to
    return dict(pred=y.detach(), loss=loss.detach().view(1), gw=list(g[0::2]), gb=list(g[1::2]), w=[None] * len(order))
