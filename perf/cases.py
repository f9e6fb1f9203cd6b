"""Timed workloads of the framework, through its public entry points.

Each case is one call that a user's program makes again and again:

* ``steady``    a steady confined model's time step on a kept handle: formulate, row fixes, ILU0 factor, CG and
                the outer loop, from start heads that a coupler holds on the GPU (``GwfSolution.run_timestep`` with
                ``mf6hip_gwf_set_x_device`` / ``get_x_device``).  With ``budget`` the step also reads the heads and
                the cell-by-cell flows to the host, as a program that saves both files every step does.
* ``newton``    time steps of the unconfined transient Newton model (BiCGSTAB + ILU0, storage, drains, recharge,
                wells), FP64 or mixed precision.
* ``dropin``    the drop-in linear solve on host arrays in the reference's CSR layout (``HipLinearSolver.solve``),
                which is what a host that keeps its own formulate calls every outer iteration.
* ``learned``   the same call with the flexible CG and an attached network.
* ``ensemble``  every realisation of an ensemble solved at once (``Ensemble.solve``).
* ``forward``, ``grad``, ``train``  the network of the learned preconditioner: one application on host planes, one
                loss and gradient, and Adam steps on samples stored on the device.

Sizes are those of the package's own workloads (3 x 100 x 100 and 10 x 1000 x 1000 steady, 5 x 500 x 500 Newton,
realisations of 2-8 layers and 64-512 rows, 16 x 256 x 256 training fields), with ragged ones between them.
``exact`` is plain torch in 64 bits: the seven-point system assembled on the grid and solved by Jacobi-preconditioned
CG (BiCGSTAB inside a Newton iteration for the unconfined model), and the network as 27 shifted products.
"""
import ctypes
import math

import numpy as np
import torch

from modflow6_amd import _lib, configs, learned
from modflow6_amd.ensemble import Ensemble, fixed_system
from modflow6_amd.ims import HipLinearSolver, ImsLinearSettings, dis_structure
from modflow6_amd.solution import GwfSolution

PRECISION = {"fp64": _lib.MF6HIP_FP64, "mixed": _lib.MF6HIP_MIXED, "mixed16": _lib.MF6HIP_MIXED_FP16}
F64 = torch.float64


def listed():
    four, six = "16-32-64-64", "16-32-64-64-64-64"
    return [
        # the smallest workload: a few dozen microseconds an iteration, every launch counts
        dict(name="steady_small", kind="steady", nlay=3, nrow=100, ncol=100, corr=0, sigma=1.0, precision="fp64",
             pre=0, budget=True),
        # an ordinary model with the stock solver (CG + ILU0 in FP64)
        dict(name="steady_ilu0", kind="steady", nlay=10, nrow=300, ncol=300, corr=20, sigma=1.0, precision="fp64",
             pre=0, budget=False),
        # odd extents: no aligned groups of columns; deflated preconditioner in FP64
        dict(name="steady_odd_deflated", kind="steady", nlay=7, nrow=251, ncol=333, corr=20, sigma=2.0,
             precision="fp64", pre=3, budget=False),
        # the headline model with the fastest solver
        dict(name="steady_10m", kind="steady", nlay=10, nrow=1000, ncol=1000, corr=20, sigma=2.0,
             precision="mixed16", pre=3, budget=False),
        # one time step of the transient Newton workload in the reference's precision
        dict(name="newton", kind="newton", nlay=5, nrow=500, ncol=500, steps=1, precision="fp64"),
        # two steps of a smaller one with odd extents in mixed precision
        dict(name="newton_odd_mixed", kind="newton", nlay=4, nrow=187, ncol=251, steps=2, precision="mixed"),
        # one linear solve for a host that formulates by itself
        dict(name="dropin_cg", kind="dropin", nlay=4, nrow=117, ncol=143, corr=8, sigma=1.0),
        # the learned preconditioner in the flexible CG
        dict(name="learned_cg", kind="learned", nlay=6, nrow=96, ncol=112, corr=12, sigma=1.0, channels=four),
        # a small ensemble of uneven realisations, two-level preconditioner
        dict(name="ensemble", kind="ensemble", count=8, nmin=64, nmax=320),
        # the network on a field of its workload's size
        dict(name="net_forward", kind="forward", nlay=16, nrow=256, ncol=256, channels=four),
        # one gradient of a small ragged field
        dict(name="net_grad_ragged", kind="grad", nlay=5, nrow=61, ncol=75, channels=six),
        # training on fields of the workload's size: two Adam steps of two samples
        dict(name="net_train", kind="train", nlay=16, nrow=256, ncol=256, channels=four, samples=4, steps=2, batch=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steady", "steady", "steady", "newton", "newton", "dropin", "learned", "ensemble", "forward",
                       "grad", "train"])
    if kind == "steady":
        pre = rng.choice([0, 0, 2, 3, 3])
        # the one-level solve needs about as many iterations as the grid is wide times its spread: it stays smaller
        n = _log(rng, 64, 700 if pre else 350)
        return dict(kind=kind, nlay=rng.randint(1, 12), nrow=n, ncol=max(48, int(n * rng.uniform(0.6, 1.4))),
                    corr=rng.choice([0, 8, 20]), sigma=rng.choice([1.0, 1.5] if not pre else [1.0, 1.5, 2.0]),
                    precision=rng.choice(["fp64", "mixed", "mixed16"]) if pre else "fp64", pre=pre,
                    budget=n <= 200 and rng.random() < 0.5)
    if kind == "newton":
        n = _log(rng, 60, 500)
        return dict(kind=kind, nlay=rng.randint(2, 6), nrow=n, ncol=max(48, int(n * rng.uniform(0.7, 1.3))),
                    steps=rng.randint(1, 2), precision=rng.choice(["fp64", "fp64", "mixed", "mixed16"]))
    if kind == "dropin":
        return dict(kind=kind, nlay=rng.randint(1, 8), nrow=_log(rng, 48, 240), ncol=_log(rng, 48, 240),
                    corr=rng.choice([0, 8]), sigma=1.0)
    if kind == "learned":
        return dict(kind=kind, nlay=rng.randint(2, 10), nrow=rng.randint(48, 140), ncol=rng.randint(48, 140), corr=12,
                    sigma=1.0, channels="16-32-64-64")
    if kind == "ensemble":
        return dict(kind=kind, count=rng.randint(3, 8), nmin=rng.randint(48, 96), nmax=rng.randint(160, 320))
    shape = dict(nlay=rng.randint(3, 16), nrow=_log(rng, 48, 256), ncol=_log(rng, 48, 256))
    if kind == "train":
        return dict(kind=kind, **shape, channels=rng.choice(["16-32-64-64", "16-16-32-32"]), samples=4, steps=2,
                    batch=rng.randint(1, 2))
    return dict(kind=kind, **shape, channels=rng.choice(["16-32-64-64", "16-32-64-64-64-64", "16-16-32-48"]))


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------

def _gaussian(shape, corr, seed):
    """Standard Gaussian field with covariance exp(-r / corr) (independent cells for corr 0), drawn on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if not corr:
        return torch.randn(shape, generator=g, device="cuda")
    ext = [n + 3 * corr + (n + corr) % 2 for n in shape]
    r2 = torch.zeros(ext, device="cuda")
    for d, e in enumerate(ext):
        a = torch.arange(e, device="cuda")
        r2 += torch.minimum(a, e - a).float().square().reshape([-1 if q == d else 1 for q in range(3)])
    amp = torch.fft.rfftn(torch.exp(-r2.sqrt() / corr)).real.clamp_min(0).sqrt()
    del r2
    f = torch.fft.irfftn(torch.fft.rfftn(torch.randn(ext, generator=g, device="cuda")) * amp, s=ext, dim=(0, 1, 2))
    f = f[: shape[0], : shape[1], : shape[2]]
    return (f - f.mean()) / f.std()


def _steady(c, seed):
    """The steady confined workload (CHD on both sides, recharge, wells) with the case's conductivity field."""
    shape = (c["nlay"], c["nrow"], c["ncol"])
    k = torch.exp(math.log(10.0) + c["sigma"] * _gaussian(shape, c["corr"], seed).double())
    nwel = max(4, c["nlay"] * c["nrow"] * c["ncol"] // 5000)
    return configs.steady_10m(seed=seed, nlay=shape[0], nrow=shape[1], ncol=shape[2], nwel=nwel,
                              k11=k.reshape(-1).cpu().numpy())


def _newton(c, seed):
    return configs.transient_newton(seed=seed, nlay=c["nlay"], nrow=c["nrow"], ncol=c["ncol"],
                                    nwel=max(4, c["nrow"] * c["ncol"] // 500), nper=1, nstp=5)


def _realisations(c, seed):
    shapes, rng = np.random.default_rng([c["count"], c["nmin"], c["nmax"]]), np.random.default_rng(seed)
    out = []
    for q in range(c["count"]):
        n, nlay = (int(v) for v in shapes.integers([c["nmin"], 2], [c["nmax"] + 1, 9]))
        d = dict(nlay=nlay, nrow=n, ncol=n, corr=0, sigma=float(rng.uniform(1.0, 2.0)))
        out.append(_steady(d, seed + 1000 * (q + 1)))
    return out


def _channels(c):
    return tuple(int(v) for v in c["channels"].split("-"))


def _params(c, seed):
    p = learned.init_params(3, _channels(c), np.random.default_rng(seed))
    return p + 0.01 * np.random.default_rng(seed + 1).standard_normal(p.size).astype(np.float32) * (p == 0)


def _planes(c, seed):
    """Network inputs and target of one field: scaled residual, standardised ln K and ln(K33 / K), scaled error."""
    shape = (c["nlay"], c["nrow"], c["ncol"])
    f = [_gaussian(shape, corr, seed + q) for q, corr in enumerate((2, 12, 8, 16))]
    return torch.stack(f).reshape(4, -1).float().cpu().numpy()


class _Kept:
    """A library handle that is given back with the state that holds it."""

    def __init__(self, what):
        self.what = what

    def __del__(self):
        self.what.destroy()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("steady", "newton"):
        model = _steady(c, seed) if kind == "steady" else _newton(c, seed)
        s = dict(kind=kind, steps=c.get("steps", 1), budget=c.get("budget", False), steady=kind == "steady",
                 delt=model.periods[0][0] / model.periods[0][1])
        s["gs"] = GwfSolution(model, precision=PRECISION[c["precision"]], preconditioner=c.get("pre", 0))
        s["x0"] = torch.from_numpy(model.strt).cuda()
        s["x"] = torch.empty_like(s["x0"])
        return s
    if kind in ("dropin", "learned"):
        model = _steady(c, seed)
        net = learned.UNet(c["nlay"], c["nrow"], c["ncol"], channels=_channels(c), params=_params(c, seed)) \
            if kind == "learned" else None
        set_ = ImsLinearSettings(dvclose=1e-6, rclose=1e-6, iter1=5000, preconditioner=1 if net else 0)
        amat, rhs, x0 = fixed_system(model)
        sv = HipLinearSolver().initialize(*dis_structure(c["nlay"], c["nrow"], c["ncol"]), set_, c["nlay"], c["nrow"],
                                          c["ncol"])
        if net:
            sv.attach_unet(net, learned.features(model), 8, 1)
        return dict(kind=kind, sv=sv, net=_Kept(net) if net else None, amat=amat, rhs=rhs, x0=x0)
    if kind == "ensemble":
        return dict(kind=kind, ens=_Kept(Ensemble(_realisations(c, seed), preconditioner=2)))
    net = learned.UNet(c["nlay"], c["nrow"], c["ncol"], channels=_channels(c), params=_params(c, seed))
    s = dict(kind=kind, net=_Kept(net))
    if kind == "train":
        s.update(params=_params(c, seed), steps=c["steps"], batch=c["batch"])
        net.set_data(np.stack([_planes(c, seed + 10 * q) for q in range(c["samples"])]))
    else:
        p = _planes(c, seed)
        s.update(x=p[:3], t=p[3])
    return s


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------

def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    s, kind = state, state["kind"]
    if kind in ("steady", "newton"):
        gs = s["gs"]
        gs.kstp, gs.log = 0, []
        _lib.check(gs.L.mf6hip_gwf_set_x_device(gs.h, _ptr(s["x0"])), "mf6hip_gwf_set_x_device")
        recs = []
        for _ in range(s["steps"]):
            recs = gs.run_timestep(s["delt"], s["steady"])
        if s["budget"]:
            b = gs.budget()
            return dict(heads=gs.heads(), flowja=b["flowja"], terms=np.array([b["terms"][k] for k in sorted(b["terms"])]),
                        converged=int(recs[-1].converged))
        _lib.check(gs.L.mf6hip_gwf_get_x_device(gs.h, _ptr(s["x"])), "mf6hip_gwf_get_x_device")
        return dict(heads=s["x"], converged=int(recs[-1].converged))
    if kind in ("dropin", "learned"):
        x = s["x0"].copy()
        ok, _ = s["sv"].solve(1, s["amat"], s["rhs"], x)
        return dict(heads=x, converged=int(ok))
    if kind == "ensemble":
        ens = s["ens"].what
        ok, _, _ = ens.solve()
        return dict(heads=[ens.heads(i) for i in range(len(ens.cases))], converged=ok)
    net = s["net"].what
    if kind == "forward":
        return net.forward(s["x"])
    if kind == "grad":
        loss, g = net.grad(s["x"], s["t"])
        return dict(loss=loss, grad=g)
    net.set_params(s["params"])
    loss = net.train(s["steps"], s["batch"], 1e-3)
    return dict(loss=loss, params=net.get_params())


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------

def _net_flops(c):
    """Multiply-adds of the 3x3x3 convolutions and the output layer, times two."""
    ch, total = _channels(c), 0.0
    h, w, vox = c["nrow"], c["ncol"], []
    for _ in ch:
        vox.append(c["nlay"] * h * w)
        h, w = (h + 1) // 2, (w + 1) // 2
    for q, (a, b) in enumerate(learned.layer_shapes(3, ch)):
        level = q // 2 if q < 2 * len(ch) else len(ch) - 2 - (q - 2 * len(ch))
        total += 2.0 * 27 * a * b * vox[level]
    return total + 2.0 * ch[0] * vox[0]


def work(case):
    c, kind = case, case["kind"]
    if kind == "ensemble":
        n = c["count"] * 5 * ((c["nmin"] + c["nmax"]) / 2) ** 2
        return dict(bytes=8.0 * (7 + 3) * n, flops=14.0 * n)      # systems in, heads out; one product with the matrix
    n = c["nlay"] * c["nrow"] * c["ncol"]
    if kind == "steady":
        # K, K33, top, bottom, cell type, start heads in; heads (and flows) out
        return dict(bytes=(52.0 + (56.0 if c["budget"] else 0.0)) * n, flops=14.0 * n)
    if kind == "newton":
        return dict(bytes=(52.0 + 28.0) * n * c["steps"], flops=28.0 * n * c["steps"])
    if kind == "dropin":
        return dict(bytes=8.0 * (7 + 3) * n, flops=14.0 * n)
    if kind == "learned":
        return dict(bytes=8.0 * (7 + 3) * n, flops=14.0 * n + 10 * _net_flops(c))   # at least ten applications
    p = 4.0 * learned.init_params(3, _channels(c), np.random.default_rng(0)).size
    if kind == "forward":
        return dict(bytes=16.0 * n + p, flops=_net_flops(c))
    if kind == "grad":
        return dict(bytes=16.0 * n + 2 * p, flops=3 * _net_flops(c))
    k = c["steps"] * c["batch"]
    return dict(bytes=8.0 * n * k + 4 * p, flops=3 * k * _net_flops(c))


def tolerance(case):
    kind = case["kind"]
    if kind in ("steady", "newton", "dropin", "learned", "ensemble"):
        # two converged solves: INNER_DVCLOSE 1e-6 m (OUTER_DVCLOSE 1e-5 m on tens of metres) on heads of metres; each
        # is within 1e-8 of the exact heads
        return dict(rel=1e-7, max=4e-6)
    # BF16 activations and gradients and ReLU masks that flip: about four times what the convolutions' taps summed in
    # the other direction change (0.004 / 0.024, 0.011 / 0.37 and 0.002 / 0.11)
    if kind == "forward":
        return dict(rel=0.016, max=0.1)
    if kind == "grad":
        return dict(rel=0.03, max=0.99)
    return dict(rel=0.008, max=0.5)


# ---------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------------

def _grid(model):
    """Arrays of a model on (nlay, nrow, ncol), 64-bit, on the GPU."""
    shape = (model.nlay, model.nrow, model.ncol)
    top, bot = model.cell_top_bot()
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device="cuda").reshape(shape)  # noqa: E731
    g = dict(top=t(top), bot=t(bot), k=t(model.k11), k33=t(model.k33), h0=t(model.strt))
    g["dx"], g["dy"] = float(model.delr[0]), float(model.delc[0])
    g["fixed"] = torch.zeros(shape, dtype=torch.bool, device="cuda")
    g["q"] = torch.zeros(shape, dtype=F64, device="cuda")
    for p in model.packages:
        n = torch.as_tensor(np.asarray(p.nodes), device="cuda")
        v = torch.as_tensor(np.asarray(p.v1, dtype=np.float64), device="cuda")
        if p.kind == "CHD":
            g["fixed"].view(-1)[n] = True
            g["h0"].view(-1)[n] = v
        elif p.kind in ("WEL", "RCH"):
            a = v if p.kind == "WEL" else v * g["dx"] * g["dy"]
            g["q"].view(-1).index_add_(0, n, a)
            g[p.kind] = (n, a)
        else:
            g["drain"] = (n, v, torch.as_tensor(np.asarray(p.v2, dtype=np.float64), device="cuda"))
    # saturated conductances of the faces to the right, front and down
    thick = g["top"] - g["bot"]
    kt = g["k"] * thick
    hm = lambda a, b, width, d: width * a * b / ((a + b) * d / 2)   # noqa: E731
    g["c"] = [hm(kt[:, :, :-1], kt[:, :, 1:], g["dy"], g["dx"]), hm(kt[:, :-1], kt[:, 1:], g["dx"], g["dy"]),
              g["dx"] * g["dy"] / (0.5 * thick[:-1] / g["k33"][:-1] + 0.5 * thick[1:] / g["k33"][1:])]
    return g


_LO = [(slice(None), slice(None), slice(None, -1)), (slice(None), slice(None, -1)), (slice(None, -1),)]
_HI = [(slice(None), slice(None), slice(1, None)), (slice(None), slice(1, None)), (slice(1, None),)]


def _solve(apply, diag, b, x, symmetric=True, tol=1e-14, most=30000):
    """CG (or BiCGSTAB) with the diagonal as preconditioner, to tol of the start residual."""
    dot = lambda u, v: (u * v).sum()   # noqa: E731
    r = b - apply(x)
    stop = float(r.abs().max()) * tol
    if symmetric:
        z = r / diag
        p, rz = z.clone(), dot(r, z)
        for it in range(most):
            q = apply(p)
            a = rz / dot(p, q)
            x = x + a * p
            r = r - a * q
            if it % 50 == 0 and float(r.abs().max()) <= stop:
                break
            z = r / diag
            new = dot(r, z)
            p, rz = z + (new / rz) * p, new
        return x
    sh, p, rho = r.clone(), r.clone(), dot(r, r)
    for it in range(most):
        ph = p / diag
        v = apply(ph)
        a = rho / dot(sh, v)
        s = r - a * v
        shat = s / diag
        t = apply(shat)
        w = dot(t, s) / dot(t, t)
        x = x + a * ph + w * shat
        r = s - w * t
        if float(r.abs().max()) <= stop:
            break
        new = dot(sh, r)
        p, rho = r + (new / rho) * (a / w) * (p - w * v), new
    return x


def _exact_steady(model):
    g = _grid(model)
    fix, c = g["fixed"], g["c"]
    diag = torch.zeros_like(g["h0"])
    for q in range(3):
        diag[_LO[q]] += c[q]
        diag[_HI[q]] += c[q]

    def flows(h):                           # into the cells
        out = torch.zeros_like(h)
        for q in range(3):
            f = c[q] * (h[_HI[q]] - h[_LO[q]])
            out[_LO[q]] += f
            out[_HI[q]] -= f
        return out

    free = (~fix).double()
    base = torch.where(fix, g["h0"], torch.zeros_like(g["h0"]))
    rhs = free * (g["q"] + flows(base))
    h = _solve(lambda p: -free * flows(free * p), torch.where(fix, torch.ones_like(diag), diag), rhs,
               torch.zeros_like(base))
    return g, base + free * h


def _exact_budget(g, h):
    """Flows in the CSR order of the grid (diagonal the residual, here zero) and (in, out) of each term by name."""
    c, fix = g["c"], g["fixed"]
    planes, have = torch.zeros((7,) + h.shape, dtype=F64, device="cuda"), torch.zeros((7,) + h.shape, dtype=torch.bool,
                                                                                     device="cuda")
    have[0] = True
    for q, (lo, hi) in enumerate(((4, 3), (5, 2), (6, 1))):
        f = c[q] * (h[_HI[q]] - h[_LO[q]])
        planes[lo][_LO[q]], planes[hi][_HI[q]] = f, -f
        have[lo][_LO[q]], have[hi][_HI[q]] = True, True
    at = have.movedim(0, -1)
    flowja = planes.movedim(0, -1)[at]
    # a fixed cell's rate: what its free neighbours take from it (in) and give to it (out)
    nb = torch.zeros_like(have)
    for q, (lo, hi) in enumerate(((4, 3), (5, 2), (6, 1))):
        nb[lo][_LO[q]], nb[hi][_HI[q]] = ~fix[_HI[q]], ~fix[_LO[q]]
    qf = torch.where(nb & fix, planes, torch.zeros_like(planes))
    terms = dict(CHD=(-qf.clamp_max(0).sum(), qf.clamp_min(0).sum()))
    for k in ("WEL", "RCH"):
        n, a = g[k]
        a = a * (~fix.view(-1)[n])
        terms[k] = (a.clamp_min(0).sum(), -a.clamp_max(0).sum())
    zero = torch.zeros((), dtype=F64, device="cuda")
    names = ("STO-SS", "STO-SY", "WEL", "DRN", "RCH", "CHD")
    return flowja, torch.stack([torch.stack(terms.get(k, (zero, zero))) for k in sorted(names)])


def _sat(top, bot, x, eps=1e-6):
    """Quadratically smoothed saturation and its derivative."""
    b = top - bot
    br = ((x - bot) / b).clamp(0.0, 1.0)
    av = 1.0 / (1.0 - eps)
    mid = av * br + 0.5 * (1.0 - av)
    y = torch.where(br < eps, av * 0.5 * br * br / eps,
                    torch.where(br < 1.0 - eps, mid, torch.where(br < 1.0, 1.0 - av * 0.5 * (1 - br) ** 2 / eps, 1.0)))
    d = torch.where(br < eps, av * br / eps,
                    torch.where(br < 1.0 - eps, torch.full_like(br, av), av * (1 - br) / eps))
    return y, d / b


def _exact_newton(model, steps, delt):
    g = _grid(model)
    c, top, bot, area = g["c"], g["top"], g["bot"], g["dx"] * g["dy"]
    shape = top.shape
    ss = torch.as_tensor(model.ss, dtype=F64, device="cuda").reshape(shape) * (top - bot) * area / delt
    sy = torch.as_tensor(model.sy, dtype=F64, device="cuda").reshape(shape) * area / delt
    dn, de, dc = g["drain"]
    thick = top - bot
    h = g["h0"].clone()
    for _ in range(steps):
        old = h.clone()
        so = _sat(top, bot, old)[0]
        for _ in range(60):
            s, d = _sat(top, bot, h)
            # net inflow of every cell (zero at the solution) and its derivative: own and neighbours'
            f, own = g["q"].clone(), torch.zeros_like(h)
            links = []
            for q in range(3):
                a, b = h[_LO[q]], h[_HI[q]]
                if q < 2:
                    up = a > b
                    cond = c[q] * torch.where(up, s[_LO[q]], s[_HI[q]])
                    der = c[q] * torch.where(up, d[_LO[q]], d[_HI[q]]) * (b - a)
                    da, db = -cond + torch.where(up, der, 0.0), cond + torch.where(up, 0.0, der)
                else:
                    cond = c[q]
                    da, db = -cond, cond
                fl = cond * (b - a)
                f[_LO[q]] += fl
                f[_HI[q]] -= fl
                own[_LO[q]] += da
                own[_HI[q]] -= db
                links.append((db, -da))      # d f(lo) / d h(hi), d f(hi) / d h(lo)
            zo, zn = bot + 0.5 * thick * so, bot + 0.5 * thick * s
            f += ss * so * (old - zo) - ss * s * (h - zn) + sy * thick * (so - s)
            own += -ss * (d * (h - zn) + s * (1 - 0.5 * thick * d)) - sy * thick * d
            wet = (h.view(-1)[dn] > de).double() * dc
            f.view(-1).index_add_(0, dn, wet * (de - h.view(-1)[dn]))
            own.view(-1).index_add_(0, dn, -wet)

            def apply(p):
                r = own * p
                for q, (lo, hi) in enumerate(links):
                    r[_LO[q]] += lo * p[_HI[q]]
                    r[_HI[q]] += hi * p[_LO[q]]
                return r

            dh = _solve(apply, own, -f, torch.zeros_like(h), symmetric=False, tol=1e-10, most=2000)
            h = h + dh
            if float(dh.abs().max()) < 1e-10:
                break
    return h


def _net64(c, params, x):
    """The network on one field (3, cells), 64-bit; params a flat 64-bit tensor."""
    ch = _channels(c)
    shapes, at, layers = learned.layer_shapes(3, ch), 0, []
    for a, b in shapes:
        layers.append((params[at:at + 27 * a * b].reshape(27, a, b), params[at + 27 * a * b:at + 27 * a * b + b]))
        at += 27 * a * b + b
    pad = torch.nn.functional.pad

    def conv(v, layer):
        w, b = layer
        d, hh, ww, _ = v.shape
        p = pad(v, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b
        for t in range(27):
            z = p[t // 9:t // 9 + d, t // 3 % 3:t // 3 % 3 + hh, t % 3:t % 3 + ww]
            y = y + z.reshape(-1, v.shape[3]) @ w[t]
        return torch.relu(y).reshape(d, hh, ww, -1)

    def pool(v):
        return torch.nn.functional.avg_pool2d(v.permute(0, 3, 1, 2), 2, ceil_mode=True).permute(0, 2, 3, 1)

    v, skips = x.reshape(3, c["nlay"], c["nrow"], c["ncol"]).permute(1, 2, 3, 0), []
    for q in range(len(ch)):
        v = conv(conv(pool(v) if q else v, layers[2 * q]), layers[2 * q + 1])
        skips.append(v)
    for q in range(len(ch) - 2, -1, -1):
        s = skips[q]
        up = v.repeat_interleave(2, 1).repeat_interleave(2, 2)[:, :s.shape[1], :s.shape[2]]
        v = conv(torch.cat([up, s], 3), layers[2 * len(ch) + len(ch) - 2 - q])
    return (v.reshape(-1, ch[0]) @ params[at:at + ch[0]]) + params[at + ch[0]]


def _loss64(c, params, planes):
    y = _net64(c, params, planes[:3])
    return ((y - planes[3]) ** 2).sum() / (planes[3] ** 2).sum()


def _f64(a):
    return torch.as_tensor(a, device="cuda").double()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("steady", "dropin", "learned"):
        if c["nlay"] * c["nrow"] * c["ncol"] > 1_500_000:
            return None                                            # minutes of unpreconditioned iterations
        g, h = _exact_steady(_steady(c, seed))
        out = dict(heads=h.reshape(-1))
        if c.get("budget"):
            out["flowja"], out["terms"] = _exact_budget(g, h)
        return out
    if kind == "newton":
        m = _newton(c, seed)
        return dict(heads=_exact_newton(m, c["steps"], m.periods[0][0] / m.periods[0][1]).reshape(-1))
    if kind == "ensemble":
        return dict(heads=[_exact_steady(m)[1].reshape(-1) for m in _realisations(c, seed)])
    if kind == "forward":
        with torch.no_grad():
            return _net64(c, _f64(_params(c, seed)), _f64(_planes(c, seed)[:3]))
    p = _f64(_params(c, seed)).requires_grad_(True)
    if kind == "grad":
        loss = _loss64(c, p, _f64(_planes(c, seed)))
        return dict(loss=loss.detach(), grad=torch.autograd.grad(loss, p)[0])
    # Adam on the samples in the order that train() takes (a permutation of them drawn from seed 0)
    rng = np.random.default_rng(0)
    n, k = c["samples"], c["steps"] * c["batch"]
    order = np.concatenate([rng.permutation(n) for _ in range(k // n + 1)])[:k]
    data = [_f64(_planes(c, seed + 10 * q)) for q in range(n)]
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for s in range(c["steps"]):
        total, grad = 0.0, 0.0
        for q in order[s * c["batch"]:(s + 1) * c["batch"]]:
            loss = _loss64(c, p, data[q])
            grad = grad + torch.autograd.grad(loss, p)[0] / c["batch"]
            total = total + loss.detach() / c["batch"]
        losses.append(total)
        m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
        step = 1e-3 * (m / (1 - 0.9 ** (s + 1))) / ((v / (1 - 0.999 ** (s + 1))).sqrt() + 1e-8)
        p = (p.detach() - step.detach()).requires_grad_(True)
    return dict(loss=torch.stack(losses), params=p.detach())
