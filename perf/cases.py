"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values.  `listed()` gives the standing list,
`draw(rng)` one more case of the same ranges, `prepare(case, seed)` what a
program holds before the call (inputs on the GPU, the Operator or Batch, the
work buffers), `run(state)` one pass through the public entry points,
`work(case)` the bytes and operations such a pass cannot do without, and
`exact(case, seed)` the result in 64 bits from plain torch, written from the
operators' definitions (dense compact-scheme matrices, autograd for the
adjoint).

Grids are (nx, ny, nz) points on the unit cube, uniform or stretched by tanh
(beta = 2) towards the walls; fields are float64 with shape (nz, ny, nx).
Velocities are sums of solenoidal Fourier modes with a k^(-5/3) spectrum plus
a swirl confined to mid-height, the flow of a stirred tank.
"""
import math

import numpy as np
import torch

from emix3d_amd import Batch, Operator
from emix3d_amd.api import adam_f32, mlp_backward_f32, mlp_forward_f32
from emix3d_amd.closure import WEIGHTS, LearnedClosure

MACH = 0.1
C4 = 1.0 / 1000.0  # 1/Re
DT = 1.0e-3
CFILT = 0.49
MODES = 48
F64 = torch.float64


def _grid(name, kind, nx, ny, nz, scheme, stretch, **more):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, scheme=scheme, stretch=stretch, **more)


def listed():
    return [
        # a coarse uniform box of the multiphase solver: velocity gradient and
        # divergence, 64 points a side, where launches and latency count
        _grid("grad_div_64", "grad_div", 64, 64, 64, "c6f", False),
        # the spatial operator of one Runge-Kutta stage on a debugging grid
        _grid("stage_coarse", "stage", 64, 56, 48, "c6c", True),
        # the same on a tank mesh whose sides are no multiple of anything,
        # with the fourth-order scheme
        _grid("stage_ragged", "stage", 187, 151, 129, "c4", True),
        # the production mesh: the stage that bench.py reports
        _grid("stage_256", "stage", 256, 256, 256, "c6f", True),
        # a whole Runge-Kutta sub-step around an immersed solid: operator,
        # update, boundary values, clip, pressure extrapolation, rebuild
        _grid("substep_tank", "substep", 208, 176, 160, "c6f", True),
        # the compact filter that runs every few time steps
        _grid("filter_tank", "filter", 192, 192, 160, "c6f", True),
        # level-set reinitialisation (ten iterations) of a two-phase run
        _grid("reinit_two_phase", "reinit", 208, 176, 160, "c6c", True),
        # the gradient of a loss through the flux divergence and the velocity
        # gradient: the backward direction of the stage
        _grid("adjoint_128", "adjoint", 128, 128, 128, "c6c", True),
        # 48 uneven boxes advanced together: gradient, divergence and one
        # WENO5 / SSP-RK3 level-set step each
        dict(name="batch_48", kind="batch", boxes=48, hx=192, hy=128, hz=96, dims_seed=20261205,
             scheme="c6c"),
        # eddy viscosity by the dynamic model, the target of the closure
        _grid("dynsmag_tank", "dynsmag", 224, 192, 160, "c6c", True),
        # eddy viscosity by the trained network (BF16 matrix cores)
        _grid("learned_tank", "learned", 224, 192, 160, "c6c", True),
        # one training step of the network: features, forward, backward, Adam
        _grid("closure_train", "train", 96, 96, 96, "c6c", True, rows=65536),
    ]


# most points a drawn grid may have, by kind: none costs more than the
# largest listed case
_CAP = {"grad_div": 1 << 24, "stage": 1 << 24, "substep": 1 << 23, "filter": 1 << 24,
        "reinit": 5_500_000, "adjoint": 1 << 23, "dynsmag": 1 << 24, "learned": 1 << 24}


def draw(rng):
    kind = rng.choice(["grad_div", "stage", "stage", "substep", "filter", "reinit", "adjoint",
                       "batch", "dynsmag", "learned", "train"])
    scheme = rng.choice(["c4", "c6f", "c6c"])
    if kind == "batch":
        return dict(kind=kind, boxes=int(round(math.exp(rng.uniform(math.log(3), math.log(48))))),
                    hx=rng.randint(48, 192), hy=rng.randint(48, 128), hz=rng.randint(40, 96),
                    dims_seed=rng.randint(1, 10 ** 6), scheme=scheme)
    if kind == "train":
        n = rng.randint(32, 96)
        return dict(kind=kind, nx=n, ny=n, nz=n, scheme=scheme, stretch=True,
                    rows=int(round(math.exp(rng.uniform(math.log(1000), math.log(131072))))))
    while True:
        total = math.exp(rng.uniform(math.log(40_000), math.log(_CAP[kind])))
        side = total ** (1.0 / 3.0)
        n = [int(round(side * math.exp(rng.uniform(-0.5, 0.5)))) for _ in range(3)]
        if min(n) >= 20 and max(n) <= 512 and n[0] * n[1] * n[2] <= _CAP[kind]:
            return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], scheme=scheme,
                        stretch=rng.random() < 0.7)


# --------------------------------------------------------------------- inputs

def _axis(n, stretch):
    s = torch.linspace(0.0, 1.0, n, dtype=F64)
    return 0.5 * (1.0 + torch.tanh(2.0 * (2.0 * s - 1.0)) / math.tanh(2.0)) if stretch else s


def _points(axes, dev):
    """The three coordinate fields of the tensor grid of the three axes."""
    x1, y1, z1 = (a.to(dev) for a in axes)
    x = torch.empty((3, z1.numel(), y1.numel(), x1.numel()), dtype=F64, device=dev)
    x[0] = x1.view(1, 1, -1)
    x[1] = y1.view(1, -1, 1)
    x[2] = z1.view(-1, 1, 1)
    return x


def _modes(axes, gen, dev, comps, kmax, modes=MODES):
    """comps fields, each a sum of plane waves with wave numbers 1..kmax; three
    components are solenoidal.  Evaluated as products of the axes' waves."""
    k = torch.exp(torch.rand(modes, generator=gen, dtype=F64) * math.log(kmax))
    d = torch.randn((modes, 3), generator=gen, dtype=F64)
    d = d / d.norm(dim=1, keepdim=True)
    if comps == 3:
        s = torch.linalg.cross(d, torch.randn((modes, 3), generator=gen, dtype=F64))
        s = s / s.norm(dim=1, keepdim=True)
    else:
        s = torch.ones((modes, comps), dtype=F64)
    amp = k ** (-1.0 / 3.0)  # k^(-5/3) energy, sampled evenly in log k
    amp = amp / (amp.square().sum() / 2.0).sqrt()
    ph = torch.rand(modes, generator=gen, dtype=F64) * (2.0 * math.pi)
    wave = [torch.exp(1j * (2.0 * math.pi * k * d[:, a])[:, None] * axes[a][None, :]) for a in range(3)]
    wave[0] = wave[0] * torch.exp(1j * ph)[:, None]
    wx, wy, wz = (w.to(dev) for w in wave)
    yz = (wz[:, :, None] * wy[:, None, :]).reshape(modes, -1)
    yr, yi = yz.real.T.contiguous(), yz.imag.T.contiguous()
    out = []
    for c in range(comps):
        a = (amp * s[:, c]).to(dev)[:, None]
        f = yr @ (a * wx.real).contiguous() - yi @ (a * wx.imag).contiguous()
        out.append(f.reshape(axes[2].numel(), axes[1].numel(), axes[0].numel()))
    return torch.stack(out)


def _swirl(axes, dev):
    x, y, z = axes[0].to(dev).view(1, 1, -1), axes[1].to(dev).view(1, -1, 1), axes[2].to(dev).view(-1, 1, 1)
    band = torch.exp(-((z - 0.5) / 0.15) ** 4) * torch.exp(-8.0 * ((x - 0.5) ** 2 + (y - 0.5) ** 2))
    return torch.stack([-4.0 * (y - 0.5) * band, 4.0 * (x - 0.5) * band, torch.zeros_like(band)])


def _ball(axes, gen, dev, radius):
    """Signed distance to a ball (negative inside) whose centre the seed moves."""
    c = 0.4 + 0.2 * torch.rand(3, generator=gen, dtype=F64)
    x, y, z = axes[0].to(dev).view(1, 1, -1), axes[1].to(dev).view(1, -1, 1), axes[2].to(dev).view(-1, 1, 1)
    return torch.sqrt((x - float(c[0])) ** 2 + (y - float(c[1])) ** 2 + (z - float(c[2])) ** 2) - radius


def _inputs(case, seed, dev):
    """The fields of a single-grid case, from the seed alone."""
    gen = torch.Generator().manual_seed(int(seed) * 1000003 + 17)
    kind = case["kind"]
    n = (case["nx"], case["ny"], case["nz"])
    axes = [_axis(m, case["stretch"]) for m in n]
    shape = (n[2], n[1], n[0])
    dgen = torch.Generator(device=dev).manual_seed(int(seed) * 7 + 3)
    f = {"axes": axes, "n": n, "ih": tuple(float(m - 1) for m in n),
         "dxyz": tuple(1.0 / (m - 1) for m in n),
         "dmin": float(min((a[1:] - a[:-1]).min() for a in axes))}
    if kind == "reinit":
        # a distance field distorted as advection leaves it: gradients off one
        d = torch.minimum(_ball(axes, gen, dev, 0.25), axes[2].to(dev).view(-1, 1, 1) - 0.8)
        f["phi"] = (d * (1.0 + 0.6 * d + 0.05 * _modes(axes, gen, dev, 1, 3, 8)[0])).contiguous()
        return f
    kmax = min(16.0, min(n) / 6.0)
    f["u"] = (0.3 * _modes(axes, gen, dev, 3, kmax) + _swirl(axes, dev)).contiguous()
    if kind in ("stage", "substep", "filter", "adjoint"):
        f["temp"] = (1.0 + 0.1 * _modes(axes, gen, dev, 1, 4, 12)[0]).contiguous()
        f["pres"] = (1.0 / MACH ** 2 + _modes(axes, gen, dev, 1, 4, 12)[0]).contiguous()
        f["um"] = torch.empty((5,) + shape, dtype=F64, device=dev)
        f["um"][0] = f["pres"] * MACH * MACH
        f["um"][1:4] = f["u"] * f["um"][0]
        f["um"][4] = f["temp"]
    if kind == "substep":
        # the sub-step starts from a state some way on from the step's start
        f["um0"] = f["um"].clone()
        f["um0"][1:4] *= 0.99
        f["mask"] = (torch.rand(shape, dtype=F64, device=dev, generator=dgen) > 0.02).double()
        f["sobject"] = (-_ball(axes, gen, dev, 0.15)).contiguous()
    if kind == "adjoint":
        f["vis"] = C4 + 1e-3 * torch.rand(shape, dtype=F64, device=dev, generator=dgen)
        f["rs_bar"] = torch.randn((5,) + shape, dtype=F64, device=dev, generator=dgen)
        f["rsv_bar"] = torch.randn((5,) + shape, dtype=F64, device=dev, generator=dgen)
    if kind == "train":
        rows, N = case["rows"], n[0] * n[1] * n[2]
        f["idx"] = torch.randint(0, N, (rows,), device=dev, generator=dgen)
        # Adam's moments as some way into a training run
        f["m"] = 1e-4 * torch.randn(9089, dtype=torch.float32, device=dev, generator=dgen)
        f["v"] = 1e-6 * (0.5 + torch.rand(9089, dtype=torch.float32, device=dev, generator=dgen))
    return f


def _box_dims(case):
    rng = np.random.default_rng(case["dims_seed"])
    hi = (case["hx"], case["hy"], case["hz"])
    dims = [(32, 32, 32), hi]
    while len(dims) < case["boxes"]:
        dims.append(tuple(int(rng.integers(32, h + 1)) for h in hi))
    return dims


def _box_inputs(case, seed, dev):
    """One dict per box: uniform grid, velocity, level set, spacings, CFL 0.5,
    and the box's place in the pools (whole cache lines apart)."""
    out, at = [], 0
    for i, d in enumerate(_box_dims(case)):
        gen = torch.Generator().manual_seed(int(seed) * 1000003 + 101 * i)
        axes = [_axis(m, False) for m in d]
        u = _modes(axes, gen, dev, 3, 5.0, 16).contiguous()
        phi = torch.minimum(_ball(axes, gen, dev, 0.25), axes[2].to(dev).view(-1, 1, 1) - 0.8)
        dxyz = tuple(1.0 / (m - 1) for m in d)
        out.append({"axes": axes, "n": d, "u": u, "phi": phi.contiguous(), "dxyz": dxyz,
                    "ih": tuple(float(m - 1) for m in d), "dt": 0.125 * min(dxyz), "at": at})
        at += (d[0] * d[1] * d[2] + 63) // 64 * 64
    return out


def _pools(boxes, dev):
    """The pools a multi-box program keeps its gradients (9 fields a box),
    divergences and level sets in."""
    nx, ny, nz = boxes[-1]["n"]
    N = boxes[-1]["at"] + (nx * ny * nz + 63) // 64 * 64
    return [torch.zeros(c * N, dtype=F64, device=dev) for c in (9, 1, 1)]


def _box_view(pool, box, comps):
    nx, ny, nz = box["n"]
    return pool[comps * box["at"]:][:comps * nx * ny * nz].view(comps, nz, ny, nx)


# ------------------------------------------------------------ prepare and run

def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    kind = case["kind"]
    if kind == "batch":
        boxes = _box_inputs(case, seed, dev)
        b = Batch([z["n"] for z in boxes], case["scheme"])
        dvel, div, phi = _pools(boxes, dev)
        for i, z in enumerate(boxes):
            jbn = Operator(*z["n"], case["scheme"]).jacobeano(_points(z["axes"], dev))
            p = _box_view(phi, z, 1)[0].copy_(z["phi"])
            b.bind(i, z["u"], jbn, p, _box_view(dvel, z, 9), _box_view(div, z, 1)[0], z["ih"],
                   z["dxyz"], z["dt"])
        b.tune(reps=3)
        return {"kind": kind, "batch": b, "dvel": dvel, "div": div, "phi": phi}
    f = _inputs(case, seed, dev)
    op = Operator(case["nx"], case["ny"], case["nz"], case["scheme"])
    x = _points(f["axes"], dev)
    s = {"kind": kind, "op": op, "jbn": op.jacobeano(x)}
    for k in ("u", "um", "um0", "temp", "pres", "mask", "sobject", "vis", "rs_bar", "rsv_bar"):
        if k in f:
            s[k] = f[k]
    s["dxyz"], s["dmin"] = f["dxyz"], f["dmin"]
    new = lambda *c: torch.empty(tuple(c) + tuple(x.shape[1:]), dtype=F64, device=dev)  # noqa: E731
    if kind == "grad_div":
        s.update(dvel=new(9), div=new())
    elif kind in ("stage", "substep"):
        s["sgd"] = op.inisgdm(x)[0]
        s["work"] = op.stage_buffers()
        if kind == "substep":
            s.update(um1=new(5), start=[f[k].clone() for k in ("u", "temp", "pres")])
    elif kind == "filter":
        s.update(um1=new(5), temp=new(), pres=new())
    elif kind == "reinit":
        s.update(phi=new(), start=f["phi"], dmins=op.inisgdm(x)[1])
    elif kind == "adjoint":
        s["dvel"] = op.deriv_vel(f["u"])[0]
        s["out"] = op.flujos_divergencia_all_adj(f["rs_bar"], f["rsv_bar"], f["um"], f["u"],
                                                 f["vis"], s["jbn"], s["dvel"])
        s["ug"] = new(3)
    elif kind in ("dynsmag", "learned", "train"):
        s["dvel"] = op.deriv_vel(f["u"])[0]
        s["delta"] = op.inisgdm(x)[0][0].contiguous()
        s.update(nut=new(), vis=new())
        if kind != "dynsmag":
            s["closure"] = LearnedClosure.load(device=dev)
        if kind == "train":
            nut = op.dynsmag(f["u"], s["dvel"], s["jbn"], s["delta"])
            s.update(idx=f["idx"], m=f["m"], v=f["v"], steps=100, work=None,
                     target=nut.reshape(-1)[f["idx"]].float(),
                     scale=2.0 / (case["rows"] * float(nut.square().mean())))
    return s


def run(s):
    kind = s["kind"]
    if kind == "batch":
        s["batch"].stage()
        return s["dvel"], s["div"], s["phi"]
    op, jbn = s["op"], s["jbn"]
    if kind == "grad_div":
        return op.grad_div(s["u"], jbn=jbn, dvel=s["dvel"], div=s["div"])
    if kind == "stage":
        return op.rk_stage(s["um"], s["u"], s["temp"], s["pres"], jbn, s["sgd"], C4, work=s["work"])
    if kind == "substep":
        # u, temp and pres are updated in place: the fields of the sub-step before
        for k, v in zip(("u", "temp", "pres"), s["start"]):
            s[k].copy_(v)
        op.rk_substep(2, s["um0"], s["um"], s["u"], s["temp"], s["pres"], jbn, s["sgd"], C4, DT,
                      MACH, s["mask"], sobject=s["sobject"], dxyz=s["dxyz"], deltamin=s["dmin"],
                      work=s["work"], um1=s["um1"])
        return {"um1": s["um1"], "u": s["u"], "temp": s["temp"], "pres": s["pres"], **s["work"]}
    if kind == "filter":
        s["um1"].copy_(s["um"])  # filtered in place: the fields the time step left
        op.filtrado(1, s["um1"], jbn, CFILT, MACH, u=s["u"], pres=s["pres"], temp=s["temp"])
        return s["um1"], s["u"], s["pres"], s["temp"]
    if kind == "reinit":
        s["phi"].copy_(s["start"])  # in place: the level set that advection left
        return op.reinit_level_set(s["phi"], jbn, s["dmins"], s["dxyz"], s["dmin"])
    if kind == "adjoint":
        out = op.flujos_divergencia_all_adj(s["rs_bar"], s["rsv_bar"], s["um"], s["u"], s["vis"],
                                            jbn, s["dvel"], out=s["out"])
        ug, _ = op.deriv_vel_adj(out["dvel_bar"], u_bar=s["ug"])
        return {**out, "u_from_dvel": ug}
    if kind == "dynsmag":
        op.dynsmag(s["u"], s["dvel"], jbn, s["delta"], nut=s["nut"], c4=C4, vis=s["vis"])
        return s["nut"], s["vis"]
    cl = s["closure"]
    if kind == "learned":
        cl.nut(op, s["dvel"], jbn, s["delta"], out=s["nut"], c4=C4, vis=s["vis"])
        return s["nut"], s["vis"]
    feat = op.mlp_gather(s["dvel"], jbn, s["delta"], s["idx"])
    act, nu = mlp_forward_f32(cl.params, cl.norm, feat)
    dnu = s["scale"] * (nu - s["target"])
    grad, s["work"] = mlp_backward_f32(cl.params, cl.norm, feat, act, dnu, s["work"])
    s["steps"] += 1
    adam_f32(cl.params, grad, s["m"], s["v"], s["steps"], lr=1e-4)
    return {"nu": nu, "grad": grad, "params": cl.params, "m": s["m"], "v": s["v"]}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n = sum(a * b * c for a, b, c in _box_dims(case))
        # u, five metrics, phi in; dvel, div, phi out; three WENO5 stages
        return {"bytes": 8.0 * n * 20, "flops": n * (4 * 3 * 18.0 + 3 * 3 * 75.0)}
    n = float(case["nx"] * case["ny"] * case["nz"])
    if kind == "train":
        r = case["rows"]
        return {"bytes": r * (13 * 8.0 + 8 + 8) + 9089 * 4.0 * 8, "flops": r * 3 * 17792.0}
    fields, flops = {
        "grad_div": (18, 4 * 3 * 18.0),      # u, five metrics in; dvel, div out
        "stage": (46, 36 * 18.0 + 250.0),    # 22 in, 24 out
        "substep": (64, 36 * 18.0 + 350.0),  # the stage's, um0, mask, solid; um1 and primitives
        "filter": (17, 15 * 30.0),           # um1, J, 1/J in; um1, u, pres, temp out
        "reinit": (6, 30 * (6 * 70.0 + 40.0)),
        "adjoint": (52, 27 * 25.0 + 150.0),
        "dynsmag": (18, 21 * 13.0 + 150.0),
        "learned": (15, 17792.0),
    }[kind]
    return {"bytes": 8.0 * fields * n, "flops": flops * n}


# ---------------------------------------------------------------- 64-bit truth

def _compact(n, scheme):
    """The dense derivative matrix A^-1 B of a line of n points, unit spacing."""
    A = torch.eye(n, dtype=F64)
    B = torch.zeros((n, n), dtype=F64)
    i = torch.arange(1, n - 1)
    if scheme == "c4":
        A[i, i - 1] = A[i, i + 1] = 0.25
        B[i, i + 1], B[i, i - 1] = 0.75, -0.75
    else:
        B[1, 0], B[1, 2] = -0.75, 0.75
        B[n - 2, n - 3], B[n - 2, n - 1] = -0.75, 0.75
        A[1, 0] = A[1, 2] = A[n - 2, n - 3] = A[n - 2, n - 1] = 0.25
        j = torch.arange(2, n - 2)
        A[j, j - 1] = A[j, j + 1] = 1.0 / 3.0
        B[j, j + 1], B[j, j - 1] = 7.0 / 9.0, -7.0 / 9.0
        B[j, j + 2], B[j, j - 2] = 1.0 / 36.0, -1.0 / 36.0
    if scheme == "c6f":  # third-order closure
        A[0, 1] = A[n - 1, n - 2] = 2.0
        edge = [-2.5, 2.0, 0.5]
    else:                # fourth-order closure
        A[0, 1] = A[n - 1, n - 2] = 3.0
        edge = [-17.0 / 6.0, 1.5, 1.5, -1.0 / 6.0]
    for k, e in enumerate(edge):
        B[0, k], B[n - 1, n - 1 - k] = e, -e
    return torch.linalg.solve(A, B)


def _filter(n, periodic):
    A = torch.eye(n, dtype=F64)
    B = torch.eye(n, dtype=F64)
    c = CFILT
    rows = torch.arange(n) if periodic else torch.arange(5, n - 5)
    up, dn = rows[rows < n - 1], rows[rows > 0]
    A[up, up + 1] = c
    A[dn, dn - 1] = c
    coef = [(193 + 126 * c) / 256, (105 + 302 * c) / 256, (-15 + 30 * c) / 64,
            (45 - 90 * c) / 512, (-5 + 10 * c) / 256, (1 - 2 * c) / 512]
    r = torch.arange(5, n - 5)
    B[r, r] = coef[0]
    for k in range(1, 6):
        B[r, r + k] = B[r, r - k] = 0.5 * coef[k]
    return torch.linalg.solve(A, B)


def _along(M, f, d):
    """M applied along direction d (0: x, the last axis) of f (nz, ny, nx)."""
    if d == 0:
        return f @ M.T.contiguous()
    if d == 1:
        return torch.stack([M @ p for p in f])
    return (M @ f.reshape(f.shape[0], -1)).reshape(f.shape)


def _derivs(n, scheme, dev):
    mats = [(_compact(m, scheme) * (m - 1)).to(dev) for m in n]
    return lambda f, d: _along(mats[d], f, d)


def _metrics(axes, scheme, dev):
    """xi_x, eta_y, zeta_z, J and 1/J of a tensor grid, as broadcastable fields."""
    h = [(_compact(a.numel(), scheme) * (a.numel() - 1)) @ a for a in axes]
    hx, hy, hz = h[0].to(dev).view(1, 1, -1), h[1].to(dev).view(1, -1, 1), h[2].to(dev).view(-1, 1, 1)
    # the inverse-metric tensor's determinant is J; comps 1, 5, 9 invert it
    det = hx * hy * hz
    return [(hy * hz) / det, (hx * hz) / det, (hx * hy) / det], det, 1.0 / det


def _sgd(axes, dev):
    """Filter width, the six cube-root factors and the smallest spacings."""
    p, m = [], []
    for a in axes:
        d = a[1:] - a[:-1]
        p.append(torch.cat([d, d[-1:]]))
        m.append(torch.cat([d[:1], d]))
    view = [(1, 1, -1), (1, -1, 1), (-1, 1, 1)]
    p = [v.to(dev).view(*s) for v, s in zip(p, view)]
    m = [v.to(dev).view(*s) for v, s in zip(m, view)]
    width = 1.0
    for a, b in zip(p, m):
        width = width * torch.maximum(a, b)
    width = width ** (1.0 / 3.0)
    least = torch.minimum(torch.minimum(torch.minimum(p[0], m[0]), torch.minimum(p[1], m[1])),
                          torch.minimum(p[2], m[2]))
    fac = [(width / v) ** (1.0 / 3.0) for a, b in zip(p, m) for v in (a, b)]
    return width, fac, least


def _at(f, d, idx):
    return f.index_select(f.dim() - 1 - d, idx)


def _clamped(f, d, o):
    n = f.shape[f.dim() - 1 - d]
    return _at(f, d, (torch.arange(n, device=f.device) + o).clamp(0, n - 1))


def _gradient(D, u):
    return torch.stack([D(u[c], d) for d in range(3) for c in range(3)])


def _fluxes(um, u, pres, vis, met, dv, d):
    """The five convective and three viscous fluxes along direction d."""
    conv = [-um[1 + d]]
    for a in range(3):
        e = -um[1 + d] * u[a]
        conv.append(e - pres if a == d else e)
    conv.append(-u[d] * um[4])
    visc = []
    for a in range(3):
        if a == d:
            visc.append(vis * 2.0 * met[a] * dv[4 * a])
        else:
            lo, hi = min(a, d), max(a, d)
            # (0,1): m0 dv1 + m1 dv3; (0,2): m0 dv2 + m2 dv6; (1,2): m2 dv7 + m1 dv5
            visc.append(vis * (met[lo] * dv[3 * lo + hi] + met[hi] * dv[3 * hi + lo]))
    return conv, visc


def _flux_div(D, um, u, pres, vis, met, J, iJ, dv):
    acc = [0.0] * 8
    for d in range(3):
        conv, visc = _fluxes(um, u, pres, vis, met, dv, d)
        for k, e in enumerate(conv + visc):
            acc[k] = acc[k] + D(J * met[d] * e, d)
    rs = torch.stack([iJ * acc[k] for k in range(5)])
    z = torch.zeros_like(rs[0])
    rsv = torch.stack([z, iJ * acc[5], iJ * acc[6], iJ * acc[7], z])
    return rs, rsv


def _structure_viscosity(u, dv, met, width, fac):
    s = 0.0
    for d in range(3):
        n = u.shape[u.dim() - 1 - d]
        i = torch.arange(n, device=u.device)
        hi = torch.where(i < n - 1, i + 1, i)
        lo = torch.where(i > 0, i - 1, i)
        up = _at(u, d, hi) - _at(u, d, hi - 1)
        dn = _at(u, d, lo + 1) - _at(u, d, lo)
        s = s + (up * fac[2 * d]).square().sum(0) + (dn * fac[2 * d + 1]).square().sum(0)
    m = 0.1781 * torch.sqrt(s / 6.0) * width
    w = torch.stack([met[1] * dv[7] - met[2] * dv[5], met[2] * dv[2] - met[0] * dv[6],
                     met[0] * dv[3] - met[1] * dv[1]])
    wn = sum(_clamped(w, d, o) for d in range(3) for o in (1, -1))
    wnn = torch.sqrt(w.square().sum(0) * wn.square().sum(0))
    return torch.where((w * wn).sum(0) / wnn > math.cos(math.pi / 9.0), torch.zeros_like(m), m)


def _stage(f, case, dev):
    D = _derivs(f["n"], case["scheme"], dev)
    met, J, iJ = _metrics(f["axes"], case["scheme"], dev)
    width, fac, _ = _sgd(f["axes"], dev)
    dv = _gradient(D, f["u"])
    dtemp = torch.stack([D(f["temp"], d) for d in range(3)])
    amut = _structure_viscosity(f["u"], dv, met, width, fac)
    vis = C4 + amut
    rs, rsv = _flux_div(D, f["um"], f["u"], f["pres"], vis, met, J, iJ, dv)
    return {"dvel": dv, "dtemp": dtemp, "amut": amut, "vis": vis, "rs": rs, "rsv": rsv}


def _mirror(n, dev):
    """Interior index of each position of a line padded by 5 mirrored points."""
    i = torch.arange(n + 10, device=dev)
    i = torch.where(i < 5, 9 - i, i)
    return torch.where(i >= n + 5, 2 * (n + 5) - 1 - i, i) - 5


def _pad(f):
    for d in range(3):
        f = _at(f, d, _mirror(f.shape[f.dim() - 1 - d], f.device))
    return f


def _inner(f):
    return f[5:-5, 5:-5, 5:-5]


def _weno5(b):
    b1, b2, b3, b4, b5 = b
    s = [13.0 / 12.0 * (b1 - 2 * b2 + b3) ** 2 + 0.25 * (b1 - 4 * b2 + 3 * b3) ** 2,
         13.0 / 12.0 * (b2 - 2 * b3 + b4) ** 2 + 0.25 * (b2 - b4) ** 2,
         13.0 / 12.0 * (b3 - 2 * b4 + b5) ** 2 + 0.25 * (3 * b3 - 4 * b4 + b5) ** 2]
    a = [c / (v + 1e-6) ** 2 for c, v in zip((0.1, 0.6, 0.3), s)]
    p = [(2 * b1 - 7 * b2 + 11 * b3) / 6, (-b2 + 5 * b3 + 2 * b4) / 6, (2 * b3 + 5 * b4 - b5) / 6]
    return (a[0] * p[0] + a[1] * p[1] + a[2] * p[2]) / (a[0] + a[1] + a[2])


def _biased(phi, d, scale):
    """Left- and right-biased WENO5 derivatives of the padded phi along d, with
    the substitutions on the outermost positions; scale: 1/spacing times metric."""
    n = phi.shape[2 - d]
    i = torch.arange(n, device=phi.device)
    diff = _at(phi, d, i.clamp(min=1)) - _at(phi, d, i.clamp(min=1) - 1)  # position 0: as 1
    take = lambda j: scale * _at(diff, d, j.clamp(0, n - 1))  # noqa: E731
    w = torch.where
    left = [i - 2, i - 1, i, i + 1, i + 2]
    left[1] = w(i == 0, 0 * i, left[1])
    left[0] = w(i == 0, 0 * i + 1, w(i == 1, 0 * i, left[0]))
    left[3] = w(i == n - 1, i, left[3])
    left[4] = w(i == n - 1, i - 1, w(i == n - 2, i + 1, left[4]))
    L = [take(j) for j in left]
    if d == 2:
        # the last plane's fifth operand: its own z difference one row down
        below = _clamped(diff[-1:], 1, -1)
        s = scale[-1:] if scale.shape[0] == n else scale
        L[4] = torch.cat([L[4][:-1], s * below])
    right = [i + 3, i + 2, i + 1, i, i - 1]
    right[4] = w(i == 0, 0 * i, right[4])
    right[2] = w(i == n - 1, i, right[2])
    right[1] = w(i == n - 1, i - 1, w(i == n - 2, i + 1, right[1]))
    right[0] = w(i == n - 1, i - 2, w(i == n - 2, i, w(i == n - 3, i + 2, right[0])))
    return _weno5(L), _weno5([take(j) for j in right])


def _ssp3(phi, rhs, dt):
    a = phi - dt * rhs(phi)
    b = 0.75 * phi + 0.25 * (a - dt * rhs(a))
    return (phi + 2.0 * (b - dt * rhs(b))) / 3.0


def _reinit(phi, met, least, dxyz, dmin):
    full = lambda v: _pad(v.expand(phi.shape))  # noqa: E731
    scale = [full(m) / h for m, h in zip(met, dxyz)]
    width = full(least)
    for _ in range(10):
        p0 = _pad(phi)
        so = p0 / torch.sqrt(p0 * p0 + width * width)

        def rhs(p):
            g = 0.0
            for d in range(3):
                L, R = _biased(p, d, scale[d])
                plus = torch.maximum(L.clamp(min=0).square(), R.clamp(max=0).square())
                minus = torch.maximum(R.clamp(min=0).square(), L.clamp(max=0).square())
                t = torch.sign(p0)
                g = g + 0.5 * (t + 1) * plus + 0.5 * (t - 1).abs() * minus
            return so * (torch.sqrt(g) - 1.0)

        phi = _inner(_ssp3(p0, rhs, 0.5 * dmin))
    return phi.contiguous()


def _advect(phi, u, met, dxyz, dt):
    vel = _pad(u)
    scale = [_pad(m.expand(phi.shape)) / h for m, h in zip(met, dxyz)]

    def rhs(p):
        r = 0.0
        for d in range(3):
            L, R = _biased(p, d, scale[d])
            r = r + torch.where(vel[d] > 0, vel[d] * L, vel[d] * R)
        return r

    return _inner(_ssp3(_pad(phi), rhs, dt)).contiguous()


def _extrapolate(pres, sobject, met, dxyz, dmin):
    """Pressure carried into the solid along its normal: ten SSP-RK3 steps at
    the solid's points of the padded grid."""
    P, S = _pad(pres), _pad(sobject)
    m = [_pad(v.expand(pres.shape)).reshape(-1) / h for v, h in zip(met, dxyz)]
    gz, gy, gx = P.shape
    ext, stride = (gx, gy, gz), (1, gx, gx * gy)
    P, S = P.reshape(-1), S.reshape(-1)
    at = torch.nonzero(S > 0).reshape(-1)
    pos = [at % gx, (at // gx) % gy, at // (gx * gy)]
    low = [pos[d] == 0 for d in range(3)]
    high = [pos[d] == ext[d] - 1 for d in range(3)]
    plus = [torch.where(high[d], at, at + stride[d]) for d in range(3)]
    minus = [torch.where(low[d], at, at - stride[d]) for d in range(3)]
    face = low[0] | low[1] | low[2] | high[0] | high[1] | high[2]
    fac = torch.where(face, 1.0, 0.5).to(F64)
    grad = [fac * m[d][at] * (S[plus[d]] - S[minus[d]]) for d in range(3)]
    mid = at
    for d in range(3):
        mid = torch.where(low[d], at + stride[d], mid)
    for d in range(3):
        mid = torch.where(high[d], at - stride[d], mid)

    def rhs(q):
        r = 0.0
        for d in range(3):
            back = m[d][at] * (q[mid] - q[minus[d]])
            fore = m[d][at] * (q[plus[d]] - q[mid])
            s = torch.sign(grad[d])
            r = r + (0.5 * (s + 1) * back + 0.5 * (s - 1).abs() * fore) * grad[d]
        return r

    def put(v):
        q = P.clone()
        q[at] = v
        return q

    dt = 0.5 * dmin
    for _ in range(10):
        a = put(P[at] - dt * rhs(P))
        b = put(0.75 * P[at] + 0.25 * (a[at] - dt * rhs(a)))
        P = put((P[at] + 2.0 * (b[at] - dt * rhs(b))) / 3.0)
    return _inner(P.reshape(gz, gy, gx)).contiguous()


def _walls(q):
    """Boundary values of the conservative variables, in place: z, y, x."""
    q[0:3, 0], q[4, 0], q[3, 0] = q[0:3, 1].clone(), q[4, 1].clone(), 0.0
    for k in (-1, -2):
        q[0, k], q[3, k] = 1.0, 0.0
        q[1:3, k], q[4, k] = q[1:3, -3].clone(), q[4, -3].clone()
    for a, b in ((0, 1), (-1, -2)):
        q[0, :, a], q[4, :, a] = q[0, :, b].clone(), q[4, :, b].clone()
        q[1:4, :, a] = 0.0
    for a, b in ((0, 1), (-1, -2)):
        q[0, :, :, a], q[4, :, :, a] = q[0, :, :, b].clone(), q[4, :, :, b].clone()
        q[1:4, :, :, a] = 0.0
    return q


def _substep(f, case, dev):
    w = _stage(f, case, dev)
    q = _walls(0.75 * f["um0"] + 0.25 * f["um"] + 0.25 * DT * (w["rs"] + w["rsv"]))
    v = (q[1:4] / q[0]).clamp(-6.0, 6.0)
    u = v * f["mask"]
    met, _, _ = _metrics(f["axes"], case["scheme"], dev)
    pres = _extrapolate(q[0] / MACH ** 2, f["sobject"], met, f["dxyz"], f["dmin"])
    um1 = torch.empty_like(q)
    um1[0] = pres * MACH ** 2
    um1[1:4] = u * um1[0]
    um1[4] = q[4]
    return {"um1": um1, "u": u, "temp": q[4].clone(), "pres": pres, **w}


def _adjoint(f, case, dev):
    D = _derivs(f["n"], case["scheme"], dev)
    mats_t = [(_compact(m, case["scheme"]) * (m - 1)).T.contiguous().to(dev) for m in f["n"]]
    Dt = lambda g, d: _along(mats_t[d], g, d)  # noqa: E731
    met, J, iJ = _metrics(f["axes"], case["scheme"], dev)
    dv = _gradient(D, f["u"])
    um, u, vis = f["um"], f["u"], f["vis"]
    # each direction's flux adjoints, then the fluxes' own derivatives
    leaves = [t.detach().clone().requires_grad_() for t in (um, u, f["pres"], vis, dv)]
    total = [torch.zeros_like(t) for t in leaves]
    for d in range(3):
        conv, visc = _fluxes(leaves[0], leaves[1], leaves[2], leaves[3], met, leaves[4], d)
        bars = [J * met[d] * Dt(iJ * f["rs_bar"][k], d) for k in range(5)]
        bars += [J * met[d] * Dt(iJ * f["rsv_bar"][k], d) for k in (1, 2, 3)]
        got = torch.autograd.grad(conv + visc, leaves, bars, allow_unused=True)
        for t, g in zip(total, got):
            if g is not None:
                t += g
    ub = torch.stack([sum(Dt(total[4][3 * d + c], d) for d in range(3)) for c in range(3)])
    return {"um_bar": total[0], "u_bar": total[1], "pres_bar": total[2], "vis_bar": total[3],
            "dvel_bar": total[4], "u_from_dvel": ub}


def _velocity_gradient(met, dv):
    """g[3a+b] = du_a/dx_b."""
    return [met[b] * dv[3 * b + a] for a in range(3) for b in range(3)]


def _dynamic(f, case, dev):
    D = _derivs(f["n"], case["scheme"], dev)
    met, _, _ = _metrics(f["axes"], case["scheme"], dev)
    width, _, _ = _sgd(f["axes"], dev)
    g = _velocity_gradient(met, _gradient(D, f["u"]))
    pairs = [(a, b) for a in range(3) for b in range(a, 3)]
    two = [1.0 if a == b else 2.0 for a, b in pairs]
    S = [0.5 * (g[3 * a + b] + g[3 * b + a]) for a, b in pairs]

    def hat(q):
        for d in range(3):
            q = 0.25 * _clamped(q, d, -1) + 0.5 * q + 0.25 * _clamped(q, d, 1)
        return q

    size = lambda s: torch.sqrt(2.0 * sum(t * v * v for t, v in zip(two, s)))  # noqa: E731
    aS = size(S)
    hS = [hat(s) for s in S]
    ahS = size(hS)
    hu = [hat(v) for v in f["u"]]
    lm = mm = 0.0
    for t, s, h, (a, b) in zip(two, S, hS, pairs):
        L = hat(f["u"][a] * f["u"][b]) - hu[a] * hu[b]
        M = 2.0 * width ** 2 * (hat(aS * s) - 4.0 * ahS * h)
        lm, mm = lm + t * L * M, mm + t * M * M
    hl, hm = hat(lm), hat(mm)
    C = torch.where(hm > 0, hl / hm, torch.zeros_like(hm))
    return (C * width ** 2 * aS).clamp(min=0.0)


def _weights():
    z = np.load(WEIGHTS, allow_pickle=False)
    return [torch.from_numpy(z[k].astype(np.float32)) for k in ("params", "norm")]


def _network(params, norm, feat):
    at = 0
    h = (feat - norm[:10]) * norm[10:20]
    for fan_in, fan_out in ((10, 64), (64, 64), (64, 64), (64, 1)):
        W = params[at:at + fan_in * fan_out].reshape(fan_out, fan_in)
        at += fan_in * fan_out
        h = h @ W.T + params[at:at + fan_out]
        at += fan_out
        h = torch.nn.functional.silu(h) if fan_out > 1 else h
    return norm[20] * torch.nn.functional.softplus(h[:, 0], threshold=200.0)


def _features(f, case, dev):
    D = _derivs(f["n"], case["scheme"], dev)
    met, _, _ = _metrics(f["axes"], case["scheme"], dev)
    width, _, _ = _sgd(f["axes"], dev)
    g = _velocity_gradient(met, _gradient(D, f["u"]))
    return torch.stack([*g, width.expand(g[0].shape)], dim=-1).reshape(-1, 10)


def _train(f, case, dev):
    params, norm = (w.to(dev).double() for w in _weights())
    params.requires_grad_()
    nut = _dynamic(f, case, dev)
    feat = _features(f, case, dev)[f["idx"]]
    nu = _network(params, norm, feat)
    scale = 2.0 / (case["rows"] * float(nut.square().mean()))
    grad, = torch.autograd.grad(nu, params, scale * (nu - nut.reshape(-1)[f["idx"]]).detach())
    m = 0.9 * f["m"].double() + 0.1 * grad
    v = 0.999 * f["v"].double() + 0.001 * grad * grad
    step = (m / (1 - 0.9 ** 101)) / (torch.sqrt(v / (1 - 0.999 ** 101)) + 1e-8)
    return {"nu": nu.detach(), "grad": grad, "params": params.detach() - 1e-4 * step, "m": m, "v": v}


def exact(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    kind = case["kind"]
    if kind == "batch":
        boxes = _box_inputs(case, seed, dev)
        dvel, div, phi = _pools(boxes, dev)
        for z in boxes:
            D = _derivs(z["n"], case["scheme"], dev)
            met, J, iJ = _metrics(z["axes"], case["scheme"], dev)
            _box_view(dvel, z, 9).copy_(_gradient(D, z["u"]))
            _box_view(div, z, 1)[0] = iJ * sum(D(J * met[d] * z["u"][d], d) for d in range(3))
            _box_view(phi, z, 1)[0] = _advect(z["phi"], z["u"], met, z["dxyz"], z["dt"])
        return dvel, div, phi
    f = _inputs(case, seed, dev)
    if kind == "stage":
        return _stage(f, case, dev)
    if kind == "substep":
        return _substep(f, case, dev)
    if kind == "adjoint":
        return _adjoint(f, case, dev)
    if kind == "train":
        return _train(f, case, dev)
    if kind == "dynsmag":
        nut = _dynamic(f, case, dev)
        return nut, C4 + nut
    if kind == "learned":
        params, norm = (w.to(dev).double() for w in _weights())
        feat = _features(f, case, dev)
        nut = torch.cat([_network(params, norm, q) for q in feat.split(1 << 20)])
        nut = nut.reshape(f["u"].shape[1:])
        return nut, C4 + nut
    met, J, iJ = _metrics(f["axes"], case["scheme"], dev)
    if kind == "grad_div":
        D = _derivs(f["n"], case["scheme"], dev)
        return _gradient(D, f["u"]), iJ * sum(D(J * met[d] * f["u"][d], d) for d in range(3))
    if kind == "reinit":
        return _reinit(f["phi"], met, _sgd(f["axes"], dev)[2], f["dxyz"], f["dmin"])
    um = f["um"]
    for d in range(3):
        F = _filter(f["n"][d], d == 2).to(dev)
        um = torch.stack([_along(F, J * q, d) * iJ for q in um])
    return um, um[1:4] / um[0], um[0] / MACH ** 2, um[4].clone()
