"""The measured workloads of this framework: what a user's program has it do,
through the public entry points, over the sizes, regimes and solver modes it
is used at.

Every case is one of these families (key "family"):

  matvec      one application of the scaled 9-point operator
  solve       operator assembly, right-hand side scaling and the pressure
              solve on fields that are already on the GPU
  batch       the pressure solves of many members of different grids together
  solve3d     assembly and solve of the 27-point operator
  projection  the drop-in second projection on host arrays, copies included
  step        one time step with the state resident on the GPU
  ensemble    one lockstep time step of several members
  letkf       one LETKF analysis of an ensemble on the GPU
  train       one training step of the coarse-level network

``exact`` restates the path in 64-bit torch and numpy.  The time step and the
ensemble have none: their result is a composition of nonlinear advection and
two solves to a relative tolerance, compared between implementations only.
"""
import math

import numpy as np
import torch

from pybella_amd import batch as pbatch
from pybella_amd import ensemble as pens
from pybella_amd import letkf as pletkf
from pybella_amd import nn as pnn
from pybella_amd import op3d as pop3
from pybella_amd import second_projection as sp
from pybella_amd import time_update as tu
from pybella_amd import workloads as W

F64 = torch.float64
DT = 0.05          # the projection's time step in units of t_ref
STEP_DT = 0.02     # the fixed step of the time-stepping cases


def listed():
    return [
        # smallest call: one operator application, as a caller's own Krylov loop issues it
        dict(name="matvec_f64_129x65", family="matvec", state="strat", nx=129, ny=65, dtype="f64"),
        # the rising bubble's grid, in the default solver mode (reference semantics)
        dict(name="solve_f64_161x81", family="solve", state="bubble", nx=161, ny=81, mode="f64"),
        # the isolated stratified solve, plain Krylov
        dict(name="solve_fast_1025x513", family="solve", state="strat", nx=1025, ny=513, mode="f64fast"),
        # the same solve with the learned preconditioner
        dict(name="solve_nn_1025x513", family="solve", state="strat", nx=1025, ny=513, mode="nn"),
        # ensemble members of uneven grids, FP32 inner solves
        dict(name="batch_mixed_513x257", family="batch", members=9, nx=513, ny=257, mode="mixed"),
        # 3D: the full-size solve in mixed precision, and an odd-sized one in FP64
        dict(name="solve3d_mixed_257x129x129", family="solve3d", nx=257, ny=129, nz=129, mode="mixed"),
        dict(name="solve3d_f64_150x75x67", family="solve3d", nx=150, ny=75, nz=67, mode="f64"),
        # the drop-in call of a host program: compressible, with Coriolis, ragged size
        dict(name="projection_f64_300x150", family="projection", state="coriolis", nx=300, ny=150, mode="f64"),
        # the rising-bubble time step
        dict(name="step_f64_161x81", family="step", state="bubble", nx=161, ny=81, mode="f64"),
        # ensemble stepping and its analysis
        dict(name="ensemble_16x161x81", family="ensemble", members=16, nx=161, ny=81, mode="f64fast"),
        dict(name="letkf_16x161x81", family="letkf", members=16, attrs=5, window=11, nx=161, ny=81),
        # training: a batch of coarse-level images
        dict(name="train_32x33x65", family="train", images=32, h=33, w=65),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _half(rng, nx):
    """Rows for a grid of nx columns: cells within a third of square (the
    domain is twice as wide as tall)."""
    return max(9, int(round(0.5 * nx * math.exp(rng.uniform(math.log(0.75), math.log(1.33))))))


def draw(rng):
    family = rng.choice(("matvec", "solve", "solve", "solve_nn", "batch", "solve3d", "projection", "step",
                         "ensemble", "letkf", "train"))
    if family == "matvec":
        return dict(family=family, state=rng.choice(("strat", "comp", "coriolis", "xwall")), nx=_log(rng, 9, 2049),
                    ny=_log(rng, 9, 1025), dtype=rng.choice(("f64", "f32")))
    if family == "solve":
        nx = _log(rng, 33, 897)
        return dict(family=family, state=rng.choice(("strat", "bubble", "comp", "coriolis", "xwall")), nx=nx,
                    ny=_half(rng, nx), mode=rng.choice(("f64", "f64fast", "mixed")))
    if family == "solve_nn":   # grids that coarsen to a level like the one the network was trained on
        k, i = 2 ** rng.randint(2, 4), rng.choice((3, 4))
        return dict(family="solve", state=rng.choice(("strat", "comp", "bubble")), nx=16 * i * k + 1, ny=8 * i * k + 1,
                    mode="nn")
    if family == "batch":
        nx = _log(rng, 97, 513)
        return dict(family=family, members=rng.randint(2, 12), nx=nx, ny=_half(rng, nx),
                    mode=rng.choice(("f64fast", "mixed")))
    if family == "solve3d":
        return dict(family=family, nx=_log(rng, 33, 257), ny=_log(rng, 17, 129), nz=_log(rng, 17, 129),
                    mode=rng.choice(("f64", "mixed")))
    if family == "projection":
        nx = _log(rng, 65, 513)
        return dict(family=family, state=rng.choice(("psinc", "comp", "coriolis", "xwall")), nx=nx,
                    ny=_half(rng, nx), mode=rng.choice(("f64", "f64fast")))
    if family == "step":
        state = rng.choice(("bubble", "bubble", "vortex"))
        nx = _log(rng, 33, 321) if state == "bubble" else 2 * _log(rng, 16, 64) + 1   # no cell at the vortex's centre
        return dict(family=family, state=state, nx=nx, ny=_half(rng, nx) if state == "bubble" else nx,
                    mode=rng.choice(("f64", "f64fast")))
    if family == "ensemble":
        nx = _log(rng, 65, 193)
        return dict(family=family, members=rng.randint(2, 20), nx=nx, ny=_half(rng, nx), mode="f64fast")
    if family == "letkf":
        return dict(family=family, members=rng.randint(3, 32), attrs=rng.randint(1, 5),
                    window=rng.choice((5, 7, 9, 11, 13)), nx=_log(rng, 33, 161), ny=_log(rng, 33, 81))
    return dict(family="train", images=rng.randint(1, 32), h=rng.choice((17, 25, 33)), w=rng.choice((33, 49, 65)))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev(a):
    """Host [x, y] array -> device [y][x] tensor."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.float64).T)).to("cuda")


def _state(kind, nx, ny, seed):
    """(Sol, mpv, elem, node, ud, th): the stratified atmosphere (pseudo-
    incompressible "strat"; compressible "comp"; with Coriolis; with walls in
    x) or the rising bubble, its bubble from the seed."""
    rng = np.random.default_rng(seed)
    if kind == "bubble":
        Sol, _, mpv, elem, node, ud, th = W.rising_bubble_state(
            nx, ny, delth=rng.uniform(1.0, 3.0), xc=rng.uniform(-0.3, 0.3), r0=rng.uniform(0.15, 0.25), dt=DT)
    else:
        Sol, mpv, elem, node, ud, th = W.stratified_state(nx, ny, theta1=rng.uniform(320.0, 340.0),
                                                          compressible=kind in ("comp", "coriolis", "xwall"))
    if kind == "coriolis":
        ud.omega = 7.292e-5 * 50
        ud.derive()
    if kind == "xwall":
        ud.bdry_type[0] = W.BdryType.WALL
    return Sol, mpv, elem, node, ud, th


def _rhs3d(nx, ny, nz, seed):
    """Smooth zero-mean node field (nz, ny, nx) of 48 seeded modes, made on
    the GPU as three contractions."""
    rng = np.random.default_rng(seed)
    m = 48
    k = rng.integers(0, 9, (3, m))
    k[2] += (k.sum(0) == 0)
    phi = rng.uniform(0.0, 2.0 * np.pi, (2, m))
    amp = rng.standard_normal(m)
    g = lambda a: torch.from_numpy(a).to("cuda")
    fx = g(np.cos(2 * np.pi * np.outer(k[0], np.linspace(0, 1, nx)) + phi[0][:, None]))
    fy = g(np.cos(np.pi * np.outer(k[1], np.linspace(0, 1, ny))) * amp[:, None])
    fz = g(np.cos(2 * np.pi * np.outer(k[2], np.linspace(0, 1, nz)) + phi[1][:, None]))
    fx[:, -1], fz[:, -1] = fx[:, 0], fz[:, 0]
    yx = (fy[:, :, None] * fx[:, None, :]).reshape(m, ny * nx)
    return (fz.t().contiguous() @ yx).reshape(nz, ny, nx).contiguous()


class _Holder:
    """What a case keeps between passes."""


def _prepare_solve(c, seed):
    s = _Holder()
    Sol, mpv, elem, node, ud, th = _state(c["state"], c["nx"], c["ny"], seed)
    s.phys = sp.phys_of(ud, th)
    s.op = sp.Operator2D(sp.grid_of(node, ud))
    s.rho, s.rhoY = _dev(Sol.rho), _dev(Sol.rhoY)
    s.dS = _dev(sp.dSdy_cells(mpv, elem, node))
    s.rhs = _dev(W.stratified_rhs(node, seed=seed))
    s.tol = 1e-8
    if c["mode"] == "nn":
        s.net = pnn.Network()
        s.net.load(pnn.default_weights_path())
        s.op.attach_nn(s.net)
    return s


def _batch_sizes(c):
    """Uneven members: every third one at the full, half and quarter size."""
    return [(max(17, ((c["nx"] - 1) >> (m % 3)) + 1), max(9, ((c["ny"] - 1) >> (m % 3)) + 1))
            for m in range(c["members"])]


def _prepare_batch(c, seed):
    s = _Holder()
    s.ops, s.bs = [], []
    for m, (nx, ny) in enumerate(_batch_sizes(c)):
        Sol, mpv, elem, node, ud, th = _state("bubble", nx, ny, seed + 1000 * m)
        op = sp.Operator2D(sp.grid_of(node, ud))
        rho, rhoY, dS = _dev(Sol.rho), _dev(Sol.rhoY), _dev(sp.dSdy_cells(mpv, elem, node))
        op.assemble(sp.phys_of(ud, th), DT, rho, rhoY, rho, rhoY, dS)
        s.ops.append(op)
        s.bs.append(op.scale_rhs(_dev(W.stratified_rhs(node, seed=seed + 1000 * m))))
    s.batch = pbatch.BatchSolver(s.ops)
    return s


def _projection_state(c, seed):
    """Host state of a projection: smooth random momenta on the state."""
    kind = {"psinc": "strat"}.get(c["state"], c["state"])
    Sol, mpv, elem, node, ud, th = _state(kind, c["nx"], c["ny"], seed)
    rng = np.random.default_rng(seed + 1)
    X, Y = np.meshgrid(elem.x, elem.y, indexing="ij")
    for f in (Sol.rhou, Sol.rhov, Sol.rhoX):
        for _ in range(6):
            kx, ky = rng.integers(1, 5, 2)
            f += rng.standard_normal() * np.cos(np.pi * kx * X + rng.uniform(0, 6.3)) * \
                np.sin(np.pi * ky * Y + rng.uniform(0, 6.3))
        f *= 0.1 * Sol.rho
    p = np.zeros_like(mpv.p2_nodes)
    xn, yn = np.meshgrid(node.x, node.y, indexing="ij")
    for _ in range(4):
        kx, ky = rng.integers(1, 4, 2)
        p += 0.01 * rng.standard_normal() * np.cos(np.pi * kx * xn + rng.uniform(0, 6.3)) * np.cos(np.pi * ky * yn)
    mpv.p2_nodes[...] = p
    ud.tol = 1e-8
    return Sol, mpv, elem, node, ud, th


def _prepare_projection(c, seed):
    s = _Holder()
    s.Sol, s.mpv, s.elem, s.node, s.ud, s.th = _projection_state(c, seed)
    s.keep = [(a, a.copy()) for a in (s.Sol.rhou, s.Sol.rhov, s.Sol.rhow, s.Sol.rhoX, s.Sol.rho, s.Sol.rhoY,
                                      s.mpv.p2_nodes)]
    s.mode = c["mode"]
    return s


def _prepare_step(c, seed):
    s = _Holder()
    rng = np.random.default_rng(seed)
    s.mode = c["mode"]
    if c["state"] == "vortex":
        ud = W.travelling_vortex_ud(c["nx"])
        ud.u_wind_speed, ud.v_wind_speed = rng.uniform(0.5, 1.5, 2)
        sp.solver_options["mode"] = c["mode"]
        host = W.travelling_vortex_init(sp.euler_backward_non_advective_impl_part, ud)
        sp.solver_options["mode"] = "f64"
    else:
        ud = W.rising_bubble_ud(c["nx"], c["ny"])
        ud.aux, ud.dtfixed, ud.dtfixed0 = "", STEP_DT, STEP_DT
        host = W.rising_bubble_init(ud, delth=rng.uniform(1.0, 3.0), xc=rng.uniform(-0.3, 0.3),
                                    r0=rng.uniform(0.15, 0.25))
    Sol, flux, mpv, elem, node, ud, th = host
    s.M = tu.DeviceModel(elem, node, ud, th, op=sp.Operator2D(sp.grid_of(node, ud)))
    s.M.upload(Sol, flux, mpv)
    s.t, s.k = 0.0, 0
    return s


def _prepare_ensemble(c, seed):
    s = _Holder()
    members, elem, node, ud, th = pens.rising_bubble_members(c["members"], c["nx"], c["ny"], base_seed=seed)
    ud.aux, ud.dtfixed, ud.dtfixed0 = "", STEP_DT, STEP_DT
    s.ens = pens.Ensemble(members, elem, node, ud, th, mode=c["mode"])
    s.ts, s.k = [0.0] * c["members"], 0
    return s


_LETKF_ATTRS = ("rho", "rhou", "rhov", "rhoY", "p2_nodes")


def _letkf_inputs(c, seed):
    """Forecast fields (ghost layers included), observations, masks and
    variances on the host: smooth member perturbations of a bubble-like field,
    a third of the locations unobserved."""
    rng = np.random.default_rng(seed)
    nx, ny, k = c["nx"], c["ny"], c["members"]
    out = []
    for a in _LETKF_ATTRS[:c["attrs"]]:
        cx, cy = (nx, ny) if a == "p2_nodes" else (nx - 1, ny - 1)
        x, y = np.linspace(-1, 1, cx + 4)[:, None], np.linspace(0, 1, cy + 4)[None, :]
        base = np.exp(-4 * (x ** 2 + (y - 0.5) ** 2))
        f = np.stack([base + 0.1 * sum(rng.standard_normal() * np.cos(np.pi * (i + 1) * x + rng.uniform(0, 6.3)) *
                                       np.cos(np.pi * j * y + rng.uniform(0, 6.3)) for i in range(3) for j in range(2))
                      for _ in range(k)])
        truth = f.mean(0) + 0.05 * rng.standard_normal(base.shape)
        out.append((a, f, truth[2:-2, 2:-2], (rng.random((cx, cy)) < 1 / 3).astype(float), 0.01 * rng.uniform(0.5, 2)))
    return out


def _prepare_letkf(c, seed):
    s = _Holder()
    ud = W.rising_bubble_ud(c["nx"], c["ny"])
    Sol, flux, mpv, elem, node, ud, th = W.rising_bubble_init(ud)
    op = sp.Operator2D(sp.grid_of(node, ud))
    s.models = [tu.DeviceModel(elem, node, ud, th, op=op) for _ in range(c["members"])]
    inputs = _letkf_inputs(c, seed)
    attrs = [i[0] for i in inputs]
    s.da = pletkf.LETKF(ud, attributes=attrs, obs_X=c["window"], obs_Y=c["window"], inflation=1.05)
    s.obs = {a: o for a, _, o, _, _ in inputs}
    s.mask = {a: m for a, _, _, m, _ in inputs}
    s.covar = {a: v for a, _, _, _, v in inputs}
    s.fields, s.forecast = [], []
    for a, f, _, _, _ in inputs:
        for m, M in enumerate(s.models):
            s.fields.append(M.p2n if a == "p2_nodes" else M.sol.f[a])
            s.forecast.append(_dev(f[m]))
    s.shape = (len(attrs), c["members"])
    return s


def _train_inputs(c, seed):
    """Normalised residual, the two coefficient features and a smooth target
    without constant and checkerboard parts."""
    g = torch.Generator().manual_seed(int(seed))
    n, h, w = c["images"], c["h"], c["w"]
    y, x = torch.arange(h, dtype=F64)[:, None], torch.arange(w, dtype=F64)[None, :]
    X = torch.randn(n, h, w, 3, generator=g, dtype=F64)
    T = torch.zeros(n, h, w, dtype=F64)
    for _ in range(6):
        a, kx, ky, p, q = (torch.rand(n, 1, 1, generator=g, dtype=F64) for _ in range(5))
        T += (a - 0.5) * torch.cos(6.28 * (4 * kx * x / w + p)) * torch.cos(6.28 * (2 * ky * y / h + q))
    X[..., 1] = 1.0 + 0.1 * torch.cos(3.0 * x / w)
    X[..., 2] = 0.2 + 0.05 * torch.cos(2.0 * y / h)
    T = _no_null(T)
    T /= T.square().mean((1, 2), keepdim=True).sqrt()
    return X.float(), T.float()


def _prepare_train(c, seed):
    s = _Holder()
    X, T = _train_inputs(c, seed)
    s.X, s.T = X.cuda(), T.cuda()
    s.net = pnn.Network(seed=3)
    return s


def _prepare_matvec(c, seed):
    s = _Holder()
    Sol, mpv, elem, node, ud, th = _state(c["state"], c["nx"], c["ny"], seed)
    s.op = sp.Operator2D(sp.grid_of(node, ud))
    rho, rhoY, dS = _dev(Sol.rho), _dev(Sol.rhoY), _dev(sp.dSdy_cells(mpv, elem, node))
    s.op.assemble(sp.phys_of(ud, th), DT, rho, rhoY, rho, rhoY, dS)
    s.x = _dev(_matvec_input(c, seed)).to(torch.float64 if c["dtype"] == "f64" else torch.float32)
    return s


def _matvec_input(c, seed):
    return np.random.default_rng(seed + 7).standard_normal((c["nx"], c["ny"]))


def _prepare_solve3d(c, seed):
    s = _Holder()
    s.st = _state3d(c, seed)
    s.op = pop3.Operator3D(pop3.grid3_of(s.st))
    s.phys = pop3.phys3_of(s.st)
    s.rho, s.rhoY = (torch.from_numpy(a).to("cuda") for a in (s.st.rho_c, s.st.rhoY_c))
    s.rhs = _rhs3d(c["nx"], c["ny"], c["nz"], seed)
    s.dinv = torch.empty(c["nz"], c["ny"], c["nx"], dtype=F64, device="cuda")
    return s


def _state3d(c, seed):
    theta1 = np.random.default_rng(seed).uniform(320.0, 340.0)
    return W.stratified_state_3d(c["nx"], c["ny"], c["nz"], theta1=theta1)


def prepare(case, seed):
    return globals()["_prepare_" + case["family"]](case, seed).__dict__ | {"case": case}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
class _View:
    def __init__(self, d):
        self.__dict__ = d


def run(state):
    s = _View(state)
    c = s.case
    fam = c["family"]
    if fam == "matvec":
        return s.op.matvec(s.x)
    if fam == "solve":
        s.op.assemble(s.phys, DT, s.rho, s.rhoY, s.rho, s.rhoY, s.dS)
        b = s.op.scale_rhs(s.rhs)
        if c["mode"] == "nn":
            x, _ = s.op.solve(b, tol=s.tol, maxiter=300, mode="nn")
        else:
            x, _ = s.op.solve(b, tol=s.tol, maxiter=6000, mode=c["mode"])
        return {"b": b, "x": x}
    if fam == "batch":
        return s.batch.solve(s.bs, tol=1e-8, mode=c["mode"])[0]
    if fam == "solve3d":
        s.op.assemble(s.phys, DT, s.rho, s.rhoY, diag_inv=s.dinv)
        return s.op.solve(s.dinv * s.rhs, tol=1e-8, mode=c["mode"])[0]
    if fam == "projection":
        for a, kept in s.keep:      # the host program's state before the call
            np.copyto(a, kept)
        sp.solver_options["mode"] = s.mode
        sp.euler_backward_non_advective_impl_part(s.Sol, s.mpv, s.elem, s.node, s.ud, s.th, 0.0, DT, 1.0)
        sp.solver_options["mode"] = "f64"
        return {"rhou": s.Sol.rhou, "rhov": s.Sol.rhov, "rhoX": s.Sol.rhoX, "p2_nodes": s.mpv.p2_nodes,
                "rhs": s.mpv.rhs}
    if fam == "step":
        sp.solver_options["mode"] = s.mode
        dt = tu.step(s.M, s.t, 1e9, s.k, s.k)[0]
        sp.solver_options["mode"] = "f64"
        state["t"], state["k"] = s.t + dt, s.k + 1
        return {**s.M.sol.f, "p2_nodes": s.M.p2n}
    if fam == "ensemble":
        recs = s.ens.step(s.ts, 1e9, s.k, s.k)
        state["ts"], state["k"] = [t + r[0] for t, r in zip(s.ts, recs)], s.k + 1
        return [[M.sol.f["rho"], M.sol.f["rhou"], M.sol.f["rhov"]] for M in s.ens.models]
    if fam == "letkf":
        torch._foreach_copy_(s.fields, s.forecast)      # the members as the forecast leaves them
        s.da.analyse(s.models, s.obs, s.mask, s.covar)
        na, k = s.shape
        return [torch.stack(s.fields[a * k:(a + 1) * k]) for a in range(na)]
    z = torch.empty(s.X.shape[:3], dtype=torch.float32, device="cuda")
    loss = s.net.step(s.X, s.T, lr=1.5e-3, out_z=z)
    return {"loss": loss, "z": z, "grads": s.net.get_grads(), "params": s.net.get_params()}


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
_CONV = ((3, 16, 1), (16, 16, 1), (16, 32, 2), (32, 32, 2), (32, 64, 4), (64, 64, 4), (64, 64, 8), (64, 64, 8),
         (128, 64, 4), (64, 64, 4), (96, 32, 2), (32, 32, 2), (48, 16, 1), (16, 16, 1), (16, 1, 1))


def work(case):
    """Inputs read once and outputs written once; floating-point operations of
    the iterations that the method needs (measured counts, by grid width)."""
    c, fam = case, case["family"]
    n = c.get("nx", 0) * c.get("ny", 0)
    if fam == "matvec":
        return {"bytes": n * 5 * (8 if c["dtype"] == "f64" else 4), "flops": 25.0 * n}
    iters = 1.1 * max(c.get("nx", 0), 2 * c.get("ny", 0))     # two applications and ten vector operations each
    if fam == "solve":
        return {"bytes": 8.0 * 6 * n, "flops": (20 * 600.0 if c["mode"] == "nn" else 70.0 * iters) * n}
    if fam == "batch":
        sizes = _batch_sizes(c)
        return {"bytes": sum(8.0 * 5 * a * b for a, b in sizes),
                "flops": sum(70.0 * 1.1 * max(a, 2 * b) * a * b for a, b in sizes)}
    if fam == "solve3d":
        m = n * c["nz"]
        return {"bytes": 8.0 * 5 * m, "flops": 160.0 * 150 * m}
    if fam == "projection":
        return {"bytes": 8.0 * 28 * n, "flops": 70.0 * iters * n}
    if fam == "step":
        return {"bytes": 8.0 * 14 * n, "flops": 2 * 70.0 * iters * n}
    if fam == "ensemble":
        return {"bytes": c["members"] * 8.0 * 14 * n, "flops": c["members"] * 2 * 70.0 * iters * n}
    if fam == "letkf":
        k, a = c["members"], c["attrs"]
        obs = a * c["window"] ** 2
        return {"bytes": 8.0 * n * a * (2 * k + 2), "flops": n * (obs * k * (k + 3.0) + 20.0 * k ** 3)}
    pix = c["images"] * c["h"] * c["w"]
    return {"bytes": 4.0 * pix * 5 + 4.0 * 302977 * 6,
            "flops": 3 * sum(2.0 * 9 * ci * co * pix / f ** 2 for ci, co, f in _CONV)}


def _null_free(case):
    """Pseudo-incompressible solves in FP32 or with FP32 preconditioning: the
    operator's null space (constant, checkerboard) stays in the solution with
    whatever amplitude that arithmetic gives it, and has no exact value."""
    return (case["family"] == "batch" or case["family"] == "solve" and case["state"] in ("strat", "bubble")) and \
        case["mode"] in ("mixed", "nn")


def tolerance(case):
    fam = case["family"]
    if fam == "matvec":
        return {"rel": 1e-13, "max": 1e-12} if case["dtype"] == "f64" else {"rel": 2e-6, "max": 1e-4}
    if _null_free(case):
        return {"rel": 3e-2, "max": 0.5} if case["mode"] == "nn" else {"rel": 2e-3, "max": 2e-2}
    # solves to a relative residual of 1e-8; another summation order moves x by
    # up to 2e-7, and a step's fields (the bubble's small momenta) by up to 4e-5
    if fam in ("solve", "batch", "solve3d", "projection"):
        return {"rel": 2e-6, "max": 1e-5}
    if fam in ("step", "ensemble"):
        return {"rel": 1.7e-4, "max": 4e-4}
    if fam == "letkf":
        return {"rel": 1e-11, "max": 1e-9}
    return {"rel": 1e-2, "max": 0.2}             # BF16 network


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _box(a):
    return a[:-1, :-1] + a[1:, :-1] + a[:-1, 1:] + a[1:, 1:]


def _dSdy(mpv, elem, node):
    S0 = np.asarray(mpv.HydroState_n.S0)
    return np.repeat(((S0[1:] - S0[:-1]) / node.dy)[None, :], elem.sc[0], axis=0)


def _wall(ud, d):
    return ud.bdry_type[d].name != "PERIODIC"


def _coriolis(rho, rhoY, dS, ud, dt):
    """The four factors of the implicit Coriolis and buoyancy matrix's inverse
    in the plane, and their common divisor applied."""
    wh1, wv, wh2 = dt * ud.coriolis_strength
    nu = -dt ** 2 * (ud.gravity_strength[1] / ud.Msq) * dS * rhoY / rho
    nh = ud.nonhydrostasy
    den = wh1 ** 2 + wh2 ** 2 + (nu + nh) * (wv ** 2 + 1.0)
    return (wh1 ** 2 + nu + nh) / den, nh * (wh1 * wv + wh2) / den, (wh1 * wv - wh2) / den, nh * (1 + wv ** 2) / den


class _Op2:
    """The scaled 9-point operator in 64-bit torch, from [x, y] cell fields (x
    periodic where it is singular)."""

    def __init__(self, rho_w, rhoY_w, rho_c, rhoY_c, dS, node, ud, th, dt):
        coeff = th.Gammainv * rhoY_w * rhoY_w / rho_w
        wc = -ud.Msq * th.gm1inv / dt ** 2 * _box(rhoY_w ** (2.0 - th.gamm)) / 4.0
        sl = [slice(2, -2), slice(2, -2)]   # wall node rows count half; the other axis' end nodes do not,
        for d in (0, 1):                    # and after x walls only the corners of the first column do
            if _wall(ud, d):
                for e in (-2, 1):
                    sl[d] = e
                    wc[tuple(sl)] *= 0.5
        if ud.is_compressible == 0:
            wc = wc * ud.compressibility
        dx, dy = node.dx, node.dy
        diag = wc - 0.75 * _box(coeff) * (1 / dx ** 2 + 1 / dy ** 2 + 2 / (dx * dy))
        self.dinv_isc = 1.0 / diag
        uu, uv, vu, vv = (a[1:-1, 1:-1] + np.zeros_like(coeff[1:-1, 1:-1]) for a in _coriolis(rho_c, rhoY_c, dS, ud, dt))
        h = coeff[1:-1, 1:-1].copy()
        if _wall(ud, 0):
            h[0] = h[-1] = 0.0
        if _wall(ud, 1):
            h[:, 0] = h[:, -1] = 0.0
        g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
        # node sums of the cell fluxes: x rows (uu, uv), y rows (vu, vv)
        self.wxx, self.wyy = g(h * uu / (4 * dx * dx)), g(h * vv / (4 * dy * dy))
        self.wyx, self.wxy = g(h * uv / (4 * dx * dy)), g(h * vu / (4 * dx * dy))
        self.hc, self.dinv = g(wc[1:-1, 1:-1]), g(self.dinv_isc[1:-1, 1:-1])
        nx, ny = self.hc.shape
        self.ix = torch.tensor([nx - 2, *range(nx), 1], device="cuda")
        self.iy = torch.tensor([ny - 2, *range(ny), 1], device="cuda")

        self.null = None
        if not np.any(wc):     # null vectors: the constant and, where the wrap closes it, the checkerboard
            w = torch.ones_like(self.hc)
            w[0], w[-1] = 0.5, 0.5
            i, j = torch.arange(nx, device="cuda")[:, None], torch.arange(ny, device="cuda")[None, :]
            n = [torch.ones_like(w)] + ([1.0 - 2.0 * ((i + j) % 2).to(F64)] if nx % 2 else [])
            self.null = torch.stack([a.reshape(-1) for a in n], 1)
            self.left = torch.stack([(a * w / self.dinv).reshape(-1) for a in n], 0)

    def clean(self, v):
        """v without what the left null vectors see of it: they are orthogonal
        to the range, so to every vector of a Krylov space from it."""
        if self.null is None:
            return v
        return v - (self.null @ torch.linalg.solve(self.left @ self.null, self.left @ v.reshape(-1))).reshape(v.shape)

    def __call__(self, p):
        e = p[self.ix][:, self.iy]
        dx, dy = e[1:] - e[:-1], e[:, 1:] - e[:, :-1]
        gx, gy = dx[:, :-1] + dx[:, 1:], dy[:-1] + dy[1:]
        fx, fy = self.wxx * gx + self.wyx * gy, self.wyy * gy + self.wxy * gx
        sx, sy = fx[:, :-1] + fx[:, 1:], fy[:-1] + fy[1:]
        return self.dinv * ((sx[1:] - sx[:-1]) + (sy[:, 1:] - sy[:, :-1]) + self.hc * p)


def _bicgstab(A, b, tol=1e-12, rounds=8, maxit=4000):
    """x with ||b - A x|| <= tol ||b|| where attainable: BiCGStab, each round
    from the true residual and ending with its best iterate.  For a singular
    operator, the solution that its Krylov space from b holds."""
    clean = getattr(A, "clean", lambda v: v)
    x, r, bn = torch.zeros_like(b), b, float(b.norm())
    best = bn
    for _ in range(rounds):
        if best <= tol * bn:
            break
        y, kept, low = torch.zeros_like(b), torch.zeros_like(b), best
        rt, p, q = r, r, r
        rho = (rt * q).sum()
        for it in range(maxit):
            v = A(p)
            alpha = rho / (rt * v).sum()
            s = q - alpha * v
            t = A(s)
            om = (t * s).sum() / (t * t).sum()
            y = y + alpha * p + om * s
            q = s - om * t
            new = (rt * q).sum()
            p = q + (new / rho) * (alpha / om) * (p - om * v)
            rho = new
            if it % 8 == 7:
                n = float(q.norm())
                if n < low:
                    kept, low = y, n
                if not math.isfinite(n) or n <= 0.1 * tol * bn or n > 1e8 * low:
                    break
        r2 = b - A(x + kept)
        if not (float(r2.norm()) < 0.9 * best):
            break
        x, r, best = clean(x + kept), clean(r2), float(r2.norm())
    return x


def _exact_op2(state, nx, ny, seed):
    Sol, mpv, elem, node, ud, th = _state(state, nx, ny, seed)
    return _Op2(Sol.rho, Sol.rhoY, Sol.rho, Sol.rhoY, _dSdy(mpv, elem, node), node, ud, th, DT), node


def _exact_solve(state, nx, ny, seed):
    A, node = _exact_op2(state, nx, ny, seed)
    b = torch.from_numpy((A.dinv_isc * W.stratified_rhs(node, seed=seed))[1:-1, 1:-1].copy()).to("cuda")
    return b, _bicgstab(A, b)


def _ghost_cells(f, elem, ud, th, mpv):
    """Cell ghost fill of the fields rho, rhou, rhov, rhow, rhoY, rhoX."""
    if _wall(ud, 0):
        pad = lambda a, s: np.concatenate([s * a[3:1:-1], a[2:-2], s * a[-3:-5:-1]])
    else:
        pad = lambda a, s: np.concatenate([a[-4:-2], a[2:-2], a[2:4]])
    for k in f:
        if not (_wall(ud, 0) and k == "rhow"):
            f[k][...] = pad(f[k], -1.0 if k == "rhov" else 1.0)
    g, n = ud.gravity_strength[1], elem.icy
    for d, order in ((1, (1, 0)), (-1, (n - 2, n - 1))):
        for j in order:
            last, src = j + d, (3 - j if d > 0 else 2 * n - 5 - j)
            S = 1.0 / ud.stratification(elem.y[j])
            Yl = f["rhoY"][:, last] / f["rho"][:, last]
            if ud.is_compressible == 1:
                dpi = d * th.Gamma * g * 0.5 * elem.dy * (1.0 / Yl + S)
                rhoY = (f["rhoY"][:, last] ** th.gm1 + dpi) ** th.gm1inv
            else:
                rhoY = mpv.HydroState.rhoY0[j] + 0 * Yl
            vY = -f["rhov"][:, src] * f["rhoY"][:, src] / f["rho"][:, src]
            rest = {k: f[k][:, src] / f["rho"][:, src] for k in ("rhou", "rhow", "rhoX")}
            f["rho"][:, j], f["rhoY"][:, j] = rhoY * S, rhoY
            f["rhov"][:, j] = rhoY * S * vY / rhoY
            for k, a in rest.items():
                f[k][:, j] = rhoY * S * a


def _ghost_nodes(p, ud):
    for d in (0, 1):
        q = np.moveaxis(p, d, 0)
        if _wall(ud, d):
            q[:2], q[-2:] = q[4:2:-1].copy(), q[-4:-6:-1].copy()
        else:
            lo, hi = q[2:5].copy(), q[-5:-2].copy()
            q[:3], q[-3:] = hi, lo


def _correct(f, p, dS, node, ud, th, dt, chi):
    a = (p[1:, :-1] - p[:-1, :-1], p[1:, 1:] - p[:-1, 1:], p[:-1, 1:] - p[:-1, :-1], p[1:, 1:] - p[1:, :-1])
    c = -dt * th.Gammainv * f["rhoY"] * f["rhoY"] / f["rho"]
    u, v = c * 0.5 * (a[0] + a[1]) / node.dx, c * 0.5 * (a[2] + a[3]) / node.dy
    uu, uv, vu, vv = _coriolis(f["rho"], f["rhoY"], dS, ud, dt)
    f["rhou"] += f["rho"] / f["rhoY"] * (uu * u + uv * v)
    f["rhov"] += f["rho"] / f["rhoY"] * (vu * u + vv * v)
    f["rhoX"] -= chi * dt * dS * f["rhov"]


def _exact_projection(c, seed):
    Sol, mpv, elem, node, ud, th = _projection_state(c, seed)
    f = {k: getattr(Sol, k) for k in ("rho", "rhou", "rhov", "rhow", "rhoY", "rhoX")}
    p2, dS = mpv.p2_nodes, _dSdy(mpv, elem, node)
    _ghost_cells(f, elem, ud, th, mpv)
    rho_w, rhoY_w = f["rho"].copy(), f["rhoY"].copy()
    _ghost_nodes(p2, ud)
    _correct(f, p2, dS, node, ud, th, DT, 0.0)
    _ghost_cells(f, elem, ud, th, mpv)
    for k in ("rhou", "rhov", "rhow"):
        f[k][:, :2] = f[k][:, -2:] = 0.0
    U, V = f["rhou"] * f["rhoY"] / f["rho"], f["rhov"] * f["rhoY"] / f["rho"]
    dU, dV = (U[1:] - U[:-1]) / elem.dx, (V[:, 1:] - V[:, :-1]) / elem.dy
    rhs = (0.5 * (dU[:, :-1] + dU[:, 1:]) + 0.5 * (dV[:-1] + dV[1:])) / DT
    A = _Op2(rho_w, rhoY_w, f["rho"], f["rhoY"], dS, node, ud, th, DT)
    x = _bicgstab(A, torch.from_numpy((A.dinv_isc * rhs)[1:-1, 1:-1].copy()).to("cuda")).cpu().numpy()
    full = np.zeros_like(p2)
    full[2:-2, 2:-2] = x
    _ghost_nodes(full, ud)
    _correct(f, full, dS, node, ud, th, DT, 1.0)
    p2 += full
    _ghost_nodes(p2, ud)
    _ghost_cells(f, elem, ud, th, mpv)
    return {"rhou": f["rhou"], "rhov": f["rhov"], "rhoX": f["rhoX"], "p2_nodes": p2, "rhs": rhs}


def _exact_solve3d(c, seed):
    st = _state3d(c, seed)
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    rho, rhoY, th, ud = g(st.rho_c), g(st.rhoY_c), st.th, st.ud
    coeff = th.Gammainv * rhoY * rhoY / rho

    def box(a):
        a = a[1:] + a[:-1]
        a = a[:, 1:] + a[:, :-1]
        return a[:, :, 1:] + a[:, :, :-1]

    wc = -ud.Msq * th.gm1inv / DT ** 2 * box(rhoY ** (2.0 - th.gamm)) / 8.0
    wc[1:-1, 0, 1:-1] *= 0.5
    wc[1:-1, -1, 1:-1] *= 0.5
    dx, dy, dz = st.dx, st.dy, st.dz
    dinv = 1.0 / (wc - box(coeff) / 16.0 * (1 / dx ** 2 + 1 / dy ** 2 + 1 / dz ** 2 + 2 / (dx * dy)))
    h = coeff / 16.0
    h[:, 0] = 0.0
    h[:, -1] = 0.0
    ext = [torch.tensor([n - 2, *range(n), 1], device="cuda") for n in (st.nz, st.ny, st.nx)]

    def pair(a, d, sign=1.0):
        n = a.shape[d] - 1
        return a.narrow(d, 1, n) + sign * a.narrow(d, 0, n)

    def A(p):
        e = p[ext[0]][:, ext[1]][:, :, ext[2]]
        y = wc * p
        for d, w in ((0, dz), (1, dy), (2, dx)):
            o = [k for k in (0, 1, 2) if k != d]
            fl = h / w ** 2 * pair(pair(pair(e, d, -1.0), o[0]), o[1])
            y = y + pair(pair(pair(fl, o[0]), o[1]), d, -1.0)
        return dinv * y

    return _bicgstab(A, dinv * _rhs3d(c["nx"], c["ny"], c["nz"], seed), maxit=1200)


def _exact_letkf(c, seed):
    inputs, k, o = _letkf_inputs(c, seed), c["members"], c["window"]
    x = np.linspace(0, 1, o) - 0.5
    Z = np.exp(-(x[:, None] ** 2 + x[None, :] ** 2) / 0.1)
    Z = (Z - Z.min()) / (Z.max() - Z.min())
    g = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    out = []
    for group in ([i for i in inputs if i[0] != "p2_nodes"], [i for i in inputs if i[0] == "p2_nodes"]):
        if not group:
            continue
        F = torch.stack([g(i[1])[:, 2:-2, 2:-2] for i in group], 1)          # (k, attrs, X, Y)
        obs, seen = g(np.stack([i[2] for i in group])), 1.0 - g(np.stack([i[3] for i in group]))
        var = g(np.array([i[4] for i in group]))
        nX, nY, r = F.shape[2], F.shape[3], (o - 1) // 2
        mean = F.mean(0)
        dY, d = F - mean, obs - mean
        Pa = torch.zeros(nX, nY, k, k, dtype=F64, device="cuda")
        wd = torch.zeros(nX, nY, k, dtype=F64, device="cuda")
        ys = torch.arange(nY, device="cuda")
        for i in range(o):
            for j in range(o):
                ix = torch.arange(nX, device="cuda") + (i - r)
                iy = ys + (j - r)
                wall = ((iy >= 0) & (iy < nY)).to(F64)
                Yw, dw, sw = (a[..., ix % nX, :][..., iy % nY] for a in (dY, d, seen))
                L = Z[i, j] * sw * wall / var[:, None, None]
                C = Yw * L
                Pa += torch.einsum("kaxy,laxy->xykl", C, Yw)
                wd += torch.einsum("kaxy,axy->xyk", C, dw)
        Pa += torch.eye(k, dtype=F64, device="cuda") * (k - 1.0) / 1.05
        lam, P = torch.linalg.eigh(Pa.reshape(-1, k, k).cpu())
        lam, P = lam.cuda(), P.cuda()
        Wa = math.sqrt(k - 1.0) * (P / lam.sqrt()[:, None, :]) @ P.transpose(1, 2).contiguous()
        wa = (P / lam[:, None, :]) @ (P.transpose(1, 2).contiguous() @ wd.reshape(-1, k, 1))
        Wa = Wa + wa.transpose(1, 2)
        Xl = dY.permute(2, 3, 0, 1).reshape(nX * nY, k, -1).contiguous()
        An = (Wa @ Xl).reshape(nX, nY, k, -1) + mean.permute(1, 2, 0)[:, :, None, :]
        for a in range(len(group)):
            full = torch.zeros(k, nY + 4, nX + 4, dtype=F64, device="cuda")
            full[:, 2:-2, 2:-2] = An[..., a].permute(2, 1, 0)
            out.append(full)
    return out


def _no_null(v):
    """Per image without its least-squares constant and checkerboard parts."""
    n, h, w = v.shape
    c = 1.0 - 2.0 * ((torch.arange(h)[:, None] + torch.arange(w)[None, :]) % 2).to(v)
    B = torch.stack([torch.ones_like(c).reshape(-1), c.reshape(-1)], 1)
    coef = torch.linalg.solve(B.t() @ B, B.t() @ v.reshape(n, -1).t())
    return v - (B @ coef).t().reshape(n, h, w)


def _exact_train(c, seed):
    """Loss, output and gradients of the network's first step."""
    X, T = (a.double() for a in _train_inputs(c, seed))
    flat = torch.from_numpy(pnn.Network(seed=3).get_params().astype(np.float64)).requires_grad_(True)
    lay, off = [], 0
    for ci, co, _ in _CONV:
        wgt = flat[off:off + 9 * ci * co].reshape(3, 3, ci, co).permute(3, 2, 0, 1)
        lay.append((wgt, flat[off + 9 * ci * co:off + 9 * ci * co + co]))
        off += 9 * ci * co + co
    conv = lambda l, a: torch.nn.functional.conv2d(a, *lay[l], padding=1)
    act = lambda l, a: torch.nn.functional.gelu(conv(l, a))
    up = lambda a: torch.nn.functional.interpolate(a, size=(2 * a.shape[2] - 1, 2 * a.shape[3] - 1), mode="bilinear",
                                                   align_corners=True)
    half = lambda a: a[:, :, ::2, ::2]
    e0 = act(1, act(0, X.permute(0, 3, 1, 2)))
    e1 = act(3, act(2, half(e0)))
    e2 = act(5, act(4, half(e1)))
    d = act(7, act(6, half(e2)))
    for l, skip in ((8, e2), (10, e1), (12, e0)):
        d = act(l + 1, act(l, torch.cat([up(d), skip], 1)))
    z = conv(14, d)[:, 0]
    loss = (_no_null(z) - T).square().mean()
    loss.backward()
    return {"loss": float(loss.detach()), "z": z.detach(), "grads": flat.grad.numpy(), "params": None}


def exact(case, seed):
    c, fam = case, case["family"]
    if fam == "matvec":
        x = _matvec_input(c, seed)
        if c["dtype"] == "f32":
            x = x.astype(np.float32).astype(np.float64)
        A, _ = _exact_op2(c["state"], c["nx"], c["ny"], seed)
        return A(torch.from_numpy(x).to("cuda")).t().contiguous()
    if fam == "solve":
        b, x = _exact_solve(c["state"], c["nx"], c["ny"], seed)
        return {"b": b.t().contiguous(), "x": None if _null_free(c) else x.t().contiguous()}
    if fam == "batch":
        return None if _null_free(c) else [_exact_solve("bubble", nx, ny, seed + 1000 * m)[1].t().contiguous()
                for m, (nx, ny) in enumerate(_batch_sizes(c))]
    if fam in ("solve3d", "projection", "letkf", "train"):
        return globals()["_exact_" + fam](c, seed)
    return None
