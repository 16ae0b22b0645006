"""Performance cases of the reacting-flow step: what users of this framework
run, from one step of a small grid to the headline tube.

A case is a dict of plain values; ``prepare`` builds what a program holds
before the call (solver, states, block grid, cotangents), ``run`` is one pass
through the public entry points and ``exact`` is the same result in plain
64-bit torch, written here from the equations (the mechanism's tables are the
package's parsed data).  Kinds:

* ``step``    one ``Simulator.advance_func`` call (the stepping loop's call)
* ``run``     ``steps`` fused steps on a copy of the initial state
* ``batch``   ``steps`` steps of ``ncase`` uneven cases in one HIP graph
* ``blocks``  one step of a uniform level of same-size AMR blocks
* ``grad``    one differentiable step, forward and backward
* ``rollout`` ``steps`` differentiable steps with checkpoints, forward and
  backward

Every state is a detonation in flight: a wavy front, burnt gas with radicals
behind it, fresh hydrogen-air ahead, a little noise everywhere.
"""
import numpy as np
import torch

from janc_amd import adjoint, cases
from janc_amd.amr import BlockSolver, UniformBlockGrid
from janc_amd.batch import BatchSimulator
from janc_amd.mechanism import Mechanism
from janc_amd.solver import Simulator

DEV = "cuda"
F64 = torch.float64
ATM = 101325.0
CFL = 0.3

# domain: (left, right, bottom, top) boundary kinds and cell size [m]
DOMAINS = {
    # detonation tube (examples and headline benchmark)
    "tube": (("slip_wall", "zero_gradient", "slip_wall", "slip_wall"), 1.25e-5),
    # unrolled rotating-detonation annulus: injector below, outlet above
    "annulus": (("periodic", "periodic", "injection_inlet", "pressure_outlet"), 1e-4),
    # periodic channel with no-slip walls
    "channel": (("periodic", "periodic", "no_slip_wall", "no_slip_wall"), 2.5e-5),
}
THETA = {"Pb": ATM, "P0_inj": 2.0e5, "T0_inj": 300.0}
SCHEMES = {
    "lf": {},
    "hllc": {"solver_type": "godunov", "riemann_solver": "HLLC"},
    "sw": {"split_method": "SW"},
}
# uneven grids of a parameter study
BATCH_SIZES = ((128, 32), (256, 64), (512, 128), (1024, 256))


def _case(name, kind, **kw):
    c = {"name": name, "kind": kind, "domain": "tube", "scheme": "lf", "precision": "fp64",
         "nx": 0, "ny": 0, "steps": 1, "ncase": 0, "nbx": 0, "nby": 0}
    c.update(kw)
    return c


def listed():
    return [
        # a unit test's or a notebook's grid, stepped from a Python loop
        _case("step_fp64_128x32", "step", nx=128, ny=32),
        # an ensemble member or a coarse study, steps fused in one call
        _case("run_mixed_256x64", "run", nx=256, ny=64, steps=20, precision="mixed"),
        # an odd grid with other walls, where tiles are ragged both ways
        _case("step_fp64_channel_333x77", "step", nx=333, ny=77, domain="channel"),
        # the unrolled annulus with injector and outlet, the stepping loop of run()
        _case("step_fp64_annulus_4000x400", "step", nx=4000, ny=400, domain="annulus"),
        # the Godunov scheme on the same domain, a coarser grid
        _case("step_hllc_annulus_1500x300", "step", nx=1500, ny=300, domain="annulus",
              scheme="hllc"),
        # the double-precision tube
        _case("run_fp64_tube_4000x500", "run", nx=4000, ny=500, steps=2),
        # the headline benchmark: the mixed-precision tube of 4M cells
        _case("run_mixed_tube_8000x500", "run", nx=8000, ny=500, steps=4, precision="mixed"),
        # the batched parameter study of the benchmark
        _case("batch_mixed_64", "batch", ncase=64, steps=4, precision="mixed"),
        # one refinement level of small AMR blocks
        _case("blocks_fp64_50x50_of_20x20", "blocks", nbx=50, nby=50, nx=20, ny=20),
        # one refinement level of larger blocks, mixed precision
        _case("blocks_mixed_50x20_of_40x50", "blocks", nbx=50, nby=20, nx=40, ny=50,
              precision="mixed"),
        # gradients through one step (sensitivity analysis, assimilation)
        _case("grad_step_1024x256", "grad", nx=1024, ny=256),
        # gradients through a short checkpointed trajectory
        _case("rollout_256x64", "rollout", nx=256, ny=64, steps=8),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step", "step", "run", "run", "batch", "blocks", "blocks", "grad",
                       "rollout"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "step":
        scheme = rng.choice(["lf", "lf", "hllc", "sw"])
        return _unnamed(kind, nx=_log(rng, 60, 4000), ny=_log(rng, 24, 500), scheme=scheme,
                        domain=rng.choice(sorted(DOMAINS)), precision=prec)
    if kind == "run":
        nx, ny = _log(rng, 100, 8000), _log(rng, 24, 500)
        return _unnamed(kind, nx=nx, ny=ny, steps=max(1, min(20, 4000000 // (nx * ny))),
                        domain=rng.choice(["tube", "channel"]), precision=prec)
    if kind == "batch":
        return _unnamed(kind, ncase=_log(rng, 4, 64), steps=rng.randint(1, 4), precision=prec)
    if kind == "blocks":
        return _unnamed(kind, nbx=_log(rng, 4, 50), nby=_log(rng, 4, 40), nx=_log(rng, 12, 50),
                        ny=_log(rng, 12, 50), precision=prec)
    if kind == "grad":
        return _unnamed(kind, nx=_log(rng, 100, 1024), ny=_log(rng, 24, 256),
                        domain=rng.choice(["tube", "channel"]))
    return _unnamed("rollout", nx=_log(rng, 64, 400), ny=_log(rng, 24, 100),
                    steps=rng.randint(3, 10))


def _unnamed(kind, **kw):
    c = _case("", kind, **kw)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs

_MECH = []


def _mech():
    if not _MECH:
        _MECH.append(Mechanism())
    return _MECH[0]


def _geometry(case):
    kinds, dx = DOMAINS[case["domain"]]
    bc = {s + "_boundary": k for s, k in zip(("left", "right", "bottom", "top"), kinds)}
    return dict(dx=dx, dy=dx, boundary_config=bc)


def _theta(case):
    if case["domain"] != "annulus":
        return None
    return dict(THETA, Yinj=_mech().injection_Y())


def _dt(case):
    """The fixed step of the block and gradient cases."""
    return 0.08 * DOMAINS[case["domain"]][1] / 1000.0


def _config(case, fixed_dt=False):
    return cases.simulation_config(
        _geometry(case), cfl=CFL, dt=_dt(case) if fixed_dt else None, theta=_theta(case),
        precision=case["precision"], flux=SCHEMES[case["scheme"]])


def _field(nx, ny, seed, floor):
    """(U, aux) float64 of a detonation in flight; floor: the least mass
    fraction of a reacting species."""
    m = _mech()
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def rnd(*shape):
        return torch.rand(shape, generator=g, device=DEV, dtype=F64)

    x = torch.arange(nx, device=DEV, dtype=F64)[:, None]
    y = torch.arange(ny, device=DEV, dtype=F64)[None, :] / ny
    r = rnd(12)
    front = nx * (0.25 + 0.4 * r[0] + 0.03 * torch.sin(2 * np.pi * (2 * y + r[1])) +
                  0.01 * torch.sin(2 * np.pi * (5 * y + r[2])))
    b = torch.sigmoid((front - x) / 1.5)               # 1 burnt, 0 fresh
    s = torch.clamp(x / front, 0.0, 1.0)               # 0 at the closed end, 1 at the front
    T = (1 - b) * 300.0 + b * (2300.0 + 600.0 * s + 80.0 * torch.sin(2 * np.pi * (3 * y + r[3])))
    p = ATM * ((1 - b) + b * (8.0 + 10.0 * s))
    u = b * 900.0 * s ** 2 + 3.0 * (2 * rnd(nx, ny) - 1)
    v = b * 60.0 * torch.sin(2 * np.pi * (2 * y + r[4])) + 3.0 * (2 * rnd(nx, ny) - 1)
    T = T * (1 + 0.005 * (2 * rnd(nx, ny) - 1))
    phi = 1 + 0.2 * torch.sin(2 * np.pi * (x / nx + r[5])) * torch.cos(2 * np.pi * (y + r[6]))
    W = torch.as_tensor(m.molecular_weight, device=DEV, dtype=F64)
    fresh = torch.zeros((m.ns, nx, ny), device=DEV, dtype=F64)
    i = m.species.index
    fresh[i("H2")] = 2 * phi * W[i("H2")]
    fresh[i("O2")] = W[i("O2")]
    fresh[i("N2")] = 3.76 * W[i("N2")]
    fresh = fresh / fresh.sum(0)
    burnt = torch.zeros(m.ns, device=DEV, dtype=F64)
    for k, f in (("H2", 4e-3), ("O2", 2e-2), ("OH", 1.5e-2), ("O", 3e-3), ("H", 8e-4),
                 ("H2O", 0.21), ("HO2", 3e-5), ("H2O2", 3e-6)):
        burnt[i(k)] = f
    Y = (1 - b) * fresh[:-1] + b * burnt[:-1, None, None] * (1 + 0.1 * (2 * rnd(m.ns - 1, nx, ny)
                                                                        - 1))
    Y = torch.clamp(Y, min=floor)
    U, aux = adjoint.initial_state(m, T, p, Y, u, v)
    return U.contiguous(), aux.contiguous()


def _dtype(case):
    return torch.float64 if case["precision"] == "fp64" else torch.float32


def _state(case, seed):
    floor = 1e-5 if case["kind"] in ("grad", "rollout") else 0.0
    U, aux = _field(case["nx"], case["ny"], seed, floor)
    return U.to(_dtype(case)), aux.to(_dtype(case))


def _batch_shapes(case):
    r = np.random.default_rng(case["ncase"])
    return [BATCH_SIZES[int(k)] for k in r.integers(0, len(BATCH_SIZES), case["ncase"])]


def _batch_state(case, seed):
    """One buffer that holds every case's U and aux, and the views into it."""
    parts, views, at = [], [], 0
    for k, (nx, ny) in enumerate(_batch_shapes(case)):
        U, aux = _field(nx, ny, seed * 1000 + k, 0.0)
        parts += [U.reshape(-1), aux.reshape(-1)]
        views.append((at, nx, ny))
        at += 14 * nx * ny
    return torch.cat(parts).to(_dtype(case)), views


def _views(flat, views):
    Us, auxs = [], []
    for at, nx, ny in views:
        n = nx * ny
        Us.append(flat[at:at + 12 * n].view(12, nx, ny))
        auxs.append(flat[at + 12 * n:at + 14 * n].view(2, nx, ny))
    return Us, auxs


def _level(case):
    return dict(case, nx=case["nbx"] * case["nx"], ny=case["nby"] * case["ny"])


def _cotangents(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 77)
    cU = torch.randn((12, case["nx"], case["ny"]), generator=g, device=DEV, dtype=F64)
    ca = torch.randn((2, case["nx"], case["ny"]), generator=g, device=DEV, dtype=F64)
    cU[1:3] *= 1e-3                                    # momenta ~1e3
    cU[3] *= 1e-6                                      # energy ~1e6
    ca[1] *= 1e-3                                      # temperature ~1e3
    return cU, ca


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        init, views = _batch_state(case, seed)
        flat = torch.empty_like(init)
        flat.copy_(init)
        Us, auxs = _views(flat, views)
        sim = BatchSimulator([_config(case)] * case["ncase"], Us, auxs)
        return {"kind": kind, "sim": sim, "init": init, "flat": flat, "steps": case["steps"]}
    if kind == "blocks":
        geo = _geometry(case)
        grid = UniformBlockGrid(geo["boundary_config"], case["nbx"], case["nby"], case["nx"],
                                case["ny"], device=DEV)
        blk = grid.split(*_state(_level(case), seed))
        return {"kind": kind, "sim": BlockSolver(_config(case, True)), "grid": grid, "blk": blk,
                "dx": geo["dx"], "dt": _dt(case)}
    U, aux = _state(case, seed)
    st = {"kind": kind, "sim": Simulator(_config(case, kind in ("grad", "rollout"))), "U": U,
          "aux": aux, "steps": case["steps"]}
    if kind in ("grad", "rollout"):
        st["cot"] = _cotangents(case, seed)
        st["dt"] = _dt(case)
        U.requires_grad_(True)
        aux.requires_grad_(True)
    return st


def run(state):
    kind, sim = state["kind"], state["sim"]
    if kind == "step":
        U, aux, _, dt = sim.advance_func(state["U"], state["aux"], 0.0)
        return {"U": U, "aux": aux, "dt": dt}
    if kind == "run":
        U, aux, dt = sim.advance(state["U"].clone(), state["aux"].clone(), state["steps"])
        return {"U": U, "aux": aux, "dt": dt}
    if kind == "batch":
        state["flat"].copy_(state["init"])
        dt = sim.advance(state["steps"], dt_hist=True)
        return {"state": state["flat"], "dt": dt}
    if kind == "blocks":
        grid, blk = state["grid"], state["blk"]
        return {"blk": sim.advance_one_step(1, None, state["dx"], state["dx"], state["dt"], blk,
                                            None, amr=grid)}
    U, aux = state["U"], state["aux"]
    if kind == "grad":
        Uo, ao = adjoint.step(sim, U, aux, state["dt"])
    else:
        Uo, ao = adjoint.rollout(sim, U, aux, state["dt"], state["steps"], 4)
    gU, ga = torch.autograd.grad([Uo, ao], [U, aux], list(state["cot"]))
    return {"U": Uo.detach(), "aux": ao.detach(), "gU": gU, "ga": ga}


# Operations of one cell and step by the algorithm's own count: per RK stage
# 48 WENO5 reconstructions of about 70 operations, the split fluxes, the
# combine and a two-update temperature solve; per step the rates, the
# Jacobian and the solve of an 8 x 8 system.
STAGE_FLOPS, CHEM_FLOPS = 4200.0, 3000.0


def work(case):
    """State read once and written once per step (a step's 14 planes do not
    stay on the chip between steps); a gradient also reads the cotangents,
    the input and the output and writes the gradients, at two forward steps'
    operations."""
    if case["kind"] == "batch":
        cells = sum(nx * ny for nx, ny in _batch_shapes(case))
    else:
        cells = case["nx"] * case["ny"] * max(1, case["nbx"] * case["nby"])
    word = 8 if case["precision"] == "fp64" else 4
    b, f = 28.0 * word, 3 * STAGE_FLOPS + CHEM_FLOPS
    if case["kind"] in ("grad", "rollout"):
        b, f = b + 56.0 * word, 3 * f
    return {"bytes": b * cells * case["steps"], "flops": f * cells * case["steps"]}


# ------------------------------------------------------------------ 64 bits
# The step in plain torch.  Arrays are (variable, group, x, y): a group is a
# block or a batched case, with its own Lax-Friedrichs maxima and dt.

class _Tables:
    def __init__(self):
        m = _mech()

        def t(a):
            return torch.as_tensor(np.asarray(a), device=DEV, dtype=F64)

        self.M, self.Tcr, self.na, self.nrx = t(m.species_M), float(m.Tcr), m.na, m.nrx
        self.cp, self.h = t(m.cp), t(m.h)
        self.hc, self.s, self.logc = t(m.h_chem)[:, :m.na], t(m.s)[:, :m.na], t(m.logc)[:, :m.na]
        self.A, self.B, self.E, self.eff, self.vsum = m.A, m.B, m.EaR, m.eff, m.vsum
        self.vf, self.vb = np.zeros((m.nrx, m.ns)), np.zeros((m.nrx, m.ns))
        for i, r in enumerate(m.reactions):
            for k, c in r.reactants.items():
                self.vf[i, k if isinstance(k, int) else m.species.index(k)] += c
            for k, c in r.products.items():
                self.vb[i, k if isinstance(k, int) else m.species.index(k)] += c
        self.three = [bool(r.three_body) for r in m.reactions]
        self.species = m.species


def _col(c, x):
    return c.reshape((-1,) + (1,) * x.dim())


def _horner(c, x):
    acc = _col(c[:, 0], x) + torch.zeros_like(x)
    for j in range(1, c.shape[1]):
        acc = acc * x + _col(c[:, j], x)
    return acc


def _fill(Y):
    return torch.cat([Y, 1.0 - Y.sum(0, keepdim=True)], 0)


def _gas(t, Y):
    return (_fill(Y) / t.M.reshape(-1, 1, 1, 1)).sum(0)


def _mixture(t, T, Y):
    """cp, dcp/dT, h and R of the mixture at T."""
    Y9, lo = _fill(Y), T < t.Tcr
    cp = torch.where(lo, _horner(t.cp[0], T), _horner(t.cp[1], T))
    h = torch.where(lo, _horner(t.h[0], T), _horner(t.h[1], T))
    d = torch.tensor([4.0, 3.0, 2.0, 1.0], device=DEV, dtype=F64)
    dcp = torch.where(lo, _horner(t.cp[0, :, :4] * d, T), _horner(t.cp[1, :, :4] * d, T))
    return cp, dcp, h, (cp * Y9).sum(0), (dcp * Y9).sum(0), (h * Y9).sum(0), _gas(t, Y)


class _Temperature(torch.autograd.Function):
    """(gamma, T) of internal energy e and Y: Halley iterations from T0 with
    the implicit derivative at the solution (none through T0)."""

    @staticmethod
    def forward(ctx, t, e, Y, T0):
        T = T0
        for _ in range(6):
            _, _, _, cp, dcp, h, R = _mixture(t, T, Y)
            res, d1 = h - R * T - e, cp - R
            T = torch.where(res.abs() > 5e-9, T - 2 * res * d1 / (2 * d1 * d1 - res * dcp), T)
        _, _, _, cp, _, _, R = _mixture(t, T, Y)
        ctx.t = t
        ctx.save_for_backward(Y, T)
        return torch.stack([cp / (cp - R), T])

    @staticmethod
    def backward(ctx, g):
        t = ctx.t
        Y, T = ctx.saved_tensors
        cpk, _, hk, cp, dcp, _, R = _mixture(t, T, Y)
        cv, iM = cp - R, (1.0 / t.M).reshape(-1, 1, 1, 1)
        ek = hk - iM * T
        dgdT = (dcp * cv - dcp * cp) / cv ** 2
        dTdY = (ek[-1:] - ek[:-1]) / cv
        dcpY = cpk[:-1] - cpk[-1:]
        dcvY = dcpY - (iM[:-1] - iM[-1:])
        dgdY = dgdT * dTdY + (dcpY * cv - dcvY * cp) / cv ** 2
        return None, (g[0] * dgdT + g[1]) / cv, g[0] * dgdY + g[1] * dTdY, None


def _update_aux(t, U, aux):
    u, v = U[1] / U[0], U[2] / U[0]
    return _Temperature.apply(t, U[3] / U[0] - 0.5 * (u * u + v * v), U[4:] / U[0], aux[1])


def _index(n):
    """Periodic padding of three cells that repeats neither end cell."""
    return torch.tensor([n - 4, n - 3, n - 2] + list(range(n)) + [1, 2, 3], device=DEV)


def _injector(t, p, P0, T0, Y):
    """Pressure-feedback injector: 20 bisections on the throat Mach number."""
    g, A1, A3 = 1.29, 1.0, 5.0
    A2 = A3 - A1
    R = _gas(t, Y)
    C0 = torch.sqrt(g * R * T0)
    lo, hi = torch.zeros_like(p), torch.ones_like(p)
    for _ in range(20):
        M = 0.5 * (lo + hi)
        f = 1 + (g - 1) / 2 * M ** 2
        P1 = P0 * f ** (-g / (g - 1))
        V1 = M * f ** -0.5 * C0
        flow = A1 * P0 / np.sqrt(T0) * torch.sqrt(g / R) * M * f ** (-(g + 1) / 2 / (g - 1))
        B = g / (g - 1) * p * A3 / flow
        V = -B + torch.sqrt(B ** 2 + 2 * g / (g - 1) * R * T0)
        up = (flow * (V - V1) - P1 * A1 + p * A3) / A2 >= P1
        hi, lo = torch.where(up, M, hi), torch.where(up, lo, M)
    return V, flow / V / A3


def _computed_ghost(t, kind, W, theta, sign):
    """Ghost state of an outlet or injector on a side whose inward normal is
    sign * y, from the wall cells W (14, ...)."""
    rho, u, v, Y = W[0], W[1] / W[0], W[2] / W[0], W[4:12] / W[0]
    R = _gas(t, Y)
    p = rho * R * W[13]
    if kind == "pressure_outlet":
        free = -sign * v / torch.sqrt(W[12] * p / rho) < 1.0
        rho_c = torch.where(free, theta["Pb"] / (p / rho), rho)
        p_c = torch.where(free, torch.full_like(p, theta["Pb"]), p)
        T_c = torch.where(free, p_c / (rho_c * R), W[13])
        _, _, _, cp, _, h, _ = _mixture(t, T_c, Y)
        gam, u_c, v_c, Y_c = cp / (cp - R), u, v, Y
    else:
        Yi = torch.as_tensor(theta["Yinj"], device=DEV, dtype=F64)
        Yi = Yi.reshape((-1,) + (1,) * p.dim()).expand_as(Y)
        Ri = _gas(t, Yi)
        V, rho_m = _injector(t, p, theta["P0_inj"], theta["T0_inj"], Yi)
        T_i = p / (Ri * rho_m)
        _, _, _, cpi, _, hi, _ = _mixture(t, T_i, Yi)
        _, _, _, _, _, hw, _ = _mixture(t, W[13], Y)
        shut = p >= theta["P0_inj"]
        rho_c = torch.where(shut, rho, p / (Ri * T_i))
        u_c, v_c = torch.where(shut, u, torch.zeros_like(u)), torch.where(shut, -v, sign * V)
        T_c, h = torch.where(shut, W[13], T_i), torch.where(shut, hw, hi)
        gam = torch.where(shut, W[12], cpi / (cpi - Ri))
        Y_c, p_c = torch.where(shut, Y, Yi), p
    E = rho_c * h - p_c + 0.5 * rho_c * (u_c ** 2 + v_c ** 2)
    return torch.cat([torch.stack([rho_c, rho_c * u_c, rho_c * v_c, E]), rho_c * Y_c,
                      torch.stack([gam, T_c])])


def _pad(t, U, aux, kinds, theta):
    F = torch.cat([U, aux])
    nx, ny = F.shape[2:]
    P = F.index_select(2, _index(nx)).index_select(3, _index(ny))
    for k, kind in enumerate(kinds):
        if kind == "periodic":
            continue
        ax, low = (2 if k < 2 else 3), k % 2 == 0
        n = F.shape[ax]
        ends = [2, 1, 0] if low else [n - 1, n - 2, n - 3]
        if kind in ("zero_gradient", "no_slip_wall"):
            G = F.index_select(ax, torch.tensor(ends, device=DEV))
        else:
            G = F.index_select(ax, torch.tensor([0 if low else n - 1] * 3, device=DEV))
        sign = torch.ones((14, 1, 1, 1), device=DEV, dtype=F64)
        if kind == "slip_wall":
            sign[1 if ax == 2 else 2] = -1.0
        if kind == "no_slip_wall":
            sign[1:3] = -1.0
        if kind in ("pressure_outlet", "injection_inlet"):
            G = _computed_ghost(t, kind, G, theta, 1.0 if low else -1.0)
        at = slice(0, 3) if low else slice(-3, None)
        P = P.clone()
        if ax == 2:
            P[:, :, at, 3:-3] = G * sign
        else:
            P[:, :, 3:-3, at] = G * sign
    return P[:12], P[12:]


def _primitive(t, U, aux):
    rho, u, v, Y = U[0], U[1] / U[0], U[2] / U[0], U[4:] / U[0]
    p = rho * _gas(t, Y) * aux[1]
    return rho, u, v, Y, p, torch.sqrt(aux[0] * p / rho)


def _weno(a, b, c, d, e):
    i1 = 0.25 * (a - 4 * b + 3 * c) ** 2 + 13 / 12 * (a - 2 * b + c) ** 2
    i2 = 0.25 * (b - d) ** 2 + 13 / 12 * (b - 2 * c + d) ** 2
    i3 = 0.25 * (3 * c - 4 * d + e) ** 2 + 13 / 12 * (c - 2 * d + e) ** 2
    w1, w2, w3 = 0.1 / (1e-6 + i1) ** 2, 0.6 / (1e-6 + i2) ** 2, 0.3 / (1e-6 + i3) ** 2
    return (w1 * (2 * a - 7 * b + 11 * c) + w2 * (-b + 5 * c + 2 * d) +
            w3 * (2 * c + 5 * d - e)) / (6 * (w1 + w2 + w3))


def _faces(Q, ax, left):
    """Face values along ax of the padded Q, from the left or the right."""
    Q = Q[..., 3:-3] if ax == 2 else Q[:, :, 3:-3]
    n = Q.shape[ax] - 5
    f = [Q.narrow(ax, k, n) for k in range(6)]
    return _weno(*f[:5]) if left else _weno(*f[:0:-1])


def _flux(ax, rho, u, v, Y, p, E):
    un = u if ax == 2 else v
    one, zero = (p, torch.zeros_like(p)) if ax == 2 else (torch.zeros_like(p), p)
    return torch.cat([torch.stack([rho * un, rho * u * un + one, rho * v * un + zero,
                                   un * (E + p)]), rho * un * Y])


def _hllc(t, ax, L, R):
    side = []
    for q in (L, R):
        rho, u, v, p, Y = q[0], q[1], q[2], q[3], q[4:]
        Rg = _gas(t, Y)
        T = p / (Rg * rho)
        _, _, _, cp, _, h, _ = _mixture(t, T, Y)
        a = torch.sqrt(cp / (cp - Rg) * p / rho)
        E = rho * h - p + 0.5 * rho * (u * u + v * v)
        side.append((rho, u, v, p, Y, a, E, u if ax == 2 else v))
    (rL, _, _, pL, _, aL, _, nL), (rR, _, _, pR, _, aR, _, nR) = side
    sL, sR = torch.minimum(nL - aL, nR - aR), torch.maximum(nL + aL, nR + aR)
    sM = (pR - pL + rL * nL * (sL - nL) - rR * nR * (sR - nR)) / \
        (rL * (sL - nL) - rR * (sR - nR))
    out = []
    for (rho, u, v, p, Y, a, E, n), s in zip(side, (sL, sR)):
        U = torch.cat([torch.stack([rho, rho * u, rho * v, E]), rho * Y])
        F = _flux(ax, rho, u, v, Y, p, E)
        star = torch.cat([torch.stack([torch.ones_like(sM), sM if ax == 2 else u,
                                       v if ax == 2 else sM,
                                       E / rho + (sM - n) * (sM + p / (rho * (s - n)))]), Y])
        out.append((F, F + s * (rho * (s - n) / (s - sM) * star - U)))
    (FL, ML), (FR, MR) = out
    F = torch.where((sL <= 0) & (sM >= 0), ML, torch.where(sL >= 0, FL, FR))
    return torch.where((sM <= 0) & (sR >= 0), MR, F)


def _steger_warming(ax, U, aux, rho, u, v, Y, p, a):
    """The two split fluxes along ax."""
    g, un, z = aux[0], (u if ax == 2 else v), torch.zeros_like(p)
    da = rho * a
    x, y = (da, z) if ax == 2 else (z, da)
    h1 = torch.cat([torch.stack([rho, rho * u - x, rho * v - y, U[3] + p - da * un]), rho * Y])
    h4 = torch.cat([torch.stack([rho, rho * u + x, rho * v + y, U[3] + p + da * un]), rho * Y])
    h2 = torch.cat([torch.stack([rho, rho * u, rho * v, 0.5 * rho * (u * u + v * v)]), rho * Y])
    out = []
    for sg in (1.0, -1.0):
        lam = [0.5 * (w + sg * torch.sqrt(w * w + 1e-12)) for w in (un - a, un, un + a)]
        out.append(lam[0] / (2 * g) * h1 + lam[1] * (g - 1) / g * h2 + lam[2] / (2 * g) * h4)
    return out


def _rhs(t, U, aux, dx, scheme):
    """-(dF/dx + dG/dy) of the padded state."""
    rho, u, v, Y, p, a = _primitive(t, U, aux)
    total = 0.0
    for ax, un in ((2, u), (3, v)):
        if scheme == "hllc":
            q = torch.cat([torch.stack([rho, u, v, p]), Y])
            F = _hllc(t, ax, _faces(q, ax, True), _faces(q, ax, False))
        elif scheme == "sw":
            hp, hm = _steger_warming(ax, U, aux, rho, u, v, Y, p, a)
            F = _faces(hp, ax, True) + _faces(hm, ax, False)
        else:
            s = un.abs() + a
            s = torch.where(torch.isnan(s), torch.zeros_like(s), s)
            alpha = torch.amax(s, dim=(-2, -1), keepdim=True)
            F = _flux(ax, rho, u, v, Y, p, U[3])
            F = _faces(0.5 * (F + alpha * U), ax, True) + _faces(0.5 * (F - alpha * U), ax, False)
        total = total + torch.diff(F, dim=ax) / dx
    return -total


def _solve(A, b):
    """x of A x = b by elimination with partial pivoting; A (n, n, ...)."""
    n = A.shape[0]
    M = torch.cat([A, b[:, None]], 1)
    rows = []
    for c in range(n):
        k = M[:, 0].abs().argmax(0)
        pick = k.reshape((1, 1) + k.shape).expand((1,) + M.shape[1:])
        top = M.gather(0, pick)
        if M.shape[0] > 1:
            first = M[:1].expand_as(M)
            at = torch.arange(M.shape[0], device=DEV).reshape((-1,) + (1,) * (M.dim() - 1))
            M = torch.where(at == k, first, M)[1:]
            M = M[:, 1:] - M[:, :1] / top[:, :1] * top[:, 1:]
        rows.append(top[0])
    x = []
    for c in range(n - 1, -1, -1):
        r = rows[c]
        s = r[-1]
        for j, xj in enumerate(x[::-1]):
            s = s - r[1 + j] * xj
        x.append(s / r[0])
    return torch.stack(x[::-1])


def _chemistry(t, U, aux, dt):
    """Increment of rho Y by the point-implicit rates."""
    na, T = t.na, aux[1]
    Y = _fill(U[4:] / U[0])
    X = U[0] * Y / t.M.reshape(-1, 1, 1, 1)
    Xc = torch.maximum(X[:na], torch.full_like(X[:na], 1e-50))
    lT, lX, lo = torch.log(T), torch.log(Xc), T < t.Tcr
    h = torch.where(lo, _horner(t.hc[0], T), _horner(t.hc[1], T))
    s = torch.where(lo, _horner(t.s[0], T) + _col(t.logc[0], T) * lT,
                    _horner(t.s[1], T) + _col(t.logc[1], T) * lT)
    g = s - h / T
    w = [torch.zeros_like(T) for _ in range(na)]
    J = [[torch.zeros_like(T) for _ in range(na)] for _ in range(na)]
    M = t.M.tolist()
    for i in range(t.nrx):
        vf, vb, eff = t.vf[i], t.vb[i], t.eff[i]
        k = t.A[i] * torch.exp(t.B[i] * lT - t.E[i] / T)
        body = sum(eff[n] * X[n] for n in range(len(eff))) if t.three[i] else torch.ones_like(T)
        kf = k * torch.exp(sum((vf[n] * lX[n] for n in range(na) if vf[n]), torch.zeros_like(T)))
        kb = k * torch.exp(sum((vb[n] * lX[n] for n in range(na) if vb[n]), torch.zeros_like(T))
                           - sum((vb[n] - vf[n]) * g[n] for n in range(na) if vb[n] != vf[n])) / \
            (ATM / T) ** t.vsum[i]
        q = kf - kb
        d = []
        for n in range(na):
            v = q * (eff[n] / M[n]) if t.three[i] and eff[n] else None
            if vf[n] or vb[n]:
                z = body * (vf[n] * kf - vb[n] * kb) / (M[n] * Xc[n])
                v = z if v is None else v + z
            d.append(v)
        for n in range(na):
            if vb[n] != vf[n]:
                w[n] = w[n] + (vb[n] - vf[n]) * M[n] * body * q
                for c in range(na):
                    if d[c] is not None:
                        J[n][c] = J[n][c] + (vb[n] - vf[n]) * M[n] * d[c]
    J = torch.stack([torch.stack(r) for r in J])
    eye = torch.eye(na, device=DEV, dtype=F64).reshape((na, na) + (1,) * T.dim())
    dY = _solve(eye / dt - J, torch.stack(w)) / U[0]
    return U[0] * torch.minimum(torch.maximum(dY, -Y[:na]), 1 - Y[:na])


def _react(t, U, aux, dt):
    """Chemistry of every group and the temperature after it, in slabs of x
    (the elimination holds some 200 planes)."""
    if U.requires_grad:
        V = torch.cat([U[:4], U[4:] + _chemistry(t, U, aux, dt)])
    else:
        nx = U.shape[2]
        step = max(1, 1000000 // (U.shape[1] * U.shape[3]))
        V = torch.cat([torch.cat([U[:4, :, i:i + step], U[4:, :, i:i + step] +
                                  _chemistry(t, U[:, :, i:i + step], aux[:, :, i:i + step], dt)])
                       for i in range(0, nx, step)], 2)
    return V, _update_aux(t, V, aux)


def _courant(t, U, aux, dx):
    _, u, v, _, _, a = _primitive(t, U, aux)
    return CFL / torch.amax((u.abs() + a) / dx + (v.abs() + a) / dx, dim=(-2, -1), keepdim=True)


def _step64(t, U, aux, dt, dx, scheme, pad):
    def rhs(V, b):
        return dt * _rhs(t, *pad(V, b), dx, scheme)
    U1 = U + rhs(U, aux)
    a1 = _update_aux(t, U1, aux)
    U2 = 0.75 * U + 0.25 * (U1 + rhs(U1, a1))
    a2 = _update_aux(t, U2, a1)
    U3 = U / 3 + 2 / 3 * (U2 + rhs(U2, a2))
    return _react(t, U3, _update_aux(t, U3, a2), dt)


def _padder(t, case):
    kinds, th = DOMAINS[case["domain"]][0], _theta(case)
    return lambda U, aux: _pad(t, U, aux, kinds, th)


def exact(case, seed):
    t, kind, dx = _Tables(), case["kind"], DOMAINS[case["domain"]][1]
    pad = _padder(t, case)
    if kind in ("step", "run"):
        U, aux = (v.to(F64)[:, None] for v in _state(case, seed))
        hist = []
        for _ in range(case["steps"]):
            dt = _courant(t, U, aux, dx)
            U, aux = _step64(t, U, aux, dt, dx, case["scheme"], pad)
            hist.append(dt.reshape(-1))
        dts = torch.cat(hist)
        return {"U": U[:, 0], "aux": aux[:, 0], "dt": dts[0] if kind == "step" else dts}
    if kind == "batch":
        flat, views = _batch_state(case, seed)
        flat = flat.to(F64)
        out = torch.zeros_like(flat)
        dts = torch.zeros((case["ncase"], case["steps"]), device=DEV, dtype=F64)
        for shape in BATCH_SIZES:                      # cases of one size together
            ids = [k for k, v in enumerate(views) if v[1:] == shape]
            if not ids:
                continue
            Us, auxs = _views(flat, [views[k] for k in ids])
            U, aux = torch.stack(Us, 1), torch.stack(auxs, 1)
            for s in range(case["steps"]):
                dt = _courant(t, U, aux, dx)
                dts[ids, s] = dt.reshape(-1)
                U, aux = _step64(t, U, aux, dt, dx, "lf", pad)
            oU, oa = _views(out, [views[k] for k in ids])
            for j in range(len(ids)):
                oU[j].copy_(U[:, j])
                oa[j].copy_(aux[:, j])
        return {"state": out, "dt": dts}
    if kind == "blocks":
        lev = _level(case)
        nx, ny, nbx, nby = case["nx"], case["ny"], case["nbx"], case["nby"]

        def split(F):
            b = F[:, 0].reshape(-1, nbx, nx, nby, ny).permute(0, 1, 3, 2, 4)
            return b.reshape(-1, nbx * nby, nx, ny)

        def join(F):
            b = F.reshape(-1, nbx, nby, nx, ny).permute(0, 1, 3, 2, 4)
            return b.reshape(-1, 1, nbx * nx, nby * ny)

        def blocks(U, aux):                            # padded level -> padded blocks
            P = torch.cat(pad(join(U), join(aux)))[:, 0]
            b = P.unfold(1, nx + 6, nx).unfold(2, ny + 6, ny)
            b = b.reshape(14, nbx * nby, nx + 6, ny + 6)
            return b[:12], b[12:]

        U, aux = (split(v.to(F64)[:, None]) for v in _state(lev, seed))
        U, aux = _step64(t, U, aux, _dt(case), dx, "lf", blocks)
        return {"blk": torch.cat([U, aux]).permute(1, 0, 2, 3)}
    U, aux = (v.requires_grad_(True) for v in _state(case, seed))
    V, b = U[:, None], aux[:, None]
    for _ in range(case["steps"]):
        V, b = _step64(t, V, b, _dt(case), dx, "lf", pad)
    gU, ga = torch.autograd.grad([V, b], [U, aux], [c[:, None] for c in _cotangents(case, seed)])
    return {"U": V[:, 0].detach(), "aux": b[:, 0].detach(), "gU": gU, "ga": ga}
