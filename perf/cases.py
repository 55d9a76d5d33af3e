"""The workloads by which this package's speed is measured.

What a user of the package has it do, through its public calls:

  step       one timestep! of a spun-up channel run (a host loop that looks at
             the fields after every step): the smallest call
  transient  run_simulation! of the 80 x 10 channel over many steps
  state      update_state! on an irregular domain of odd sizes (a calving
             front, holes, interior Dirichlet points)
  solve      one update_velocities! of the channel, 20 Picard iterations (the
             package's benchmark; fewer on the finest grid)
  gradient   misfit_gradient: the misfit and its gradient with respect to
             log C, the step of an inversion
  batch      update_velocities! of an ensemble of small members in one call

in both precisions of the solver ("fp64" and "mixed"), from 37 x 22 to
2560 x 320 cells.  Host arrays go in and come out, as the model's fields are
host arrays; a pass starts from the same fields every time.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its folder's name holds a dot, so it is loaded by path)."""
    if "wavi_jl_amd" not in sys.modules:
        folder = os.path.join(ROOT, "wavi.jl_amd")
        spec = importlib.util.spec_from_file_location("wavi_jl_amd", os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["wavi_jl_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["wavi_jl_amd"]


W = _package()


def listed():
    return [
        # a host loop that steps the 80 x 10 channel one call at a time
        {"name": "step_80x10_fp64", "kind": "step", "nx": 80, "ny": 10, "ns": 4, "precision": "fp64"},
        # the 80 x 10 channel transient of the package's benchmark, 200 steps
        {"name": "transient_80x10_fp64", "kind": "transient", "nx": 80, "ny": 10, "ns": 4, "precision": "fp64",
         "steps": 200},
        {"name": "transient_80x10_mixed", "kind": "transient", "nx": 80, "ny": 10, "ns": 4, "precision": "mixed",
         "steps": 200},
        # one state update of a regional model: odd sizes, irregular front, holes
        {"name": "state_61x37_fp64", "kind": "state", "nx": 61, "ny": 37, "ns": 5, "precision": "fp64", "picard": 6},
        # ensemble-member sized solves
        {"name": "solve_320x40_fp64", "kind": "solve", "nx": 320, "ny": 40, "ns": 8, "precision": "fp64",
         "picard": 20},
        {"name": "solve_640x80_mixed", "kind": "solve", "nx": 640, "ny": 80, "ns": 8, "precision": "mixed",
         "picard": 20},
        # the package's benchmark solve at 500 m, in both precisions
        {"name": "solve_1280x160_fp64", "kind": "solve", "nx": 1280, "ny": 160, "ns": 8, "precision": "fp64",
         "picard": 20},
        {"name": "solve_1280x160_mixed", "kind": "solve", "nx": 1280, "ny": 160, "ns": 8, "precision": "mixed",
         "picard": 20},
        # the finest grid (250 m), a few Picard iterations from a cold start
        {"name": "solve_2560x320_mixed", "kind": "solve", "nx": 2560, "ny": 320, "ns": 8, "precision": "mixed",
         "picard": 5},
        # an inversion's gradient: a coarse regional one and one at 500 m
        {"name": "gradient_64x16_fp64", "kind": "gradient", "nx": 64, "ny": 16, "ns": 4, "precision": "fp64",
         "picard": 5},
        {"name": "gradient_1280x160_mixed", "kind": "gradient", "nx": 1280, "ny": 160, "ns": 8,
         "precision": "mixed", "picard": 5},
        # an ensemble of small members (perturbed physics, coarse grids)
        {"name": "batch_16_160x20_mixed", "kind": "batch", "nx": 160, "ny": 20, "ns": 4, "precision": "mixed",
         "picard": 10, "members": 16},
    ]


def draw(rng):
    """One more case: a kind, a precision, and a grid whose cell count spans
    the kind's range evenly in its logarithm, about four to ten times as long
    as wide, odd sizes included; the Picard count is cut where the grid is
    large, so that no case costs more than the largest listed one."""
    kind = rng.choice(["step", "transient", "state", "solve", "solve", "solve", "gradient", "gradient", "batch"])
    lo, hi = {"step": (400, 20000), "transient": (400, 13000), "state": (800, 50000), "solve": (2000, 800000),
              "gradient": (800, 200000), "batch": (800, 13000)}[kind]
    cells = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    aspect = rng.uniform(3.0, 9.0) if kind != "state" else rng.uniform(1.2, 2.5)
    ny = max(10, int(round(math.sqrt(cells / aspect))))
    nx = max(24, int(round(cells / ny)))
    case = {"kind": kind, "nx": nx, "ny": ny, "ns": rng.choice([4, 5, 8]), "precision": rng.choice(["fp64", "mixed"])}
    if kind == "transient":
        case["steps"] = max(4, min(200, int(200 * 800 / (nx * ny))))
    elif kind == "state":
        case["picard"] = rng.randint(2, 8)
    elif kind == "solve":
        case["picard"] = max(2, min(20, int(1.5e6 / (nx * ny)) + rng.randint(0, 2)))
    elif kind == "gradient":
        case["picard"] = rng.randint(2, 5) if nx * ny > 20000 else rng.randint(3, 8)
    elif kind == "batch":
        case["members"] = rng.randint(3, 16)
        case["picard"] = rng.randint(4, 10)
        case["precision"] = "mixed" if rng.random() < 0.7 else "fp64"
    return case


# ---------------------------------------------------------------------------
# inputs


def _channel_run(case, seed):
    """The channel of the transient workload at the case's grid."""
    m = W.workloads.channel_transient(precision=case["precision"], seed=seed, nx=case["nx"], ny=case["ny"])
    if case["ns"] != 4:
        g = m.grid
        grid = W.Grid(nx=g.nx, ny=g.ny, nσ=case["ns"], x0=0.0, y0=-40000.0, dx=g.dx, dy=g.dy, u_iszero=["north"],
                      v_iszero=["west", "east"])
        m = W.Model(grid=grid, bed_elevation=m.fields.gh.b, params=m.params, solver_params=m.solver_params,
                    parallel_spec=W.HIPSpec(case["precision"]))
    return m


def _irregular(case, seed):
    """An irregular domain: a front that moves in steps of two rows, holes
    that keep apart, grounded upstream and floating downstream, and interior
    Dirichlet points (a tributary's inflow)."""
    nx, ny, rng = case["nx"], case["ny"], np.random.default_rng(seed)
    dx = dy = 4000.0
    h_mask = np.ones((nx, ny), bool)
    front = np.repeat(nx - 2 - rng.integers(0, max(nx // 5, 2), (ny + 1) // 2), 2)[:ny]
    for j in range(ny):
        h_mask[front[j]:, j] = False
    holes = []
    for _ in range(200):
        i, j = int(rng.integers(nx // 5, nx // 2)), int(rng.integers(2, ny - 4))
        if all(abs(i - a) > 3 or abs(j - b) > 3 for a, b in holes):
            holes.append((i, j))
            h_mask[i:i + 2, j:j + 2] = False
        if len(holes) == 3:
            break
    u_isfixed = np.zeros((nx + 1, ny), bool)
    u_isfixed[nx // 4, 1:4] = True
    grid = W.Grid(nx=nx, ny=ny, nσ=case["ns"], x0=0.0, y0=-ny * dy / 2, dx=dx, dy=dy, h_mask=h_mask,
                  u_iszero=["north"], v_iszero=["west", "east"], u_isfixed=u_isfixed)
    x = grid.xxh
    bed = 150.0 - 900.0 * x / (nx * dx) + rng.normal(0.0, 10.0, x.shape)
    thick = np.where(h_mask, np.maximum(1200.0 * (1.0 - 0.8 * x / (nx * dx)), 50.0) + rng.normal(0.0, 5.0, x.shape), 0.0)
    u0 = np.zeros((nx + 1, ny))
    u0[u_isfixed] = 80.0
    return W.Model(grid=grid, bed_elevation=np.asfortranarray(bed),
                   params=W.Params(default_temperature=265.700709, accumulation_rate=0.3),
                   solver_params=W.SolverParams(maxiter_picard=case["picard"]),
                   initial_conditions=W.InitialConditions(initial_thickness=np.asfortranarray(thick),
                                                          initial_u_veloc=u0),
                   parallel_spec=W.HIPSpec(case["precision"]))


def _channel(case, seed, member=0):
    nx, ny = case["nx"], case["ny"]
    c, a_ref = 1e4, None
    if case["kind"] == "batch":  # perturbed drag and rate factor, as an ensemble has them
        rng = np.random.default_rng(1000 * seed + member)
        c = np.asfortranarray(1e4 * np.exp(W.workloads.gaussian_random_field(nx, ny, 640000.0 / nx, 80000.0 / ny, 0.3,
                                                                              10000.0, seed=[seed, member])))
        a_ref = W.Params().glen_a_ref * float(np.exp(rng.uniform(np.log(0.5), np.log(2.0))))
    elif case["kind"] == "gradient":  # an iterate of the inversion, away from the prior
        c = np.asfortranarray(1e4 * np.exp(W.workloads.gaussian_random_field(nx, ny, 640000.0 / nx, 80000.0 / ny, 0.2,
                                                                              10000.0, seed=[seed, 1])))
    return W.workloads.channel_solve(nx=nx, ny=ny, precision=case["precision"], seed=100 * seed + member, nσ=case["ns"],
                                     maxiter_picard=case["picard"], weertman_c=c, glen_a_ref=a_ref)


def _observed(m, seed):
    """Observed velocities: a plausible channel flow with noise."""
    rng = np.random.default_rng([seed, 2])
    g = m.grid
    x = g.xxu / 640000.0
    u = 900.0 * x ** 2 * np.cos(np.pi * g.yyu / 100000.0) * (1 + 0.01 * rng.standard_normal(x.shape))
    v = 5.0 * np.sin(np.pi * g.yyv / 40000.0) * (1 + 0.01 * rng.standard_normal(g.yyv.shape))
    return np.asfortranarray(u), np.asfortranarray(v)


STEP_DT = 0.5   # a
SPIN_UP = 10    # steps before the single step that is measured


def _fields_of(m):
    return [(c, a, m._array(c, a)) for c, a, _ in W.model.FIELD_MAP]


def _reset(m, start):
    """The model's fields as they were: a call replaces the arrays of the
    fields, so putting the first ones back costs nothing."""
    for c, a, v in start:
        setattr(m.params if c == "params" else getattr(m.fields, c), a, v)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("step", "transient"):
        m = _channel_run(case, seed)
        steps = case["steps"] if kind == "transient" else SPIN_UP + 1
        s["sim"] = W.Simulation(model=m, timestepping_params=W.TimesteppingParams(dt=STEP_DT, n_iter_total=steps))
        if kind == "step":
            for _ in range(SPIN_UP):
                W.timestep(s["sim"])
        s["models"] = [m]
    elif kind == "state":
        s["models"] = [_irregular(case, seed)]
    else:
        s["models"] = [_channel(case, seed, k) for k in range(case.get("members", 1))]
        for m in s["models"]:
            W.update_geometry(m)
        if kind == "gradient":
            s["obs"] = _observed(s["models"][0], seed)
            s["picard"] = case["picard"]
    for m in s["models"]:
        W.update_preconditioner(m)  # the device context, which a program keeps with its model
    s["start"] = [_fields_of(m) for m in s["models"]]
    if "sim" in s:
        s["clock"] = (s["sim"].clock.n_iter, s["sim"].clock.time)
    return s


def _solved(m):
    f = m.fields
    return {"u": f.gu.u, "v": f.gv.v, "resid_u": f.gu.residual, "resid_v": f.gv.residual, "eta": f.g3d.η,
            "eta_av": f.gh.ηav, "beta": f.gh.β, "quad_f2": f.gh.quad_f2}


def _stepped(m):
    f = m.fields
    return {"h": f.gh.h, "s": f.gh.s, "dhdt": f.gh.dhdt, "gf": f.gh.grounded_fraction, "us": f.gh.us,
            "ub": f.gh.ub, **_solved(m)}


def run(state):
    kind = state["kind"]
    for m, start in zip(state["models"], state["start"]):
        _reset(m, start)
    m = state["models"][0]
    if kind == "step" or kind == "transient":
        sim = state["sim"]
        sim.clock.n_iter, sim.clock.time = state["clock"]
        if kind == "step":
            W.timestep(sim)
        else:
            W.run_simulation(sim)
        return _stepped(m)
    if kind == "state":
        W.update_state(m)
        return _stepped(m)
    if kind == "solve":
        W.update_velocities(m)
        return _solved(m)
    if kind == "gradient":
        J, grad, _ = W.misfit_gradient(m, state["picard"], *state["obs"])
        return {"J": J, "grad": grad, "u": m.fields.gu.u, "v": m.fields.gv.v}
    W.update_velocities_batch(state["models"])
    return [{"u": k.fields.gu.u, "v": k.fields.gv.v, "eta_av": k.fields.gh.ηav} for k in state["models"]]


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    """bytes: the fields in and out once.  flops: the coarse CG's iterations
    (1000, the cap, where a solve's tolerance is 1e-8; about 6 in a time
    step), each one operator application, two Haar transforms and the
    vector updates, the smoother's sweeps and the viscosity update."""
    n = case["nx"] * case["ny"]
    unknowns = 2 * n
    fields = 8.0 * n * (2 * 43 + 3 * case["ns"])
    cycle = unknowns * 10 * 45.0 + n * case["ns"] * 2 * 150.0
    per_iter = unknowns * 85.0
    kind = case["kind"]
    cg = {"step": 6, "transient": 6, "state": 200, "solve": 1000, "batch": 600, "gradient": 2500}[kind]
    cycles = case.get("steps", 1) * case.get("picard", 1) * case.get("members", 1) * (2 if kind == "gradient" else 1)
    return {"bytes": fields * case.get("members", 1), "flops": cycles * (cycle + cg * per_iter)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch on the CPU


class _Plain:
    """WAVI's state update, velocity solve and time step on one model's
    arrays, written with whole-array operations on (nx, ny) tensors."""

    def __init__(self, m):
        t = lambda a: torch.tensor(np.array(a, dtype=np.float64))
        g, p, s, f = m.grid, m.params, m.solver_params, m.fields
        self.nx, self.ny, self.ns, self.p, self.s = g.nx, g.ny, g.nσ, p, s
        self.rdx, self.rdy = 1.0 / g.dx, 1.0 / g.dy
        self.zeta, self.qw = [float(z) for z in g.ζ], [float(q) for q in g.quadrature_weights]
        self.hm, self.um, self.vm, self.cm = t(f.gh.mask), t(f.gu.mask), t(f.gv.mask), t(f.gc.mask)
        self.ui, self.vi = t(f.gu.mask_inner), t(f.gv.mask_inner)
        self.ufix, self.vfix = t(g.u_isfixed), t(g.v_isfixed)
        self.hfix = t(g.h_isfixed)
        self.melt = m.melt_rate.m
        self.C, self.acc_param = t(p.weertman_c), t(p.accumulation_rate)
        self.b, self.h, self.glen_b = t(f.gh.b), t(f.gh.h), t(f.g3d.glen_b)
        self.u, self.v, self.eta = t(f.gu.u), t(f.gv.v), t(f.g3d.η)
        self.beta, self.f2, self.etaav = t(f.gh.β), t(f.gh.quad_f2), t(f.gh.ηav)
        self.sur, self.hu, self.su = t(f.gh.s), t(f.gu.h), t(f.gu.s)
        self.hv, self.sv, self.dhdt = t(f.gv.h), t(f.gv.s), t(f.gh.dhdt)
        self.mw = [torch.ones(self.nx + 1, self.ny), torch.ones(self.nx, self.ny + 1)]
        self.mw = [a.double() for a in self.mw]
        self.xc = [torch.zeros_like(a) for a in self.mw]
        self.resid = [torch.zeros_like(a) for a in self.mw]
        self.haar = [(self._haar(n, False), self._haar(n, True)) for n in (self.nx, self.nx + 1, self.ny, self.ny + 1)]
        self.P = {n: h[0] for n, h in zip((self.nx, self.nx + 1, self.ny, self.ny + 1), self.haar)}
        self.F = {n: h[1] for n, h in zip((self.nx, self.nx + 1, self.ny, self.ny + 1), self.haar)}
        self.colour = []
        for n, k in ((self.nx + 1, self.ny), (self.nx, self.ny + 1)):
            par = (torch.arange(n)[:, None] - torch.arange(k)[None, :]) % 2
            self.colour += [(par == 0).double(), (par == 1).double()]

    def _haar(self, n, forward):
        """wavelet_matrix: the composed lifting steps as a matrix."""
        M, step = torch.eye(n, dtype=torch.float64), 1
        for _ in range(self.s.levels + 1):
            step *= 2
            o = torch.arange(0, n, step)
            o = o[o + step // 2 < n]
            e = o + step // 2
            if forward:
                a, b = M[o].clone(), M[e].clone()
                M[o], M[e] = 0.5 * (a + b), 0.5 * (b - a)
            else:
                a, b = M[:, o].clone(), M[:, e].clone()
                M[:, o], M[:, e] = b + a, b - a
        return M

    # -- differences and averages between the grids (absent neighbours are zero)
    @staticmethod
    def _pad(a, dim):
        z = torch.zeros_like(a.narrow(dim, 0, 1))
        return torch.cat([z, a, z], dim)

    def _diff(self, a, dim, rd):
        """Differences: from faces to cells where a has one more entry."""
        return rd * (a.narrow(dim, 1, a.shape[dim] - 1) - a.narrow(dim, 0, a.shape[dim] - 1))

    def _mean(self, a, dim):
        return 0.5 * (a.narrow(dim, 1, a.shape[dim] - 1) + a.narrow(dim, 0, a.shape[dim] - 1))

    def _to_faces(self, a, dim, mask):
        """Mean over the masked cells of a face, zero off `mask`."""
        num, den = self._mean(self._pad(self.hm * a, dim), dim), self._mean(self._pad(self.hm, dim), dim)
        return torch.where(mask > 0, num / torch.where(den > 0, den, torch.ones_like(den)), torch.zeros_like(num))

    # -- update_state! before the solve
    def geometry(self):
        p = self.p
        ri, rw, sl = p.density_ice, p.density_ocean, p.sea_level_wrt_geoid
        on = self.hm > 0
        self.sur = torch.where(on, torch.maximum(self.b + self.h, sl + self.h * (1.0 - ri / rw)), self.sur)
        for dim, (hf, sf, mask) in enumerate((("hu", "su", self.um), ("hv", "sv", self.vm))):
            setattr(self, hf, torch.where(mask > 0, self._to_faces(self.h, dim, mask), getattr(self, hf)))
            setattr(self, sf, torch.where(mask > 0, self._to_faces(self.sur, dim, mask), getattr(self, sf)))
        haf = self.h - (rw / ri) * (sl - self.b)
        q = self._quadrants(haf)
        self.gf = 0.25 * (q[0] + q[1] + q[2] + q[3])
        left, right = self._pad(0.25 * (q[0] + q[3]), 0), self._pad(0.25 * (q[1] + q[2]), 0)
        self.gfu = left[:-1] + right[1:]
        low, high = self._pad(0.25 * (q[0] + q[1]), 1), self._pad(0.25 * (q[2] + q[3]), 1)
        self.gfv = low[:, :-1] + high[:, 1:]
        self.acc, self.mel = self.acc_param.clone(), torch.full_like(self.h, self.melt)
        self.wc = self.C * self.gf
        self.dsdh = (1.0 - ri / rw) + (ri / rw) * self.gf

    def _quadrants(self, z):
        """Grounded area of a cell's four quadrants: the part of the triangle
        of the cell and two neighbours on which the plane through them is
        positive, as pos_fraction lays it out."""
        nb = {}
        for name, dim, by in (("E", 0, 1), ("W", 0, -1), ("N", 1, 1), ("S", 1, -1)):
            idx = torch.clamp(torch.arange(z.shape[dim]) + by, 0, z.shape[dim] - 1)
            zn, mn = z.index_select(dim, idx), self.hm.index_select(dim, idx)
            nb[name] = torch.where(mn > 0, zn, z)
        out = []
        for a, b in (("E", "N"), ("N", "W"), ("W", "S"), ("S", "E")):
            v1, v2, v3 = z, nb[a], nb[b]
            same = (torch.sign(v1) == torch.sign(v2)) & (torch.sign(v1) == torch.sign(v3))
            flip = (v3 - v1).abs() < (v2 - v1).abs()
            d_hi, d_lo = torch.where(flip, v2 - v1, v3 - v1), torch.where(flip, v3 - v1, v2 - v1)
            d_hi = torch.where(same | (d_hi == 0), torch.ones_like(d_hi), d_hi)
            al, be = -d_lo / d_hi, -2.0 * v1 / d_hi
            one = torch.where(al == 0, torch.ones_like(al), al)
            a1, a2, a3 = 0.5 * be * be / one, 0.5 * (1.0 - be) ** 2 / one, 0.5 * al + be
            t1 = (be > 0).long() + (be > 1).long()
            t2 = (al + be > 0).long() + (al + be > 1).long()
            table = torch.stack([torch.zeros_like(a1), -a1, a2 - a1, a1 + a3, a3, a2 + a3, (1.0 - a2) + a1, 1.0 - a2,
                                 torch.ones_like(a1)])
            area = torch.gather(table, 0, (t1 + 3 * t2)[None])[0]
            area = torch.where(be < 0, 1.0 - area, area)
            area = torch.where(v1 < 0, 1.0 - area, area)
            area = torch.where(same, torch.zeros_like(area), area)
            area = torch.where((v1 > 0) & (v2 > 0) & (v3 > 0), torch.ones_like(area), area)
            area = torch.where((v1 <= 0) & (v2 <= 0) & (v3 <= 0), torch.zeros_like(area), area)
            out.append(torch.where(self.hm > 0, area, torch.zeros_like(area)))
        return out

    # -- inner_update!
    def inner(self):
        p, um, vm, hm = self.p, self.um * self.u, self.vm * self.v, self.hm
        ux, vy = hm * self._diff(um, 0, self.rdx), hm * self._diff(vm, 1, self.rdy)
        shear = self.cm * (self._diff(um, 1, self.rdy)[1:-1] + self._diff(vm, 0, self.rdx)[:, 1:-1])
        sh = hm * self._mean(self._mean(self._pad(self._pad(shear, 0), 1), 0), 1)
        sr2 = ux * ux + vy * vy + ux * vy + 0.25 * sh * sh
        ub, vb = hm * self._mean(um, 0), hm * self._mean(vm, 1)
        sp2 = ub * ub + vb * vb
        speed = torch.sqrt(torch.where(sp2 > 0, sp2, torch.ones_like(sp2))) * (sp2 > 0)
        bs = speed / (1.0 + self.f2 * self.beta)
        beta = self.wc * (bs * bs + p.weertman_reg_speed ** 2) ** (0.5 * (1.0 / p.weertman_m - 1.0))
        tau = beta * bs
        av = f1 = f2 = torch.zeros_like(self.h)
        on = hm > 0
        levels = []
        for k in range(self.ns):
            eta = self.eta[:, :, k]
            for _ in range(self.s.n_iter_viscosity):
                q = tau * self.zeta[k] / eta
                new = 0.5 * self.glen_b[:, :, k] * (sr2 + 0.25 * q * q + p.glen_reg_strain_rate ** 2) ** (
                    0.5 * (1.0 / p.glen_n - 1.0))
                eta = torch.where(on, new, eta)
            levels.append(eta)
            w, z = self.qw[k], self.zeta[k]
            av, f1, f2 = av + hm * w * eta, f1 + hm * w * self.h * z / eta, f2 + hm * w * self.h * z * z / eta
        self.eta, self.etaav, self.f1, self.f2, self.beta = torch.stack(levels, 2), av, f1, f2, beta
        beff = beta / (1.0 + f2 * beta)
        self.bu, self.bv = self._drag_on_faces(beff, 0, self.um, self.gfu), self._drag_on_faces(beff, 1, self.vm, self.gfv)
        he = self.h * av
        self.heta = hm * he
        self.hetac = self.cm * self._mean(self._mean(he, 0), 1)
        self.dimp = hm * (-p.density_ice * p.g * self.s.super_implicitness * p.dt) * self.dsdh

    def _drag_on_faces(self, beff, dim, mask, gff):
        b, ip = self._to_faces(beff, dim, mask), self._to_faces(self.gf, dim, mask)
        return torch.where(ip > 0, b * gff / torch.where(ip > 0, ip, torch.ones_like(ip)), b)

    # -- the momentum operator, its diagonal and the right-hand side
    def op(self, u, v):
        dudx, dvdy = self._diff(u, 0, self.rdx), self._diff(v, 1, self.rdy)
        rxx, ryy = 2.0 * self.heta * (2.0 * dudx + dvdy), 2.0 * self.heta * (2.0 * dvdy + dudx)
        rxy = self.hetac * (self._diff(u, 1, self.rdy)[1:-1] + self._diff(v, 0, self.rdx)[:, 1:-1])
        ext = self.dimp * (self._diff(self.um * self.hu * u, 0, self.rdx) + self._diff(self.vm * self.hv * v, 1, self.rdy))
        du = self._diff(self._pad(rxx, 0), 0, self.rdx) + self._diff(self._pad(self._pad(rxy, 0), 1), 1, self.rdy)
        dv = self._diff(self._pad(ryy, 1), 1, self.rdy) + self._diff(self._pad(self._pad(rxy, 1), 0), 0, self.rdx)
        yu = du - self.um * self.bu * u - self.hu * self._diff(self._pad(ext, 0), 0, self.rdx)
        yv = dv - self.vm * self.bv * v - self.hv * self._diff(self._pad(ext, 1), 1, self.rdy)
        return self.ui * yu, self.vi * yv

    def diag(self):
        out = [torch.zeros_like(self.u), torch.zeros_like(self.v)]
        for c in (0, 1):
            for a in range(3):
                for b in range(3):
                    e = [torch.zeros_like(self.u), torch.zeros_like(self.v)]
                    e[c][a::3, b::3] = 1.0
                    out[c] = out[c] + e[c] * self.op(*e)[c]
        return out

    def rhs(self):
        p, theta = self.p, self.s.super_implicitness * self.p.dt
        ri, rw, gr, sl = p.density_ice, p.density_ocean, p.g, p.sea_level_wrt_geoid
        fu, fv = self.op(self.ufix * self.u, self.vfix * self.v)
        sa = self.hm * (self.sur + theta * self.dsdh * (self.acc - self.mel))
        out = []
        for dim, rd, h, s, inner, f3 in ((0, self.rdx, self.hu, self.su, self.ui, fu),
                                         (1, self.rdy, self.hv, self.sv, self.vi, fv)):
            f1 = ri * gr * h * self._diff(self._pad(sa, dim), dim, rd)
            d = torch.clamp(h - (s - sl), min=0.0)
            f2 = self._diff(self._pad(self.hm, dim), dim, rd) * gr * (0.5 * ri * h * h - 0.5 * rw * d * d - ri * h * s)
            out.append(inner * (f1 + f2 - f3))
        return out

    # -- the V-cycle and the Picard loop
    def _inverse(self, x):
        return [m * (self.P[a.shape[0]] @ a @ self.P[a.shape[1]].T) for a, m in zip(x, (self.ui, self.vi))]

    def _restrict(self, y):
        return [w * (self.P[a.shape[0]].T @ a @ self.P[a.shape[1]]) for a, w in zip(y, self.mw)]

    def _coarse(self, x):
        return self._restrict(self.op(*self._inverse([w * a for w, a in zip(self.mw, x)])))

    @staticmethod
    def _dot(a, b):
        return float((a[0] * b[0]).sum() + (a[1] * b[1]).sum())

    def _cg(self, b, x):
        """cg!: conjugate gradients from x, stopped at max(sqrt(eps) |r0|,
        tol_coarse |b|)."""
        r = [p - q for p, q in zip(b, self._coarse(x))]
        res = math.sqrt(self._dot(r, r))
        tol = max(math.sqrt(2.0 ** -52) * res, self.s.tol_coarse * math.sqrt(self._dot(b, b)))
        u, prev, it = [torch.zeros_like(a) for a in r], 1.0, 0
        while it < self.s.maxiter_coarse and res > tol:
            u = [a + (res * res / (prev * prev)) * p for a, p in zip(r, u)]
            c = self._coarse(u)
            alpha = res * res / self._dot(u, c)
            x = [a + alpha * p for a, p in zip(x, u)]
            r = [a - alpha * q for a, q in zip(r, c)]
            prev, res, it = res, math.sqrt(self._dot(r, r)), it + 1
        return x

    def _smooth(self, e, r, d, order):
        e = list(e)
        inner = (self.ui, self.vi)
        d = [torch.where(i > 0, a, torch.ones_like(a)) for a, i in zip(d, inner)]
        for _ in range(self.s.nsmooth):
            for col in order:
                c = 0 if col <= 2 else 1
                q = (r[c] - self.op(*e)[c]) * self.s.smoother_omega / d[c]
                e[c] = e[c] + inner[c] * self.colour[col - 1] * q
        return e

    def vcycle(self, r):
        d = self.diag()
        e = self._smooth([torch.zeros_like(a) for a in r], r, d, (1, 3, 2, 4))
        self.xc = self._cg(self._restrict([a - q for a, q in zip(r, self.op(*e))]), self.xc)
        e = [a + q for a, q in zip(e, self._inverse([w * a for w, a in zip(self.mw, self.xc)]))]
        return self._smooth(e, r, d, (4, 2, 3, 1))

    def solve(self):
        for _ in range(self.s.maxiter_picard):
            self.inner()
            x = [self.ui * self.u, self.vi * self.v]
            b = self.rhs()
            r = [p - q for p, q in zip(b, self.op(*x))]
            self.resid = [torch.where(i > 0, a, o) for i, a, o in zip((self.ui, self.vi), r, self.resid)]
            if math.sqrt(self._dot(r, r) / self._dot(b, b)) < self.s.tol_picard:
                break
            e = self.vcycle(r)
            self.u = torch.where(self.ui > 0, x[0] + e[0], self.u)
            self.v = torch.where(self.vi > 0, x[1] + e[1], self.v)

    def state(self):
        self.geometry()
        self.solve()
        uh = self._mean(self.u, 0)
        self.ub = uh / (1.0 + self.beta * self.f2)
        self.us = self.ub * (1.0 + self.beta * self.f1)
        div = self._diff(self.um * self.hu * self.u, 0, self.rdx) + self._diff(self.vm * self.hv * self.v, 1, self.rdy)
        self.dhdt = torch.where(self.hm > 0, self.acc - self.mel - div, self.dhdt)
        for k, (a, m) in enumerate(((self.u, self.um), (self.v, self.vm))):
            w = self.F[a.shape[0]] @ (m * a) @ self.F[a.shape[1]].T
            self.mw[k] = (w.abs() >= self.s.wavelet_threshold).double()
            self.xc[k] = torch.zeros_like(w)

    def step(self, dt):
        self.state()
        up = torch.maximum(self.p.minimum_thickness - self.h, dt * self.dhdt)
        self.h = torch.where((self.hm > 0) & (self.hfix == 0), self.h + up, self.h)

    def solved(self):
        return {"u": self.u, "v": self.v, "resid_u": self.resid[0], "resid_v": self.resid[1], "eta": self.eta,
                "eta_av": self.etaav, "beta": self.beta, "quad_f2": self.f2}

    def stepped(self):
        return {"h": self.h, "s": self.sur, "dhdt": self.dhdt, "gf": self.gf, "us": self.us, "ub": self.ub,
                **self.solved()}

    def matrix(self):
        """The operator on the inner points, dense (columns by unit vectors
        three cells apart, whose images do not overlap)."""
        ku, kv = self.ui.reshape(-1).nonzero()[:, 0], self.vi.reshape(-1).nonzero()[:, 0]
        nu, shapes = self.u.numel(), (self.u.shape, self.v.shape)
        rows, cols, values = [], [], []
        for c in (0, 1):
            for a in range(3):
                for b in range(3):
                    e = [torch.zeros_like(self.u), torch.zeros_like(self.v)]
                    e[c][a::3, b::3] = 1.0
                    e[c] = e[c] * (self.ui, self.vi)[c]
                    src = e[c].nonzero()
                    y = self.op(*e)
                    for di in (-1, 0, 1):
                        for dj in (-1, 0, 1):
                            for o in (0, 1):
                                ti, tj = src[:, 0] + di, src[:, 1] + dj
                                ok = (ti >= 0) & (tj >= 0) & (ti < shapes[o][0]) & (tj < shapes[o][1])
                                cols.append((src[:, 0] * shapes[c][1] + src[:, 1] + c * nu)[ok])
                                rows.append((ti * shapes[o][1] + tj + o * nu)[ok])
                                values.append(y[o][ti[ok], tj[ok]])
        n = nu + self.v.numel()
        place = torch.full((n,), -1)
        keep = torch.cat([ku, nu + kv])
        place[keep] = torch.arange(len(keep))
        row, col, value = place[torch.cat(rows)], place[torch.cat(cols)], torch.cat(values)
        ok = (row >= 0) & (col >= 0)
        A = torch.zeros(len(keep), len(keep), dtype=torch.float64).index_put((row[ok], col[ok]), value[ok])
        return A, ku, kv

    def misfit(self, logc, picard, uo, vo):
        """The map whose gradient misfit_gradient takes: Picard iterations
        with exact linear solves."""
        self.C = torch.exp(logc)
        self.wc = self.C * self.gf
        for _ in range(picard):
            self.inner()
            A, ku, kv = self.matrix()
            b = self.rhs()
            x = torch.linalg.solve(A, torch.cat([b[0].reshape(-1)[ku], b[1].reshape(-1)[kv]]))
            self.u = torch.zeros(self.u.numel(), dtype=torch.float64).index_put((ku,), x[:len(ku)]).reshape(self.u.shape)
            self.v = torch.zeros(self.v.numel(), dtype=torch.float64).index_put((kv,), x[len(ku):]).reshape(self.v.shape)
        return 0.5 * ((self.ui * (self.u - uo)) ** 2).sum() + 0.5 * ((self.vi * (self.v - vo)) ** 2).sum()


# Cells for which the plain computation stays within a few seconds: a step or
# a Picard iteration takes up to 1000 coarse iterations, a gradient dense solves.
EXACT_CELLS = {"step": 2000, "transient": 900, "state": 2600, "solve": 2500, "batch": 0, "gradient": 1600}


def exact(case, seed):
    kind = case["kind"]
    if case["nx"] * case["ny"] > EXACT_CELLS[kind]:
        return None
    threads = torch.get_num_threads()
    torch.set_num_threads(min(4, threads))  # small arrays
    try:
        if kind in ("step", "transient"):
            m = _channel_run(case, seed)
            m.params.dt = STEP_DT
            r = _Plain(m)
            for _ in range(case["steps"] if kind == "transient" else SPIN_UP + 1):
                r.step(STEP_DT)
            return r.stepped()
        if kind == "state":
            r = _Plain(_irregular(case, seed))
            r.state()
            return r.stepped()
        m = _channel(case, seed)
        r = _Plain(m)
        r.geometry()
        if kind == "solve":
            r.solve()
            return r.solved()
        logc = torch.log(r.C).requires_grad_(True)
        uo, vo = (torch.tensor(np.array(a)) for a in _observed(m, seed))
        J = r.misfit(logc, case["picard"], uo, vo)
        J.backward()
        return {"J": float(J.detach()), "grad": logc.grad, "u": r.u.detach(), "v": r.v.detach()}
    finally:
        torch.set_num_threads(threads)
