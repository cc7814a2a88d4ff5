"""The work a user of this framework has it do, as cases that can be timed and
checked: SSPRK3 steps of Euler and Navier-Stokes runs in 2D and 3D, the
right-hand side on a curvilinear mesh, the tangent and the adjoint of a step,
and a batched ensemble.

A case is a dict of plain values.  `prepare` builds the solver and the seeded
state a program holds before the call, `run` is one pass through the public
entry points, `exact` is the same result from plain torch operations (its own
discretisation, below), `work` counts what a pass cannot do without.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import dgsem_amd as dg

F64 = torch.float64
GAMMA = 1.4


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _case(kind, cells, degree, state, **kw):
    c = {"kind": kind, "dim": 3 if len(cells) == 3 else 2, "nx": cells[0], "ny": cells[1],
         "nz": cells[2] if len(cells) == 3 else 1, "degree": degree, "state": state,
         "viscous": False, "capturing": False, "surface": "llf", "subcell": "llf", "alpha_max": 0.5,
         "alpha_min": 0.001, "floor": 0.0, "mesh": "box", "bounds": "periodic", "mu": 0.0,
         "prandtl": 0.72, "cfl": 0.3, "steps": 1}
    c.update(kw)
    return c


def listed():
    khi = dict(capturing=True, alpha_max=0.002, cfl=0.5)
    viscous = dict(viscous=True, mu=6.25e-4)
    cases = {
        # the smallest run: the 2D Kelvin-Helmholtz example on a coarse grid, a
        # few steps at a time; launches and latency
        "khi2d_16_n3_steps": _case("steps", (16, 16), 3, "khi", steps=10, **khi),
        # the Kelvin-Helmholtz example at its usual resolution
        "khi2d_64_n3_steps": _case("steps", (64, 64), 3, "khi", steps=10, **khi),
        # the Riemann-problem example: outflow on every face, N = 5, odd grid
        "riemann2d_101x97_n5_steps": _case("steps", (101, 97), 5, "riemann", capturing=True,
                                           bounds="outflow", steps=4),
        # the viscous shock tube: Navier-Stokes between walls, shock capturing
        "shock_tube2d_200x100_n3_steps": _case(
            "steps", (200, 100), 3, "shock_tube", viscous=True, capturing=True, alpha_max=1.0,
            alpha_min=0.1, bounds="tube", mu=1e-3, prandtl=0.73, steps=4),
        # the Taylor-Green vortex of the benchmark, and its high-order run
        "tgv3d_64_n3_step": _case("steps", (64, 64, 64), 3, "tgv"),
        "tgv3d_32_n7_step": _case("steps", (32, 32, 32), 7, "tgv"),
        # the Sedov blast: shock capturing with HLLC subcells and the floor
        "sedov3d_32_n3_step": _case("steps", (32, 32, 32), 3, "sedov", capturing=True,
                                    subcell="hllc", floor=1e-13),
        # the viscous Taylor-Green vortex, low and high order
        "ns_tgv3d_32_n3_step": _case("steps", (32, 32, 32), 3, "tgv", **viscous),
        "ns_tgv3d_24_n7_step": _case("steps", (24, 24, 24), 7, "tgv", **viscous),
        # tangent and adjoint of one step of a viscous run: the two products of
        # a Gauss-Newton or sensitivity iteration
        "ns_tgv3d_16_n3_derivatives": _case("derivatives", (16, 16, 16), 3, "tgv", **viscous),
        # a residual on a curvilinear mesh of odd sizes, HLLC faces
        "warped3d_27x19x22_n4_rhs": _case("rhs", (27, 19, 22), 4, "flow", surface="hllc",
                                          mesh="warped"),
        # many small cases of different grids and degrees at once
        "ensemble2d_64_steps": _case("ensemble", (64, 64), 5, "khi", members=64, mix=1, steps=2, **khi),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _size(rng, lo, hi):
    """A size spread evenly over its logarithm, odd ones among them."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["steps2d", "steps2d", "steps3d", "steps3d", "rhs", "derivatives", "ensemble"])
    if kind == "ensemble":
        return _case("ensemble", (64, 64), 5, "khi", members=_size(rng, 4, 64), mix=rng.randint(2, 9999),
                     steps=rng.randint(1, 2), capturing=True, alpha_max=0.002, cfl=0.5)
    if kind == "steps2d" or (kind == "derivatives" and rng.random() < 0.4):
        degree = rng.choice([1, 2, 3, 3, 4, 5, 7])
        cells = tuple(_size(rng, 4, 160) for _ in range(2))
        state, opts = rng.choice([
            ("khi", dict(capturing=True, alpha_max=0.002)),
            ("khi", dict(capturing=True, alpha_max=0.5, subcell="hllc")),
            ("flow", dict()),
            ("flow", dict(surface="hllc", bounds="channel")),
            ("riemann", dict(capturing=True, bounds="outflow")),
            ("flow", dict(viscous=True, mu=5e-3, prandtl=0.73)),
            ("shock_tube", dict(viscous=True, capturing=True, alpha_max=1.0, alpha_min=0.1,
                                bounds="tube", mu=1e-3, prandtl=0.73))])
        if kind == "steps2d":
            return _case("steps", cells, degree, state, steps=_size(rng, 1, 10), **opts)
        # the derivatives at smooth states, where they exist
        opts = dict(opts, bounds="channel" if opts.get("bounds") == "outflow" else opts.get("bounds", "periodic"))
        return _case(kind, cells, min(degree, 5), "flow", **opts)
    degree = rng.choice([2, 3, 3, 4, 5, 7])
    # about 10 M nodes at most, an eighth of that with derivatives
    most = {2: 72, 3: 56, 4: 44, 5: 36, 7: 24}[degree] // (2 if kind == "derivatives" else 1)
    cells = tuple(_size(rng, 4, most) for _ in range(3))
    state, opts = rng.choice([
        ("tgv", dict()),
        ("tgv", dict(mesh="affine")),
        ("flow", dict(surface="hllc")),
        ("tgv", dict(viscous=True, mu=6.25e-4)),
        ("sedov", dict(capturing=True, subcell="hllc", floor=1e-13)),
        ("flow", dict(capturing=True, alpha_max=0.5))])
    if kind == "rhs":
        return _case("rhs", cells, degree, "flow", **dict(opts, mesh="warped"))
    if kind == "derivatives":
        return _case(kind, cells, min(degree, 5), "flow", **dict(opts, floor=0.0))
    return _case("steps", cells, degree, state, steps=_size(rng, 1, 2), **opts)


# ---------------------------------------------------------------------------
# Meshes, states and time steps, as functions of the case and the seed alone
# ---------------------------------------------------------------------------

_BOX = {"tgv": ((0.0,) * 3, (2.0 * math.pi,) * 3), "khi": ((-1.0,) * 3, (1.0,) * 3),
        "sedov": ((-1.0,) * 3, (1.0,) * 3), "flow": ((-1.0,) * 3, (1.0,) * 3),
        "riemann": ((0.0,) * 3, (1.0,) * 3), "shock_tube": ((0.0,) * 3, (1.0, 0.5, 1.0))}


def _lobatto(degree):
    """Gauss-Lobatto nodes and weights on [-1, 1]."""
    p = np.polynomial.legendre.Legendre.basis(degree)
    x = np.concatenate([[-1.0], np.sort(p.deriv().roots().real), [1.0]])
    for _ in range(3):  # (1 - x^2) P'' = 2 x P' - N (N + 1) P polishes the inner roots
        for i in range(1, degree):
            d1 = p.deriv()(x[i])
            d2 = (2 * x[i] * d1 - degree * (degree + 1) * p(x[i])) / (1 - x[i] ** 2)
            x[i] -= d1 / d2
    x = 0.5 * (x - x[::-1])
    return x, 2.0 / (degree * (degree + 1) * p(x) ** 2)


def _cells(case):
    return [case["nx"], case["ny"], case["nz"]][:case["dim"]]


def _coordinates(case):
    """Node coordinates, one tensor per component, of shape
    (elements per direction..., nodes of the last direction, ..., first)."""
    dim, n = case["dim"], case["degree"] + 1
    x, _ = _lobatto(case["degree"])
    lo, hi = _BOX[case["state"]]
    ref, out = [], []
    for d, count in enumerate(_cells(case)):
        at = (np.arange(count)[:, None] + 0.5 * (x[None, :] + 1.0)) * (2.0 / count) - 1.0
        shape = [1] * (2 * dim)
        shape[d], shape[2 * dim - 1 - d] = count, n
        ref.append(torch.from_numpy(at).cuda().view(shape).expand(*_cells(case), *[n] * dim))
    bump = 0.0
    if case["mesh"] == "warped":  # a smooth map that leaves the faces of the box periodic
        bump = 0.06 * math.prod(torch.sin(math.pi * r) for r in ref)
    for d in range(dim):
        out.append(lo[d] + 0.5 * (ref[d] + bump + 1.0) * (hi[d] - lo[d]))
    return out


def _modes(case, seed, count, amplitude, x):
    """`count` seeded fields, periodic on the box, of a few Fourier modes."""
    rng = np.random.default_rng(seed)
    lo, hi = _BOX[case["state"]]
    fields = []
    for _ in range(count):
        f = 0.0
        for _ in range(4):
            k = rng.integers(1, 4, case["dim"])
            phase, a = rng.uniform(0.0, 2.0 * math.pi), amplitude * rng.uniform(0.3, 1.0)
            arg = sum(2.0 * math.pi * int(k[d]) / (hi[d] - lo[d]) * (x[d] - lo[d])
                      for d in range(case["dim"]))
            f = f + a * torch.sin(arg + phase)
        fields.append(f)
    return fields


def _initial(case, seed):
    """(rho, momenta..., energy): the examples' states with a seeded perturbation."""
    x, dim, state = _coordinates(case), case["dim"], case["state"]
    if state == "sedov":
        # a Gaussian blast of energy 1, its centre drawn near the origin
        at = np.random.default_rng(seed).uniform(-0.05, 0.05, dim)
        r2 = sum((x[d] - float(at[d])) ** 2 for d in range(dim))
        width = 2.0 / min(_cells(case))
        rho = torch.ones_like(r2)
        p = 1e-5 + (GAMMA - 1.0) * torch.exp(-r2 / (2.0 * width ** 2)) / ((2.0 * math.pi) ** 1.5 * width ** 3)
        v = [torch.zeros_like(r2)] * dim
    elif state == "khi":
        w = _modes(case, seed, 2, 0.01, x)
        band = torch.tanh(15.0 * x[1] + 7.5) - torch.tanh(15.0 * x[1] - 7.5)
        rho = 0.5 + 0.75 * band
        v = [0.5 * (band - 1.0) + w[0], 0.1 * torch.sin(2.0 * math.pi * x[0]) + w[1]]
        p = torch.ones_like(rho)
    elif state == "tgv":
        w = _modes(case, seed, 4, 0.01, x)
        c, s = [torch.cos(t) for t in x], [torch.sin(t) for t in x]
        rho = 1.0 + 0.1 * w[3]
        v = [s[0] * c[1] * c[2] + w[0], -c[0] * s[1] * c[2] + w[1], w[2]]
        c2 = [torch.cos(2.0 * t) for t in x]
        p = 100.0 / GAMMA + (c2[0] * c2[2] + 2.0 * c2[1] + 2.0 * c2[0] + c2[1] * c2[2]) / 16.0
    elif state == "riemann":
        # four quadrants meeting near (0.8, 0.8), the fronts a few cells wide
        at = 0.8 + np.random.default_rng(seed).uniform(-0.03, 0.03, 2)
        a, b = (0.5 * (1.0 + torch.tanh((x[d] - float(at[d])) * 0.5 * _cells(case)[d])) for d in range(2))
        mix = lambda q: q[0] * a * b + q[1] * (1 - a) * b + q[2] * (1 - a) * (1 - b) + q[3] * a * (1 - b)  # noqa: E731
        rho, p = mix((1.5, 0.5323, 0.138, 0.5323)), mix((1.5, 0.3, 0.029, 0.3))
        v = [mix((0.0, 1.206, 1.206, 0.0)), mix((0.0, 0.0, 1.206, 1.206))]
    elif state == "shock_tube":
        at = 0.5 + float(np.random.default_rng(seed).uniform(-0.02, 0.02))
        s = 0.5 * (1.0 - torch.tanh((x[0] - at) * 0.5 * case["nx"]))
        rho = 1.2 + 118.8 * s
        v = _modes(case, seed, 2, 0.02, x)
        p = rho / GAMMA
    else:  # "flow": a drifting smooth field
        w = _modes(case, seed, dim + 2, 0.05, x)
        rho, p = 1.0 + w[0], 1.0 + w[1]
        v = [0.4 + 0.15 * d + w[2 + d] for d in range(dim)]
    return [rho] + [rho * c for c in v] + [p / (GAMMA - 1.0) + 0.5 * rho * sum(c * c for c in v)]


def _timestep(case, fields):
    """cfl dx / (dim (2 N + 1) max(|v_d| + c))."""
    dim, rho = case["dim"], fields[0]
    p = (GAMMA - 1.0) * (fields[-1] - 0.5 * sum(m * m for m in fields[1:-1]) / rho)
    c = torch.sqrt(GAMMA * p / rho)
    speed = max(float((torch.abs(m / rho) + c).max()) for m in fields[1:-1])
    lo, hi = _BOX[case["state"]]
    dx = min((hi[d] - lo[d]) / n for d, n in enumerate(_cells(case)))
    return case["cfl"] * dx / (dim * (2 * case["degree"] + 1) * speed)


def _to_state(case, fields):
    """Fields -> the solver's layout [element][variable][node]."""
    dim, n = case["dim"], case["degree"] + 1
    u = torch.stack([f.expand(*_cells(case), *[n] * dim) for f in fields], dim)
    return u.reshape(math.prod(_cells(case)), dim + 2, n ** dim).contiguous()


def _from_state(case, u):
    dim, n = case["dim"], case["degree"] + 1
    return list(u.view(*_cells(case), dim + 2, *[n] * dim).unbind(dim))


_CHANNEL_INFLOW = (1.0, 0.4, 0.55)  # rho, vx, vy; p = 1


def _faces(case):
    """Boundary kind per face, -x, +x, -y, +y."""
    return {"periodic": None,
            "outflow": [dg.BC_OUTFLOW] * 4,
            "channel": [dg.BC_DIRICHLET, dg.BC_OUTFLOW, dg.BC_SLIP_WALL, dg.BC_SLIP_WALL],
            "tube": [dg.BC_NS_NOSLIP_WALL] * 3 + [dg.BC_NS_SLIP_WALL]}[case["bounds"]]


def _inflow():
    rho, vx, vy = _CHANNEL_INFLOW
    return [rho, rho * vx, rho * vy, 1.0 / (GAMMA - 1.0) + 0.5 * rho * (vx * vx + vy * vy)]


def _solver(case):
    dim = case["dim"]
    lo, hi = ((-1.0,) * 3, (1.0,) * 3) if case["mesh"] == "warped" else _BOX[case["state"]]
    flux = {"llf": dg.FLUX_LLF, "hllc": dg.FLUX_HLLC}
    s = dg.StructuredSolver(dg.SolverConfig(
        dim=dim, polydeg=case["degree"], cells=_cells(case), domain_left=lo[:dim], domain_right=hi[:dim],
        equation=dg.NAVIER_STOKES if case["viscous"] else dg.EULER, gamma=GAMMA, mu=case["mu"],
        prandtl=case["prandtl"],
        volume_integral=dg.SHOCK_CAPTURING if case["capturing"] else dg.SPLIT_FORM,
        surface_flux=flux[case["surface"]], fv_flux=flux[case["subcell"]],
        alpha_max=case["alpha_max"], alpha_min=case["alpha_min"], positivity_floor=case["floor"],
        geometry=dg.GEOMETRY_AFFINE if case["mesh"] == "affine" else dg.GEOMETRY_NODAL,
        face_boundary=_faces(case),
        face_state=[_inflow(), None, None, None] if case["bounds"] == "channel" else None))
    if case["mesh"] == "warped":
        x = torch.stack([c.expand(*_cells(case), *[case["degree"] + 1] * dim)
                         for c in _coordinates(case)], -1)
        s.set_node_coordinates(x.reshape(s.n_elements, s.ndofs, dim).contiguous())
    return s


def _direction(case, seed):
    """A seeded perturbation or cotangent of a state."""
    g = torch.Generator(device="cuda").manual_seed(seed + 7)
    shape = (math.prod(_cells(case)), case["dim"] + 2, (case["degree"] + 1) ** case["dim"])
    return torch.randn(shape, generator=g, dtype=F64, device="cuda")


def _members(case, seed):
    """The ensemble's members: grids and degrees of the mix, modes of the seed."""
    from dgsem_amd import ensemble
    sizes = ensemble.khi_ensemble(case["mix"], case["members"])
    modes = ensemble.khi_ensemble(seed, case["members"])
    return [ensemble.KhiCase(a.cells, a.polydeg, b.modes) for a, b in zip(sizes, modes)]


# ---------------------------------------------------------------------------
# What is measured
# ---------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        from dgsem_amd import ensemble
        batch, u0, _ = ensemble.khi_batch(_members(case, seed))
        return {"case": case, "batch": batch, "u0": u0, "u": batch.empty(), "tmp1": batch.empty(),
                "tmp2": batch.empty()}
    solver, fields = _solver(case), _initial(case, seed)
    s = {"case": case, "solver": solver, "u0": _to_state(case, fields)}
    if kind == "rhs":
        s["out"] = solver.empty()
        return s
    s["dt"] = _timestep(case, fields)
    s.update(u=solver.empty(), tmp1=solver.empty(), tmp2=solver.empty())
    if kind == "derivatives":
        s["v"], s["w"], s["back"] = _direction(case, seed), _direction(case, seed + 1), solver.empty()
        s["u1"], s["u2"] = solver.ssprk3_stages(s["u0"], s["dt"])
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        batch, u = state["batch"], state["u"]
        u.copy_(state["u0"])
        batch.ssprk3_steps(u, case["steps"], state["tmp1"], state["tmp2"])
        return u
    solver = state["solver"]
    if kind == "rhs":
        solver.calc_rhs(state["u0"], state["out"])
        return state["out"]
    dt, tmp1, tmp2 = state["dt"], state["tmp1"], state["tmp2"]
    if kind == "derivatives":
        stages = (dt, state["u0"], state["u1"], state["u2"])
        return [solver.step_jvp(*stages, state["v"], out=state["u"], tmp1=tmp1, tmp2=tmp2),
                solver.step_vjp(*stages, state["w"], out=state["back"], tmp1=tmp1, tmp2=tmp2)]
    # the first step from the kept initial state, the others in place
    u0, u = state["u0"], state["u"]
    solver.ssprk3_stage(1, dt, None, u0, tmp1)
    solver.ssprk3_stage(2, dt, u0, tmp1, tmp2)
    solver.ssprk3_stage(3, dt, u0, tmp2, u)
    if case["steps"] > 1:
        solver.ssprk3_steps(u, dt, case["steps"] - 1, tmp1, tmp2)
    return u


def work(case):
    """Each stage reads its input (stages 2 and 3 the base state too) and
    writes its result; a curvilinear mesh's metric terms are read once a
    stage.  Flops: the two-point fluxes of every pair on a line (107 in 3D, 90
    in 2D), plus the numerical fluxes, derivatives and updates per node."""
    dim, kind = case["dim"], case["kind"]

    def nodes_and_flops(cells, degree):
        n, elements = degree + 1, math.prod(cells)
        nodes, lines = elements * n ** dim, elements * dim * n ** (dim - 1)
        flops = lines * degree * n // 2 * (107 if dim == 3 else 90) + nodes * 15
        if case["viscous"]:
            flops += lines * n * n * 4 * (dim + 2) + nodes * 90
        return nodes, flops

    if kind == "ensemble":
        nodes = flops = 0
        for m in _members(case, 0):
            a, b = nodes_and_flops(m.cells, m.polydeg)
            nodes, flops = nodes + a, flops + b
    else:
        nodes, flops = nodes_and_flops(_cells(case), case["degree"])
    state = 8.0 * nodes * (dim + 2)
    metric = 8.0 * nodes * (dim * dim + 1) if case["mesh"] == "warped" else 0.0
    if kind == "rhs":
        return {"bytes": 2.0 * state + metric, "flops": float(flops)}
    if kind == "derivatives":
        # per stage and product: the linearisation state, the direction, the
        # combination with the step's, and the result; the pair derivatives
        # cost about three fluxes
        return {"bytes": 6.0 * (3.5 * state + metric), "flops": 18.0 * flops}
    return {"bytes": case["steps"] * (8.0 * state + 3.0 * metric), "flops": 3.0 * case["steps"] * flops}


# ---------------------------------------------------------------------------
# The same results from plain torch operations
# ---------------------------------------------------------------------------

class _Exact:
    """DGSEM right-hand side on fields of shape (elements per direction...,
    nodes of the last direction, ..., first): direction d has its elements on
    axis d and its nodes on axis -1 - d."""

    def __init__(self, case):
        self.case, self.dim, self.n = case, case["dim"], case["degree"] + 1
        n = self.n
        x, w = _lobatto(case["degree"])
        wb = np.array([1.0 / np.prod([x[i] - x[j] for j in range(n) if j != i]) for i in range(n)])
        D = np.array([[0.0 if i == j else wb[j] / wb[i] / (x[i] - x[j]) for j in range(n)] for i in range(n)])
        D -= np.diag(D.sum(1))
        self.w, self.D, self.Dhat = w, D, -(D.T * w[None, :]) / w[:, None]
        legendre = np.array([[np.polynomial.legendre.Legendre.basis(k)(t) * math.sqrt(k + 0.5)
                              for k in range(n)] for t in x])
        self.modal = torch.from_numpy(np.linalg.inv(legendre)).cuda()
        self.faces = _faces(case)
        self._metric()

    # -- mesh ----------------------------------------------------------------
    def along(self, M, f, d):
        """sum_m M[i, m] f_m along direction d."""
        return torch.movedim(torch.movedim(f, -1 - d, -1) @ torch.as_tensor(M, dtype=F64, device="cuda").T, -1, -1 - d)

    def _metric(self):
        case, dim = self.case, self.dim
        if case["mesh"] != "warped":
            lo, hi = _BOX[case["state"]]
            h = [0.5 * (hi[d] - lo[d]) / c for d, c in enumerate(_cells(case))]
            det = math.prod(h)
            self.Ja = [[det / h[d] if c == d else 0.0 for c in range(dim)] for d in range(dim)]
            self.inv_j = 1.0 / det
            return
        X = [c.contiguous() for c in _coordinates(case)]
        J = [[self.along(self.D, X[c], r) for c in range(dim)] for r in range(dim)]  # dX_c / dxi_r
        if dim == 2:
            self.Ja = [[J[1][1], -J[1][0]], [-J[0][1], J[0][0]]]
            det = J[0][0] * J[1][1] - J[1][0] * J[0][1]
        else:
            self.Ja = [[None] * 3 for _ in range(3)]
            for c in range(3):
                m, l = (c + 1) % 3, (c + 2) % 3
                t = [0.5 * (X[m] * J[r][l] - X[l] * J[r][m]) for r in range(3)]
                for r in range(3):
                    a, b = (r + 1) % 3, (r + 2) % 3
                    self.Ja[r][c] = self.along(self.D, t[b], a) - self.along(self.D, t[a], b)
            det = sum(J[0][c] * (J[1][(c + 1) % 3] * J[2][(c + 2) % 3] - J[1][(c + 2) % 3] * J[2][(c + 1) % 3])
                      for c in range(3))
        self.inv_j = 1.0 / det

    def node(self, f, d, i):
        """f at node i of every line of direction d (a number stays one)."""
        return f.select(-1 - d, i) if torch.is_tensor(f) else f

    def nodes(self, fields, d, i):
        return [self.node(f, d, i) for f in fields]

    # -- pointwise -----------------------------------------------------------
    def primitive(self, u):
        v = [m / u[0] for m in u[1:-1]]
        return v, (GAMMA - 1.0) * (u[-1] - 0.5 * u[0] * sum(c * c for c in v))

    def normal_flux(self, u, n):
        v, p = self.primitive(u)
        vn = sum(a * b for a, b in zip(v, n))
        return [u[0] * vn] + [m * vn + p * c for m, c in zip(u[1:-1], n)] + [(u[-1] + p) * vn]

    @staticmethod
    def log_mean(x, y):
        f2 = ((x - y) / (x + y)) ** 2
        near = f2 < 1e-4
        ratio = torch.where(near, torch.full_like(x, 2.0), y / x)
        series = (x + y) / (2.0 + f2 * (2.0 / 3.0 + f2 * (2.0 / 5.0 + f2 * (2.0 / 7.0 + f2 * (2.0 / 9.0)))))
        return torch.where(near, series, (y - x) / torch.log(ratio))

    def two_point(self, a, b, n):
        """Chandrashekar's kinetic-energy-preserving, entropy-conservative flux."""
        (ra, va, ba), (rb, vb, bb) = a, b
        rho, beta = self.log_mean(ra, rb), self.log_mean(ba, bb)
        v = [0.5 * (s + t) for s, t in zip(va, vb)]
        p = 0.5 * (ra + rb) / (ba + bb)
        f0 = rho * sum(s * t for s, t in zip(v, n))
        f = [f0] + [f0 * s + p * t for s, t in zip(v, n)]
        square = 0.5 * sum(s * s + t * t for s, t in zip(va, vb))
        return f + [f0 * (0.5 / ((GAMMA - 1.0) * beta) - 0.5 * square) + sum(s * t for s, t in zip(f[1:], v))]

    def llf(self, ul, ur, n):
        (vl, pl), (vr, pr) = self.primitive(ul), self.primitive(ur)
        norm = sum(c * c for c in n) ** 0.5
        speed = torch.maximum(torch.abs(sum(a * b for a, b in zip(vl, n))), torch.abs(sum(a * b for a, b in zip(vr, n))))
        speed = speed + torch.maximum(torch.sqrt(GAMMA * pl / ul[0]), torch.sqrt(GAMMA * pr / ur[0])) * norm
        return [0.5 * (a + b) - 0.5 * speed * (s - r)
                for a, b, r, s in zip(self.normal_flux(ul, n), self.normal_flux(ur, n), ul, ur)]

    def hllc(self, ul, ur, n):
        norm = sum(c * c for c in n) ** 0.5
        h = [c / norm for c in n]
        (vl, pl), (vr, pr) = self.primitive(ul), self.primitive(ur)
        nl, nr = (sum(a * b for a, b in zip(v, h)) for v in (vl, vr))
        cl, cr = torch.sqrt(GAMMA * pl / ul[0]), torch.sqrt(GAMMA * pr / ur[0])
        sl, sr = torch.sqrt(ul[0]), torch.sqrt(ur[0])
        roe = lambda a, b: (sl * a + sr * b) / (sl + sr)  # noqa: E731
        vn, H = roe(nl, nr), roe((ul[-1] + pl) / ul[0], (ur[-1] + pr) / ur[0])
        c = torch.sqrt((GAMMA - 1.0) * (H - 0.5 * sum(roe(a, b) ** 2 for a, b in zip(vl, vr))))
        SL, SR = torch.minimum(nl - cl, vn - c), torch.maximum(nr + cr, vn + c)
        ml, mr = ul[0] * (SL - nl), ur[0] * (SR - nr)
        S = (pr - pl + nl * ml - nr * mr) / (ml - mr)

        def star(u, v, p, un, K, m):
            r = m / (K - S)
            us = [r] + [r * (a + (S - un) * b) for a, b in zip(v, h)]
            us.append(r * (u[-1] / u[0] + (S - un) * (S + p / m)))
            return [f + K * (a - b) for f, a, b in zip(self.normal_flux(u, h), us, u)]

        left, right = star(ul, vl, pl, nl, SL, ml), star(ur, vr, pr, nr, SR, mr)
        fl, fr = self.normal_flux(ul, h), self.normal_flux(ur, h)
        return [norm * torch.where(SL >= 0, a, torch.where(SR <= 0, d, torch.where(S >= 0, b, c)))
                for a, b, c, d in zip(fl, left, right, fr)]

    def numerical(self, kind, ul, ur, n):
        return self.hllc(ul, ur, n) if kind == "hllc" else self.llf(ul, ur, n)

    # -- blending factor -----------------------------------------------------
    def alpha(self, u):
        """Modal indicator on p rho: the energy of the highest modes.  In 3D
        the sums over the layers leave out the highest mode of the first
        direction where the other two are not the highest."""
        case, n, dim = self.case, self.n, self.dim
        _, p = self.primitive(u)
        m = p * u[0]
        for d in range(dim):
            m = self.along(self.modal, m, d)
        e = m * m
        if dim == 2:
            total = e.sum((-1, -2))
            clip1, clip2 = e[..., :n - 1, :n - 1].sum((-1, -2)), e[..., :n - 2, :n - 2].sum((-1, -2))
        else:
            s = lambda t: t.sum((-1, -2, -3))  # noqa: E731
            clip2 = s(e[..., :n - 2, :n - 2, :n - 2])
            clip1 = clip2 + s(e[..., n - 2:n - 1, :n - 1, :n - 1]) + s(e[..., :n - 2, n - 2:n - 1, :n - 1]) \
                + s(e[..., :n - 2, :n - 2, n - 2:n - 1])
            total = clip1 + s(e[..., n - 1:, :, :]) + s(e[..., :n - 1, n - 1:, :])
        share = lambda a, b: torch.where(a != 0, (a - b) / torch.where(a != 0, a, torch.ones_like(a)), torch.zeros_like(a))  # noqa: E731
        energy = torch.maximum(share(total, clip1), share(clip1, clip2))
        threshold, sharp = 0.5 * 10.0 ** (-1.8 * n ** 0.25), math.log((1.0 - 0.0001) / 0.0001)
        a = 1.0 / (1.0 + torch.exp(-sharp / threshold * (energy - threshold)))
        a = torch.where(a < case["alpha_min"], torch.zeros_like(a), a)
        a = torch.where(a > 1.0 - case["alpha_min"], torch.ones_like(a), a)
        return torch.clamp(a, max=case["alpha_max"]).detach()

    # -- boundaries (2D) -----------------------------------------------------
    def outer(self, kind, u, d, inner, n):
        """The state beyond a boundary face, u: the boundary elements' fields
        with the direction's elements on axis d cut to one."""
        if kind == dg.BC_DIRICHLET:
            return [torch.full_like(i, v) for i, v in zip(inner, _inflow())]
        if kind == dg.BC_OUTFLOW:
            return [f.mean(-1 - d) for f in u]
        nn, mn = sum(c * c for c in n), sum(m * c for m, c in zip(inner[1:-1], n))
        return [inner[0]] + [m - 2.0 * mn / nn * c for m, c in zip(inner[1:-1], n)] + [inner[-1]]

    def edge(self, f, d, last):
        return f.narrow(d, f.shape[d] - 1 if last else 0, 1) if torch.is_tensor(f) else f

    # -- right-hand side -----------------------------------------------------
    def rhs(self, u, alpha=None):
        case, dim, n, w = self.case, self.dim, self.n, self.w
        v, p = self.primitive(u)
        prims = [u[0], v, u[0] / (2.0 * p)]
        blend = None
        if case["capturing"]:
            a = self.alpha(u) if alpha is None else alpha
            blend = a.reshape(*a.shape, *[1] * (dim - 1))
        total = [0.0] * (dim + 2)
        for d in range(dim):
            acc = [[0.0] * n for _ in range(dim + 2)]
            for i in range(n):
                for j in range(i + 1, n):
                    pick = lambda k: [self.node(prims[0], d, k), self.nodes(prims[1], d, k), self.node(prims[2], d, k)]  # noqa: E731
                    nrm = [0.5 * (self.node(c, d, i) + self.node(c, d, j)) for c in self.Ja[d]]
                    f = self.two_point(pick(i), pick(j), nrm)
                    for q in range(dim + 2):
                        acc[q][i] = acc[q][i] + 2.0 * self.D[i, j] * f[q]
                        acc[q][j] = acc[q][j] + 2.0 * self.D[j, i] * f[q]
            if blend is not None:
                fv = [[0.0] * n for _ in range(dim + 2)]
                nrm = [self.node(c, d, 0) for c in self.Ja[d]]
                for i in range(n - 1):
                    nrm = [a + w[i] * sum(self.D[i, m] * self.node(c, d, m) for m in range(n))
                           for a, c in zip(nrm, self.Ja[d])]
                    f = self.numerical(case["subcell"], self.nodes(u, d, i), self.nodes(u, d, i + 1), nrm)
                    for q in range(dim + 2):
                        fv[q][i] = fv[q][i] + f[q] / w[i]
                        fv[q][i + 1] = fv[q][i + 1] - f[q] / w[i + 1]
                acc = [[(1.0 - blend) * a + blend * b for a, b in zip(x, y)] for x, y in zip(acc, fv)]
            lower, upper = self.face_fluxes(u, d)
            for q in range(dim + 2):
                acc[q][0] = acc[q][0] - lower[q] / w[0]
                acc[q][-1] = acc[q][-1] + upper[q] / w[-1]
                total[q] = total[q] + torch.stack(acc[q], -1 - d)
        if case["viscous"]:
            total = [a + b for a, b in zip(total, self.viscous(u))]
        return [-self.inv_j * t for t in total]

    def face_fluxes(self, u, d):
        """Numerical fluxes at the lower and the upper face of every element."""
        inner, far = self.nodes(u, d, 0), self.nodes(u, d, self.n - 1)
        nrm = self.nodes(self.Ja[d], d, 0)
        flux = self.numerical(self.case["surface"], [torch.roll(f, 1, d) for f in far], inner, nrm)
        upper = [torch.roll(f, -1, d) for f in flux]
        if self.faces is not None and self.faces[2 * d] != dg.BC_PERIODIC:
            lo, hi = [self.edge(f, d, False) for f in u], [self.edge(f, d, True) for f in u]
            own, end = self.nodes(lo, d, 0), self.nodes(hi, d, self.n - 1)
            nl = [self.edge(c, d, False) for c in nrm]
            nh = [self.edge(c, d, True) for c in self.nodes(self.Ja[d], d, self.n - 1)]
            first = self.numerical(self.case["surface"], self.outer(self.faces[2 * d], lo, d, own, nl), own, nl)
            last = self.numerical(self.case["surface"], end, self.outer(self.faces[2 * d + 1], hi, d, end, nh), nh)
            count = flux[0].shape[d]
            flux = [torch.cat([a, f.narrow(d, 1, count - 1)], d) for a, f in zip(first, flux)]
            upper = [torch.cat([f.narrow(d, 0, count - 1), a], d) for a, f in zip(last, upper)]
        return flux, upper

    def with_ends(self, f, d, lower, upper):
        """f plus face terms at the first and last node of direction d."""
        parts = list(f.unbind(-1 - d))
        parts[0], parts[-1] = parts[0] - lower / self.w[0], parts[-1] + upper / self.w[-1]
        return torch.stack(parts, -1 - d)

    def viscous(self, u):
        """BR1: lifted gradients of (rho, v, T), then the divergence of the
        viscous flux with the upper element's value at each interface."""
        case, dim, n = self.case, self.dim, self.n
        v, p = self.primitive(u)
        q = [u[0]] + v + [p / u[0]]
        bounded = lambda d: self.faces is not None and self.faces[2 * d] != dg.BC_PERIODIC  # noqa: E731
        G = []
        for d in range(dim):
            lo, hi = self.nodes(q, d, 0), self.nodes(q, d, n - 1)
            lower = [0.5 * (torch.roll(b, 1, d) + a) for a, b in zip(lo, hi)]
            upper = [torch.roll(f, -1, d) for f in lower]
            if bounded(d):
                count = lo[0].shape[d]
                for side in (0, 1):
                    own = [self.edge(f, d, side) for f in (hi if side else lo)]
                    nrm = [self.edge(c, d, side) for c in self.nodes(self.Ja[d], d, n - 1 if side else 0)]
                    kind = self.faces[2 * d + side]
                    if kind == dg.BC_DIRICHLET:
                        rho, vx, vy = _CHANNEL_INFLOW
                        wall = [torch.full_like(own[0], x) for x in (rho, vx, vy, 1.0 / rho)]
                    elif kind == dg.BC_NS_NOSLIP_WALL:
                        wall = [own[0]] + [torch.zeros_like(c) for c in own[1:-1]] + [own[-1]]
                    elif kind == dg.BC_NS_SLIP_WALL:
                        vn = sum(a * b for a, b in zip(own[1:-1], nrm)) / sum(c * c for c in nrm)
                        wall = [own[0]] + [a - vn * b for a, b in zip(own[1:-1], nrm)] + [own[-1]]
                    else:
                        wall = [torch.zeros_like(c) for c in own]
                    if side:
                        upper = [torch.cat([f.narrow(d, 0, count - 1), a], d) for f, a in zip(upper, wall)]
                    else:
                        lower = [torch.cat([a, f.narrow(d, 1, count - 1)], d) for f, a in zip(lower, wall)]
            G.append([self.with_ends(self.along(self.Dhat, f, d), d, a, b) for f, a, b in zip(q, lower, upper)])
        g = [[self.inv_j * sum(self.Ja[d][c] * G[d][k] for d in range(dim)) for k in range(dim + 2)]
             for c in range(dim)]  # g[c][k] = d q_k / d x_c
        mu, kappa = case["mu"], GAMMA / ((GAMMA - 1.0) * case["prandtl"])
        div = sum(g[c][1 + c] for c in range(dim))
        F = []
        for c in range(dim):
            # the 2D equations use the 3D stress tensor with no flow in z
            tau = [g[c][1 + k] + g[k][1 + c] - (2.0 / 3.0 * div if k == c else 0.0) for k in range(dim)]
            F.append([torch.zeros_like(u[0])] + [mu * t for t in tau]
                     + [mu * (sum(a * b for a, b in zip(v, tau)) + kappa * g[c][dim + 1])])
        total = [0.0] * (dim + 2)
        for d in range(dim):
            H = [-sum(self.Ja[d][c] * F[c][k] for c in range(dim)) for k in range(dim + 2)]
            for k in range(dim + 2):
                lower = self.node(H[k], d, 0)
                upper = torch.roll(lower, -1, d)
                if bounded(d):
                    count = lower.shape[d]
                    carried = [1.0 if kind == dg.BC_DIRICHLET else float(kind == dg.BC_NS_NOSLIP_WALL and 0 < k <= dim)
                               for kind in self.faces[2 * d:2 * d + 2]]
                    end = self.node(H[k], d, n - 1).narrow(d, count - 1, 1)
                    upper = torch.cat([upper.narrow(d, 0, count - 1), carried[1] * end], d)
                    lower = torch.cat([carried[0] * lower.narrow(d, 0, 1), lower.narrow(d, 1, count - 1)], d)
                total[k] = total[k] + self.with_ends(self.along(self.Dhat, H[k], d), d, lower, upper)
        return total

    # -- SSPRK3 --------------------------------------------------------------
    def limit(self, u):
        floor = self.case["floor"]
        if floor <= 0.0:
            return u
        rho = torch.clamp(u[0], min=floor)
        kinetic = 0.5 * sum(m * m for m in u[1:-1]) / rho
        low = (GAMMA - 1.0) * (u[-1] - kinetic) < floor
        return [rho] + u[1:-1] + [torch.where(low, floor / (GAMMA - 1.0) + kinetic, u[-1])]

    def step(self, u, dt, at=(None, None, None)):
        f = self.rhs(u, at[0])
        u1 = self.limit([a + dt * b for a, b in zip(u, f)])
        f = self.rhs(u1, at[1])
        u2 = self.limit([0.75 * a + 0.25 * b + 0.25 * dt * c for a, b, c in zip(u, u1, f)])
        f = self.rhs(u2, at[2])
        return self.limit([a / 3.0 + 2.0 / 3.0 * b + 2.0 / 3.0 * dt * c for a, b, c in zip(u, u2, f)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return _exact_ensemble(case, seed)
    fields = [f.contiguous() for f in _initial(case, seed)]
    solver = _Exact(case)
    if kind == "rhs":
        return _to_state(case, solver.rhs(fields))
    dt = _timestep(case, fields)
    if kind == "steps":
        for _ in range(case["steps"]):
            fields = solver.step(fields, dt)
        return _to_state(case, fields)
    # adjoint by backpropagation; tangent as the derivative of w -> J^T w
    fields = [f.requires_grad_() for f in fields]
    out = solver.step(fields, dt)
    cotangent = [f.detach().clone().requires_grad_() for f in _from_state(case, _direction(case, seed + 1))]
    back = torch.autograd.grad(out, fields, cotangent, create_graph=True)
    forward = torch.autograd.grad(back, cotangent, _from_state(case, _direction(case, seed)))
    return [_to_state(case, forward), _to_state(case, [f.detach() for f in back])]


def _exact_ensemble(case, seed):
    from dgsem_amd import ensemble
    out = []
    for m in _members(case, seed):
        one = dict(case, nx=m.cells[0], ny=m.cells[1], degree=m.polydeg)
        x = _coordinates(one)
        u = ensemble.khi_state(torch.stack([c.expand(*m.cells, m.polydeg + 1, m.polydeg + 1) for c in x], -1)
                               .cpu().numpy(), m.modes)
        dt = ensemble.khi_dt(u, m.polydeg, m.cells)
        fields = [f.contiguous() for f in torch.from_numpy(u).cuda().unbind(-1)]
        solver = _Exact(one)
        for _ in range(case["steps"]):
            fields = solver.step(fields, dt)
        out.append(_to_state(one, fields).reshape(-1))
    return torch.cat(out)
