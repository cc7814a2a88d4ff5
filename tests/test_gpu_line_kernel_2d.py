"""2D grids past the sizes of the pair kernel, where a thread takes a whole line,
and past 100 000 line threads on 256 CUs, where box meshes' metric terms come from
the compact table.

Checks:
  * table against full metric arrays (see test_gpu_box_tables.py), periodic and with
    boundaries on every face, Euler and Navier-Stokes: the same bits;
  * every boundary kind on faces of both directions, also per-node Dirichlet states
    and the mixed wall, against the oracle, on both sides of the table's line
    (relative L2 <= 1e-12, the bar of test_gpu_boundaries.py; identical troubled
    sets).

The sizes are derived from the two lines, so that they cannot drift below them."""
import math

import numpy as np
import pytest
import torch

import dgsem_amd as dg
from gpu_pairs import gpu_rhs, rel_l2
from oracle import oracle as O
from test_gpu_boundaries import INFLOW, make_bc_pair, state
from test_gpu_box_tables import pair_run
from test_gpu_ns_walls import LAYOUTS as NS_LAYOUTS
from test_gpu_ns_walls import make_ns_pair, smooth_state

pytestmark = pytest.mark.gpu

RHS_TOL = 1e-12
WALLS = [dg.BC_SLIP_WALL] * 4
OPEN = [dg.BC_DIRICHLET, dg.BC_OUTFLOW, dg.BC_OUTFLOW, dg.BC_DIRICHLET]
TALL = [dg.BC_SLIP_WALL, dg.BC_OUTFLOW, dg.BC_DIRICHLET, dg.BC_OUTFLOW]
NOSLIP, SLIP = dg.BC_NS_NOSLIP_WALL, dg.BC_NS_SLIP_WALL


def grid(polydeg, table):
    """Cells of an odd-sized grid on the wanted side of the table's line and above
    the largest grid of the pair kernel (its blocks of 64 // nodes elements have four
    waves at N = 1 and five or more beyond; 24 waves fit a CU, at N = 7 twice over)."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    line = math.ceil(100000 * cus / 256 / (2 * (polydeg + 1)))
    pair = 64 // (polydeg + 1) ** 2 * cus * (24 // (4 if polydeg == 1 else 5)) + 1
    least = line if table else max(pair, line // 2)
    ny = math.isqrt(least) | 1
    nx = (least // ny + 1) | 1
    assert nx * ny >= pair and (nx * ny >= line) == table
    return nx, ny


def perturbed(x):
    """Noise on density, velocity and pressure, and a jump."""
    rng = np.random.default_rng(x.shape[0])
    rho = 1.0 + 0.3 * rng.random(x.shape[:-1]) + (x[..., 0] < 0.1)
    v = 0.3 * rng.standard_normal((2,) + rho.shape)
    p = 1.0 + 0.3 * rng.random(rho.shape)
    return np.stack([rho, rho * v[0], rho * v[1], p / 0.4 + 0.5 * rho * (v ** 2).sum(0)], -1)


TABLE = {
    "periodic": (3, dict(volume_integral=dg.SHOCK_CAPTURING)),
    "periodic_split_hllc": (2, dict(surface_flux=dg.FLUX_HLLC)),
    "walls": (5, dict(volume_integral=dg.SHOCK_CAPTURING, face_boundary=WALLS)),
    "open": (3, dict(face_boundary=OPEN)),
    "tall_hllc": (4, dict(volume_integral=dg.SHOCK_CAPTURING, surface_flux=dg.FLUX_HLLC,
                          fv_flux=dg.FLUX_HLLC, face_boundary=TALL)),
    "walls_n1": (1, dict(face_boundary=WALLS)),
    "walls_n7": (7, dict(face_boundary=WALLS)),
    "viscous": (3, dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73)),
    "viscous_tube": (3, dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73,
                             volume_integral=dg.SHOCK_CAPTURING, face_boundary=NS_LAYOUTS["shock_tube"])),
    "viscous_open": (5, dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73,
                             face_boundary=NS_LAYOUTS["euler_kinds"])),
}


@pytest.mark.parametrize("name", TABLE)
def test_table_is_bitwise_the_nodal_arrays(gpu, name):
    polydeg, options = TABLE[name]
    cells = grid(polydeg, True)
    print(f"case 2D box table {name} N={polydeg} {cells}", flush=True)
    states = [INFLOW if k == dg.BC_DIRICHLET else [0.0] * 4
              for k in options.get("face_boundary", [dg.BC_PERIODIC] * 4)]
    cfg = dg.SolverConfig(dim=2, polydeg=polydeg, cells=cells, domain_left=(-1.0, -0.5),
                          domain_right=(1.0, 0.75), face_state=states, alpha_max=0.5,
                          alpha_min=0.001, **options)
    du_box, du, st_box, st = pair_run(cfg, perturbed, 1e-6)
    assert torch.isfinite(du).all()
    assert torch.equal(du_box, du)
    assert torch.equal(st_box, st)


BOUNDED = [
    # N, table, faces, volume integral, surface flux, geometry
    (3, True, OPEN, dg.SHOCK_CAPTURING, dg.FLUX_LLF, dg.GEOMETRY_NODAL),
    (5, True, WALLS, dg.SPLIT_FORM, dg.FLUX_HLLC, dg.GEOMETRY_NODAL),
    (3, False, TALL, dg.SHOCK_CAPTURING, dg.FLUX_HLLC, dg.GEOMETRY_NODAL),
    (4, False, OPEN, dg.SPLIT_FORM, dg.FLUX_LLF, dg.GEOMETRY_NODAL),
    (2, False, TALL, dg.SPLIT_FORM, dg.FLUX_LLF, dg.GEOMETRY_AFFINE),
    (5, False, WALLS, dg.SHOCK_CAPTURING, dg.FLUX_LLF, dg.GEOMETRY_AFFINE),
    (7, False, OPEN, dg.SHOCK_CAPTURING, dg.FLUX_LLF, dg.GEOMETRY_NODAL),
]


@pytest.mark.parametrize("case", BOUNDED, ids=lambda c: f"N{c[0]}-{'table' if c[1] else 'arrays'}-{c[5]}")
def test_boundaries_match_oracle(gpu, case):
    polydeg, table, faces, volume, surface, geometry = case
    cells = grid(polydeg, table)
    print(f"case 2D line boundaries N={polydeg} {cells} {faces} {volume} {surface} {geometry}", flush=True)
    oc, gs = make_bc_pair(polydeg, cells, faces, volume=volume, surface=surface, geometry=geometry)
    u = state(oc, seed=polydeg)
    ref, alpha = oc.rhs(u, with_alpha=True)
    assert rel_l2(gpu_rhs(gs, u), ref) <= RHS_TOL
    if volume == dg.SHOCK_CAPTURING:
        assert (alpha > 0).any()
        assert np.array_equal(gs.alpha().cpu().numpy() > 0, alpha > 0)


@pytest.mark.parametrize("table", [True, False])
def test_per_node_states_match_oracle(gpu, table):
    """The mixed wall below, per-node Dirichlet states above and on the left."""
    polydeg = 3
    nx, ny = cells = grid(polydeg, table)
    print(f"case 2D line per-node states {cells}", flush=True)
    faces = [dg.BC_DIRICHLET, dg.BC_OUTFLOW, dg.BC_MIXED_DIRICHLET_SLIP_WALL, dg.BC_DIRICHLET]
    oc, gs = make_bc_pair(polydeg, cells, faces, volume=dg.SHOCK_CAPTURING)
    rng = np.random.default_rng(4)
    kept = []
    for face, kind, count in ((0, O.BC_DIRICHLET, ny), (2, O.BC_MIXED_DIRICHLET_SLIP_WALL, nx),
                              (3, O.BC_DIRICHLET, nx)):
        vals = np.tile(np.asarray(INFLOW), (count * (polydeg + 1), 1))
        vals[:, 0] += 0.1 * rng.random(len(vals))
        vals[:, 3] += 0.2 * rng.random(len(vals))
        if kind == O.BC_MIXED_DIRICHLET_SLIP_WALL:
            vals = np.column_stack([vals, rng.random(len(vals)) < 0.5])
            oc.set_boundary(face, kind, values=vals)
        else:
            oc.set_boundary(face, kind, state=INFLOW, values=vals)
        kept.append(torch.from_numpy(vals).cuda())
        gs.set_boundary_values(face, kept[-1])
    u = state(oc, seed=9)
    assert rel_l2(gpu_rhs(gs, u), oc.rhs(u)) <= RHS_TOL


@pytest.mark.parametrize("polydeg,table,layout,volume", [
    (3, True, "shock_tube", dg.SHOCK_CAPTURING),
    (5, True, "euler_kinds", dg.SPLIT_FORM),
    (4, False, "noslip_box", dg.SPLIT_FORM),
    (2, False, "mixed_channel", dg.SHOCK_CAPTURING),
])
def test_viscous_walls_match_oracle(gpu, polydeg, table, layout, volume):
    cells = grid(polydeg, table)
    print(f"case 2D line viscous N={polydeg} {cells} {layout}", flush=True)
    oc, gs = make_ns_pair(polydeg, cells, NS_LAYOUTS[layout], volume=volume)
    u = smooth_state(oc, seed=polydeg)
    assert rel_l2(gpu_rhs(gs, u), oc.rhs(u)) <= RHS_TOL
