"""The pair kernel and the line kernel to the bit where test_gpu_pair_kernel.py does
not reach it: with nodal metric terms at N = 1 and 2, whose node positions and
derivative matrix are binary fractions, so that node coordinates of 1/4-wide cells
set as such give the same metric terms in every repetition (checked first); and at
N = 7 with boundaries, without which the split form takes the node kernel there."""
import numpy as np
import pytest
import torch

import dgsem_amd as dg
from test_gpu_pair_kernel import OPTIONS, solver

pytestmark = pytest.mark.gpu

BOUNDED = {
    "split_walls": dict(face_boundary=[dg.BC_SLIP_WALL, dg.BC_OUTFLOW]),
    "split_hllc_walls": dict(surface_flux=dg.FLUX_HLLC, face_boundary=[dg.BC_OUTFLOW, dg.BC_SLIP_WALL]),
    "viscous_split_walls": dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73,
                                face_boundary=[dg.BC_NS_NOSLIP_WALL, dg.BC_NS_SLIP_WALL]),
}


def set_exact_coordinates(s, polydeg, cells):
    """The node positions of 1/4-wide cells, exact for N = 1 and 2."""
    n = polydeg + 1
    at = np.arange(n) * (0.25 / polydeg)
    ie, je, j, i = np.meshgrid(*(np.arange(k) for k in (*cells, n, n)), indexing="ij")
    x = np.stack([0.25 * ie + at[i], 0.25 * je + at[j]], -1).reshape(-1, n * n, 2)
    s.set_node_coordinates(torch.from_numpy(x).cuda())


CASES = [(n, dg.GEOMETRY_NODAL, name, OPTIONS[name]) for n in (1, 2) for name in OPTIONS]
CASES += [(7, dg.GEOMETRY_AFFINE, name, o) for name, o in BOUNDED.items()]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"N{c[0]}-{c[2]}")
def test_small_grid_is_bitwise_its_repetition(gpu, case):
    polydeg, geometry, name, options = case
    print(f"case pair kernel exact N={polydeg} {name}", flush=True)
    nx, ny, nn = 5, 3, (polydeg + 1) ** 2
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    times = (64 // nn) * cus * (24 // 3) // (nx * ny) + 2  # beyond the pair kernel's grids
    small = solver(polydeg, (nx, ny), geometry, options)
    long = solver(polydeg, (nx, ny * times), geometry, options)
    if geometry == dg.GEOMETRY_NODAL:
        set_exact_coordinates(small, polydeg, (nx, ny))
        set_exact_coordinates(long, polydeg, (nx, ny * times))
        for metric in ("contravariant_vectors", "inverse_jacobian"):
            a, b = getattr(small, metric)(), getattr(long, metric)()
            assert np.array_equal(b.reshape(nx, times, ny, *a.shape[1:]),
                                  np.broadcast_to(a.reshape(nx, 1, ny, *a.shape[1:]),
                                                  (nx, times, ny, *a.shape[1:])))
    rng = np.random.default_rng(polydeg)
    rho = 1.0 + 0.3 * rng.random((nx * ny, nn)) + (rng.random((nx * ny, 1)) < 0.3)
    v = 0.4 * rng.standard_normal((2, nx * ny, nn))
    p = 1.0 + 0.3 * rng.random((nx * ny, nn))
    u = torch.tensor(np.stack([rho, rho * v[0], rho * v[1],
                               p / 0.4 + 0.5 * rho * (v ** 2).sum(0)], 1), device="cuda").contiguous()

    def repeat(a):
        a = a.view(nx, 1, ny, 4, nn).expand(nx, times, ny, 4, nn)
        return a.reshape(-1, 4, nn).contiguous()

    for step in (False, True):
        out = []
        for s, start in ((small, u), (long, repeat(u))):
            r = start.clone() if step else s.empty()
            if step:
                s.ssprk3_steps(r, 1e-3, 1, s.empty(), s.empty())
            else:
                s.calc_rhs(start, r)
            out.append(r.view(-1, 4, nn))
        torch.cuda.synchronize()
        assert torch.isfinite(out[1]).all()
        assert torch.equal(out[1], repeat(out[0]))
