"""Small 2D grids run one thread per flux, larger ones one per line, in the same
order of operations: a small grid and its periodic repetition along y, long enough
for the line kernel, must give the same numbers.  With affine geometry, whose
metric terms do not depend on the position, to the bit; with nodal geometry up to
the rounding of the long grid's coordinates, about 120 repetitions * epsilon of
the fluxes, below 1e-9 of the largest value for every length used here."""
import numpy as np
import pytest
import torch

import dgsem_amd as dg

pytestmark = pytest.mark.gpu

INFLOW = [1.1, 0.3, -0.2, 2.4]
OPTIONS = {
    "split": dict(),
    "capturing": dict(volume_integral=dg.SHOCK_CAPTURING, alpha_max=0.6),
    "capturing_outflow": dict(volume_integral=dg.SHOCK_CAPTURING, alpha_max=0.6, positivity_floor=1e-13,
                              face_boundary=[dg.BC_OUTFLOW, dg.BC_SLIP_WALL]),
    "hllc_channel": dict(surface_flux=dg.FLUX_HLLC, face_boundary=[dg.BC_DIRICHLET, dg.BC_OUTFLOW],
                         face_state=[INFLOW, None, None, None]),
    "capturing_hllc": dict(volume_integral=dg.SHOCK_CAPTURING, surface_flux=dg.FLUX_HLLC,
                           fv_flux=dg.FLUX_HLLC, alpha_max=0.6),
    "central": dict(volume_flux=dg.FLUX_CENTRAL, surface_flux=dg.FLUX_CENTRAL),
    "viscous": dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73),
    "viscous_walls": dict(equation=dg.NAVIER_STOKES, mu=5e-3, prandtl=0.73,
                          volume_integral=dg.SHOCK_CAPTURING, alpha_max=0.6,
                          face_boundary=[dg.BC_NS_NOSLIP_WALL, dg.BC_NS_SLIP_WALL]),
}


def solver(polydeg, cells, geometry, options):
    o = dict(options)
    if "face_boundary" in o:
        o["face_boundary"] = list(o["face_boundary"]) + [dg.BC_PERIODIC] * 2
    return dg.StructuredSolver(dg.SolverConfig(
        dim=2, polydeg=polydeg, cells=cells, domain_left=(0.0, 0.0),
        domain_right=tuple(0.25 * c for c in cells), geometry=geometry, **o))


@pytest.mark.parametrize("geometry", [dg.GEOMETRY_AFFINE, dg.GEOMETRY_NODAL])
@pytest.mark.parametrize("name", OPTIONS)
@pytest.mark.parametrize("polydeg", [1, 2, 3, 4, 5, 7])
def test_small_grid_matches_its_repetition(gpu, polydeg, name, geometry):
    if name == "central" and polydeg == 7:
        pytest.skip("CentralFlux is built up to N = 5")
    print(f"case pair kernel N={polydeg} {name} {geometry}", flush=True)
    nx, ny, nn = 5, 3, (polydeg + 1) ** 2
    small = solver(polydeg, (nx, ny), geometry, OPTIONS[name])
    # beyond the pair kernel's grids: six blocks of 64 // nn elements on each of 256 CUs
    times = (64 // nn) * 256 * 6 // (nx * ny) + 2
    long = solver(polydeg, (nx, ny * times), geometry, OPTIONS[name])
    rng = np.random.default_rng(polydeg)
    rho = 1.0 + 0.3 * rng.random((nx * ny, nn)) + (rng.random((nx * ny, 1)) < 0.3)
    v = 0.4 * rng.standard_normal((2, nx * ny, nn))
    p = 1.0 + 0.3 * rng.random((nx * ny, nn))
    u = torch.tensor(np.stack([rho, rho * v[0], rho * v[1],
                               p / 0.4 + 0.5 * rho * (v ** 2).sum(0)], 1), device="cuda")
    repeat = lambda a: a.view(nx, 1, ny, 4, nn).expand(nx, times, ny, 4, nn).reshape(-1, 4, nn).contiguous()  # noqa: E731
    for step in (False, True):
        out = []
        for s, state in ((small, u.contiguous()), (long, repeat(u))):
            if step:
                r = state.clone()
                s.ssprk3_steps(r, 1e-3, 1, s.empty(), s.empty())
            else:
                r = s.empty()
                s.calc_rhs(state, r)
            out.append(r)
        torch.cuda.synchronize()
        want = repeat(out[0].view(-1, 4, nn))
        got = out[1].view(-1, 4, nn)
        assert torch.isfinite(got).all()
        if geometry == dg.GEOMETRY_AFFINE:
            assert torch.equal(got, want)
        else:
            scale = want.abs().max()
            assert float((got - want).abs().max() / scale) < 1e-9
