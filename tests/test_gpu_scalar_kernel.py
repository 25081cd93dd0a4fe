"""The passive-scalar kernel (several scalars in one pass after the hydro kernel, which stores the
face mass fluxes) against the oracle, bit for bit, where its tiles and groups can go wrong: extents
one below, at and one above a whole number of tiles (62 columns in 2D, 14 x 14 in 3D), ragged last
segments, every group size, and one scalar in a kernel of its own."""

import numpy as np
import pytest

from heraclespp_amd import Grid, HydroSolver, PerfectGas
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

CASES = [
    (1, (131, 1, 1), "Cartesian", 4, "HLLC", "VanLeer"),
    (1, (64, 1, 1), "Spherical", 2, "HLL", "Minmod"),
    (2, (61, 9, 1), "Cartesian", 2, "HLLC", "Minmod"),
    (2, (62, 7, 1), "Cartesian", 3, "Low Mach", "VanAlbada"),
    (2, (63, 5, 1), "Spherical", 5, "HLL", "VanLeer"),
    (2, (125, 40, 1), "Cartesian", 6, "HLLC", "VanLeer"),
    (3, (13, 14, 5), "Cartesian", 2, "HLLC", "Minmod"),
    (3, (14, 15, 6), "Cartesian", 4, "HLLC", "VanLeer"),
    (3, (15, 28, 4), "Spherical", 3, "HLLC", "VanAlbada"),
    (3, (29, 13, 7), "Spherical", 9, "HLL", "Minmod"),
]


@pytest.mark.parametrize("nd,n,geom,nfx,riemann,limiter", CASES)
def test_scalar_kernel_matches_oracle(cuda, nd, n, geom, nfx, riemann, limiter):
    lo, hi = ((0.2, 0.5, 0.1), (1.0, 2.5, 3.0)) if geom == "Spherical" else ((0.0,) * 3, (1.0, 0.8, 1.2))
    bc = (["Reflexive", "NullGradient", "Periodic", "Periodic", "NullGradient", "Reflexive"] if geom == "Cartesian"
          else ["Reflexive", "NullGradient", "Reflexive", "Reflexive", "Periodic", "Periodic"])[:2 * nd]
    o = orc.Oracle(nd, n, geom=geom, limiter=limiter, riemann=riemann, gamma=1.4, bc=bc, xmin=lo, xmax=hi, nfx=nfx)
    rng = np.random.default_rng(3)
    rho, P = 0.5 + rng.random(o.shape3), 0.5 + rng.random(o.shape3)
    u = rng.uniform(-0.6, 0.6, size=(nd,) + o.shape3)
    fx = rng.random((nfx,) + o.shape3)
    steps = 4
    o.init_from_prim(rho, u, P, fx)
    for _ in range(steps):
        o.step(0.3, 1e30, steps)
    sol = HydroSolver(Grid(nd, n, 2, geom, lo, hi), PerfectGas(1.4, 1.0), reconstruction=limiter, riemann_solver=riemann, bc=bc, cfl=0.3, nfx=nfx)
    sol.init_from_prim(rho, u, P, fx=fx)
    assert sol.run(1e30, steps) == steps and sol.t == o.t
    for name in ("rho", "rhou", "E", "fx"):
        np.testing.assert_array_equal(getattr(sol, name).cpu().numpy(), o.state(name), err_msg=name)


def test_one_scalar_in_a_kernel_of_its_own(cuda):
    """From 2^21 cells on a 3D FP64 Cartesian run takes its one scalar apart from the hydro kernel."""
    n = (128, 128, 128)
    grid = Grid(3, n, 2, "Cartesian", (0.0,) * 3, (1.0,) * 3)
    rng = np.random.default_rng(5)
    rho, P = 0.5 + rng.random(grid.shape3), 0.5 + rng.random(grid.shape3)
    u, fx = rng.uniform(-0.6, 0.6, size=(3,) + grid.shape3), rng.random((1,) + grid.shape3)
    out = []
    for fused in (True, False):
        sol = HydroSolver(grid, PerfectGas(1.4, 1.0), reconstruction="Minmod", riemann_solver="HLLC", nfx=1, fused=fused)
        sol.init_from_prim(rho, u, P, fx=fx)
        assert sol.run(1e30, 2) == 2
        out.append([t.cpu().numpy() for t in (sol.rho, sol.rhou, sol.E, sol.fx)])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
