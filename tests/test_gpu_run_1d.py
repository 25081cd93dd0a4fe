"""Runs of small 1D grids, which one workgroup takes through many steps in one launch, against the
same steps launched one by one (hclpp_step): states, clock and the discarded step of a run that fails,
bit for bit; the conserved totals to their summation order."""

import numpy as np
import pytest
import torch

from heraclespp_amd import Grid, HydroSolver, PerfectGas, UniformGravity

pytestmark = pytest.mark.gpu


def _solver(n, geom, ng, riemann, limiter, precision, bc):
    grid = Grid(1, (n, 1, 1), ng, geom, (0.3, 0.0, 0.0), (1.0, 1.0, 1.0))
    return HydroSolver(grid, PerfectGas(1.4, 0.7), reconstruction=limiter, riemann_solver=riemann, bc=bc, cfl=0.4, precision=precision,
                       gravity=UniformGravity((-0.05, 0.0, 0.0)))


def _initial(grid, seed):
    rng = np.random.default_rng(seed)
    x = np.linspace(0, 1, grid.shape3[2])[None, None, :]
    rho = np.where(x < 0.5, 1.0, 0.125) * (1 + 0.1 * rng.random(grid.shape3))
    return rho, 0.2 * rng.standard_normal((1,) + grid.shape3), np.where(x < 0.5, 1.0, 0.1) + 0 * rho


def _one_by_one(sol, steps, t_end=1e30):
    sol.start_clock(t_end, steps)
    for _ in range(steps):
        sol.step_async()
    return sol.finish()


CASES = [
    (2, "Cartesian", 2, "HLL", "Minmod", "fp64", ["Periodic", "Periodic"]),
    (64, "Spherical", 2, "HLLC", "VanLeer", "fp64", ["Reflexive", "NullGradient"]),
    (1000, "Cartesian", 2, "HLL", "Minmod", "fp64", ["NullGradient", "NullGradient"]),
    (1022, "Spherical", 3, "Low Mach", "VanAlbada", "fp64", ["Reflexive", "Reflexive"]),
    (1023, "Cartesian", 4, "HLLC", "VanLeer", "fp64", ["Periodic", "Periodic"]),
    (2046, "Cartesian", 2, "HLLC", "Constant", "fp64", ["NullGradient", "Reflexive"]),
    (2047, "Cartesian", 2, "HLLC", "VanLeer", "fp64", ["Periodic", "Periodic"]),
    (700, "Spherical", 2, "HLLC", "Minmod", "fp32", ["Reflexive", "NullGradient"]),
    (1500, "Cartesian", 2, "HLL", "VanLeer", "fp32", ["Periodic", "Periodic"]),
]


@pytest.mark.parametrize("steps", [70, 3])
@pytest.mark.parametrize("n,geom,ng,riemann,limiter,precision,bc", CASES)
def test_one_launch_is_the_steps_one_by_one(cuda, n, geom, ng, riemann, limiter, precision, bc, steps):
    sols = [_solver(n, geom, ng, riemann, limiter, precision, bc) for _ in range(2)]
    init = _initial(sols[0].grid, n)
    for s in sols:
        s.init_from_prim(*init)
    assert sols[0].run(1e30, steps) == steps
    clk = sols[0].clock()
    ref = _one_by_one(sols[1], steps)
    for name in ("t", "iter", "dt", "min_eint", "done", "status"):
        assert getattr(clk, name) == getattr(ref, name), name
    assert clk.mass == pytest.approx(ref.mass, rel=1e-13) and clk.energy == pytest.approx(ref.energy, rel=1e-13)
    for name in ("rho", "rhou", "E"):
        assert torch.equal(getattr(sols[0], name), getattr(sols[1], name)), name


def test_t_end_and_the_discarded_step(cuda):
    """A run that ends inside a batch at t_end, and one whose first step finds an invalid state: the state,
    the count and the time are those of the steps that were completed."""
    for kill in (False, True):
        sols = [_solver(300, "Cartesian", 2, "HLLC", "VanLeer", "fp64", ["Periodic", "Periodic"]) for _ in range(2)]
        init = _initial(sols[0].grid, 1)
        for s in sols:
            s.init_from_prim(*init)
        t_end = 1e30
        if kill:
            for s in sols:  # a cold supersonic inflow into a cell: the energy fails after some steps, or at once
                s.E[0, 0, 150] = 0.5 * float(s.rhou[0, 0, 0, 150]) ** 2 / float(s.rho[0, 0, 150]) - 1e-3
        else:
            t_end = 0.03
        got = []
        for s, go in ((sols[0], lambda s: s.run(t_end, 500)), (sols[1], lambda s: _one_by_one(s, 500, t_end))):
            try:
                go(s)
                failed = False
            except RuntimeError:
                failed = True
            got.append((failed, s.t, s.iter, s.rho.clone(), s.rhou.clone(), s.E.clone()))
        assert got[0][:3] == got[1][:3] and got[0][0] == kill
        for a, b in zip(got[0][3:], got[1][3:]):
            assert torch.equal(a, b)
