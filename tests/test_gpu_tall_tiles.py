"""The march kernels' second tile shape (16 x 32 columns, 3D FP64) against the oracle, bit for bit, on
grids whose launch plan takes it: a last tile row that is full or ragged; scalars and the
pressure fix in it; and the fast arithmetic."""

import ctypes

import numpy as np
import pytest

from heraclespp_amd import Grid, HydroSolver, PerfectGas, UniformGravity, _lib
from oracle import oracle as orc
from tests.helpers import rel_l1

pytestmark = pytest.mark.gpu

CASES = [
    ((70, 30, 90), "Cartesian", 0, "HLLC", "Minmod"),
    ((60, 29, 100), "Cartesian", 0, "HLL", "VanLeer"),
    ((160, 60, 60), "Spherical", 2, "HLLC", "Minmod"),
    ((96, 200, 64), "Cartesian", 3, "Low Mach", "VanAlbada"),
]


def _solver(n, geom, nfx, riemann, limiter, **kw):
    lo, hi = ((0.3, 0.6, 0.1), (1.0, 2.4, 2.0)) if geom == "Spherical" else ((0.0,) * 3, (1.0, 0.5, 1.5))
    bc = ["Reflexive", "NullGradient", "Periodic", "Periodic", "Reflexive", "NullGradient"]
    g = (0.1, -0.2, -0.3)
    sol = HydroSolver(Grid(3, n, 2, geom, lo, hi), PerfectGas(1.4, 1.0), reconstruction=limiter, riemann_solver=riemann, bc=bc, cfl=0.3, nfx=nfx,
                      gravity=UniformGravity(g), **kw)
    occ = [ctypes.c_int(), ctypes.c_longlong(), ctypes.c_int()]
    _lib.check(_lib.lib().hclpp_fused_plan(sol.ctx.handle, *[ctypes.byref(v) for v in occ]))
    assert occ[2].value == 1, "the plan does not take the tall shape"
    o = orc.Oracle(3, n, geom=geom, limiter=limiter, riemann=riemann, gamma=1.4, bc=bc, xmin=lo, xmax=hi, g=g, nfx=nfx)
    rng = np.random.default_rng(7)
    rho, P = 0.5 + rng.random(o.shape3), 0.5 + rng.random(o.shape3)
    u = rng.uniform(-0.6, 0.6, size=(3,) + o.shape3)
    return sol, o, rho, u, P, (rng.random((nfx,) + o.shape3) if nfx else None)


@pytest.mark.parametrize("n,geom,nfx,riemann,limiter", CASES)
def test_tall_tiles_match_oracle(cuda, n, geom, nfx, riemann, limiter):
    sol, o, rho, u, P, fx = _solver(n, geom, nfx, riemann, limiter)
    o.init_from_prim(rho, u, P, fx) if nfx else o.init_from_prim(rho, u, P)
    for _ in range(2):
        o.step(0.3, 1e30, 2)
    sol.init_from_prim(rho, u, P, fx=fx)
    assert sol.run(1e30, 2) == 2 and sol.t == o.t
    for name in ("rho", "rhou", "E") + (("fx",) if nfx else ()):
        np.testing.assert_array_equal(getattr(sol, name).cpu().numpy(), o.state(name), err_msg=name)


def test_pressure_fix_and_fast_arithmetic_in_tall_tiles(cuda):
    """The fix follows the march kernel's workgroups: fused and operator runs agree bit for bit (eps large
    enough that it acts in most tiles).  The fast arithmetic: close to the reference arithmetic."""
    n, geom, _, riemann, limiter = CASES[2]
    sol, _, rho, u, P, fx = _solver(n, geom, 2, riemann, limiter, pressure_fix="On", eps_pf=4.0)
    out = []
    for s in (sol, HydroSolver(sol.grid, sol.eos, reconstruction=limiter, riemann_solver=riemann, bc=sol.ctx.bc, cfl=0.3, nfx=2,
                               gravity=sol.gravity, pressure_fix="On", eps_pf=4.0, fused=False)):
        s.init_from_prim(rho, u, P, fx=fx)
        assert s.run(1e30, 2) == 2
        out.append([t.cpu().numpy() for t in (s.rho, s.rhou, s.E, s.fx)])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    fast, o, rho, u, P, _ = _solver(*CASES[0], arithmetic="fast")
    fast.init_from_prim(rho, u, P)
    assert fast.run(1e30, 2) == 2
    o.init_from_prim(rho, u, P)
    for _ in range(2):
        o.step(0.3, 1e30, 2)
    for name in ("rho", "rhou", "E"):
        assert rel_l1(getattr(fast, name).cpu().numpy(), o.state(name)) <= 1e-13, name
