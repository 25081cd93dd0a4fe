"""The march kernels' tall tile shape (16 x 32 columns, 30 rows of output) on grids whose last tile row holds
a single row of output, so that most of its waves only keep the barriers, against the oracle, bit for bit:
the hydro kernel alone, and the mass fluxes it stores with the scalar kernel that reads them."""

import ctypes

import numpy as np
import pytest

from heraclespp_amd import Grid, HydroSolver, PerfectGas, UniformGravity, _lib
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nfx,riemann,limiter", [((42, 601, 4), 0, "HLLC", "VanLeer"), ((28, 451, 16), 0, "HLL", "Minmod"),
                                                   ((42, 601, 4), 2, "HLLC", "Minmod"), ((28, 451, 16), 5, "Low Mach", "VanAlbada")])
def test_one_row_in_the_last_tile(cuda, n, nfx, riemann, limiter):
    bc = ["Reflexive", "NullGradient", "Reflexive", "NullGradient", "Periodic", "Periodic"]
    g = (0.1, -0.2, -0.3)
    sol = HydroSolver(Grid(3, n, 2, "Cartesian", (0.0,) * 3, (1.0, 0.5, 1.5)), PerfectGas(1.4, 1.0), reconstruction=limiter, riemann_solver=riemann,
                      bc=bc, cfl=0.3, nfx=nfx, gravity=UniformGravity(g))
    seg, blocks, per_cu = ctypes.c_int(), ctypes.c_longlong(), ctypes.c_int()
    _lib.check(_lib.lib().hclpp_fused_plan(sol.ctx.handle, ctypes.byref(seg), ctypes.byref(blocks), ctypes.byref(per_cu)))
    assert n[1] % 30 == 1
    assert blocks.value == -(-n[0] // 14) * -(-n[1] // 30) * -(-n[2] // seg.value), "the plan does not take the tall shape"
    o = orc.Oracle(3, n, limiter=limiter, riemann=riemann, gamma=1.4, bc=bc, xmax=(1.0, 0.5, 1.5), g=g, nfx=nfx)
    rng = np.random.default_rng(9)
    rho, P = 0.5 + rng.random(o.shape3), 0.5 + rng.random(o.shape3)
    u = rng.uniform(-0.6, 0.6, size=(3,) + o.shape3)
    fx = [rng.random((nfx,) + o.shape3)] if nfx else []
    o.init_from_prim(rho, u, P, *fx)
    for _ in range(2):
        o.step(0.3, 1e30, 2)
    sol.init_from_prim(rho, u, P, *fx)
    assert sol.run(1e30, 2) == 2 and sol.t == o.t
    for name in ("rho", "rhou", "E") + (("fx",) if nfx else ()):
        np.testing.assert_array_equal(getattr(sol, name).cpu().numpy(), o.state(name), err_msg=name)
