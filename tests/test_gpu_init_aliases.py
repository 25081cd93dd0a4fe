"""HydroSolver.init_from_prim with arrays of the solver's own state: the same start as with copies of them."""

import numpy as np
import pytest
import torch

from heraclespp_amd import Grid, HydroSolver, PerfectGas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given", [("rho", "rho", "rho"), ("E", None, "rho"), ("rho", "rhou", "E"), ("P", "u", "P")])
def test_init_from_arrays_of_the_state(cuda, given):
    grid = Grid(2, (21, 13, 1), 2, "Cartesian", (0.0,) * 3, (1.0,) * 3)
    rng = np.random.default_rng(4)
    rho, P = 0.5 + rng.random(grid.shape3), 0.5 + rng.random(grid.shape3)
    u = rng.uniform(-0.3, 0.3, (2,) + grid.shape3)
    out = []
    for copies in (False, True):
        sol = HydroSolver(grid, PerfectGas(1.4, 1.0), reconstruction="Minmod", riemann_solver="HLLC")
        sol.init_from_prim(rho, u, P)
        sol.E.copy_(2.0 * sol.E)
        args = []
        for name, lead in zip(given, ((), (2,), ())):
            t = torch.as_tensor(u).cuda() if name is None else getattr(sol, name)
            if len(lead) == 1 and t.dim() == 3:  # a scalar field as both velocity components
                t = torch.stack([t, t])
            args.append(t.clone() if copies else t)
        sol.init_from_prim(*args)
        out.append([t.cpu().numpy() for t in (sol.rho, sol.rhou, sol.E, sol.u, sol.P)])
    for name, a, b in zip(("rho", "rhou", "E", "u", "P"), *out):
        np.testing.assert_array_equal(a, b, err_msg=name)
