"""The mass-flux planes between the hydro and the scalar kernel (ndim planes, two or more scalars): held
by contexts whose clock has started only, and done without, at the same results, where the device has no
memory for them."""

import ctypes
import gc

import numpy as np
import pytest
import torch

from heraclespp_amd import Grid, HydroSolver, PerfectGas, _lib
from heraclespp_amd.hydro import Context

pytestmark = pytest.mark.gpu


def _free():
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def _context(n, nfx):
    grid = Grid(3, (n, n, n), 2, "Cartesian", (0.0,) * 3, (1.0,) * 3)
    return grid, Context(grid, PerfectGas(1.4, 1.0), None, None, None, nfx, "Minmod", "HLLC")


def test_a_context_for_operators_holds_no_mass_fluxes(cuda):
    """A context of a grid whose mass fluxes alone exceed the card's memory can be created: the operators
    it serves work on the arrays its user has.  And a small one holds no planes before its clock starts."""
    _context(8, 2)
    n = round((torch.cuda.mem_get_info()[1] / 24) ** (1 / 3)) + 64
    print(f"[scalar memory] context of {n}^3, two scalars", flush=True)
    _context(n, 2)
    before = _free()
    grid, ctx = _context(400, 2)
    assert before - _free() < 8 * np.prod(grid.shape3)


STATE = ("rho", "rhou", "E", "fx")


def _run(n, steps, save):
    """A two-scalar run of n^3 cells through the C interface (no arrays but the two states); whether the
    context took memory for its mass fluxes, and the final state, compared with `save` if given."""
    grid, ctx = _context(n, 2)
    gen = torch.Generator(device="cuda").manual_seed(n)
    states = [[grid.zeros(), grid.zeros(3), grid.zeros(), grid.zeros(2)] for _ in range(2)]
    rho, m, E, fx = states[0]
    for t in (rho, E, fx):
        t.uniform_(0.5, 1.0, generator=gen)
    m.uniform_(-0.2, 0.2, generator=gen)
    E += 1.0
    L, p = _lib.lib(), lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.check(L.hclpp_fill_ghosts(ctx.handle, p(rho), p(m), p(E), p(fx)))
    _lib.check(L.hclpp_set_pressure_fix(ctx.handle, 1, 20.0))
    before = torch.cuda.mem_get_info()[0]
    _lib.check(L.hclpp_clock_start(ctx.handle, 0.0, 0, 1e30, 0.3, steps, p(rho), p(m), p(E)))
    held = before - torch.cuda.mem_get_info()[0]
    print(f"[scalar memory] {held >> 20} MiB taken by the clock start", flush=True)
    took = held > 12 * np.prod(grid.shape3)  # all of their 24 bytes a cell or none: the runtime returns some of its own meanwhile
    _lib.check(L.hclpp_run_steps(ctx.handle, steps, *[p(t) for t in states[0] + states[1]]))
    clk = _lib.Clock()
    _lib.check(L.hclpp_clock_read(ctx.handle, ctypes.byref(clk)))
    assert clk.iter == steps and clk.status == 0
    final = states[steps % 2]
    if save is None:
        return took, [clk.t, clk.dt] + final
    assert [clk.t, clk.dt] == save[:2]
    for name, a, b in zip(STATE, final, save[2:]):
        assert torch.equal(a, b), name
    return took, None


def test_steps_without_memory_for_the_mass_fluxes(cuda):
    """The same run with memory to spare and with less left than the mass fluxes need (which is several
    gigabytes: nothing else in the run comes near the end of the card's memory)."""
    n, steps = 512, 3
    took, save = _run(n, steps, None)
    assert took
    planes = 3 * 8 * (n + 4) ** 3
    state = 2 * 7 * 8 * (n + 4) ** 3
    filler = torch.empty(_free() - state - planes, dtype=torch.uint8, device="cuda")
    try:
        print(f"[scalar memory] {filler.numel() >> 20} MiB set aside, {_free() >> 20} MiB free", flush=True)
        took, _ = _run(n, steps, save)
        assert not took
    finally:
        filler.untyped_storage().resize_(0)  # also where a failure's traceback holds the tensor
        del save
        _free()


def test_steps_captured_before_the_clock_starts(cuda):
    """Two steps recorded in a graph before the context's clock has started, replayed three times with
    other work in between: the six steps of a run."""
    grid = Grid(3, (20, 17, 15), 2, "Cartesian", (0.0,) * 3, (1.0,) * 3)
    rng = np.random.default_rng(2)
    rho, P = 0.5 + rng.random(grid.shape3), 0.5 + rng.random(grid.shape3)
    u, fx = rng.uniform(-0.5, 0.5, (3,) + grid.shape3), rng.random((2,) + grid.shape3)
    sols = [HydroSolver(grid, PerfectGas(1.4, 1.0), reconstruction="Minmod", riemann_solver="HLLC", nfx=2) for _ in range(2)]
    for s in sols:
        s.init_from_prim(rho, u, P, fx=fx)
    a, b = sols[0]._bufs()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        sols[0]._launch_step(a, b)
        sols[0]._launch_step(b, a)
    sols[0].start_clock(1e30, 100)
    sols[1].start_clock(1e30, 100)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for _ in range(2):
            sols[1].step_async()
        clk = sols[1].finish()
        sols[1]._launched, sols[1]._cur0, sols[1]._it0 = 0, sols[1]._cur, sols[1].iter
        mine = sols[0].clock()
        assert (mine.iter, mine.t, mine.dt, mine.status) == (clk.iter, clk.t, clk.dt, 0)
        for name in STATE:
            assert torch.equal(getattr(sols[0], name), getattr(sols[1], name)), name
