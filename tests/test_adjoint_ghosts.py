"""The part of the reverse step that goes through ghost cells, beyond two ghost layers and with dims
shorter than both ghost regions together, where a cell is the source of ghosts at either end.

* On the CPU: the host build against central finite differences of the oracle's step, one unit
  direction per interior value.
* On the GPU: 3D grids from 2^17 cells on, whose gather leaves that part to a pass over the shell of
  cells that ghosts are filled from, against the host build (which gathers in one pass): the state
  adjoints bit for bit; dL/dgamma, a sum of as many terms of order one as there are cells in
  another order, to 1e-12 of the square root of their number.  One step, and runs of steps whose
  gather overwrites the primitives with the next state's before the shell's pass."""

import ctypes

import numpy as np
import pytest

import heraclespp_amd as H
from heraclespp_amd import _lib
from oracle import oracle as orc
from tests.adjoint_support import Problem, _p, host_lib

PERIODIC, REFLEXIVE, CLAMP = ["Periodic"] * 2, ["Reflexive"] * 2, ["NullGradient"] * 2
MIXED = ["Reflexive", "NullGradient"]
SPH = dict(geom="Spherical", xmin=(0.5, 0.3, 0.0), xmax=(1.5, np.pi - 0.3, 2 * np.pi))


class _Ghosts(Problem):
    """A Problem with ng ghost layers."""

    def __init__(self, n, ng, lim, rs, bc, g=(0.0, 0.0, 0.0), **kw):
        self.layers = ng
        super().__init__(len(n), n, limiter=lim, riemann=rs, bc=bc, g=g, **kw)
        self.ng = ng
        self.nodes = [orc.regular_nodes(self.n[d], ng if d < self.ndim else 0, self.xmin[d], self.xmax[d]) for d in range(3)]

    def oracle(self, gamma):
        return orc.Oracle(self.ndim, self.n, geom=self.geom, limiter=self.limiter, riemann=self.riemann, gamma=gamma, bc=self.bc, g=self.g,
                          xmin=self.xmin, xmax=self.xmax, ng=self.layers)

    def interior(self):
        sl = [slice(None)] * 3
        for d in range(self.ndim):
            sl[2 - d] = slice(self.ng, self.ng + self.n[d])
        return tuple(sl)

    def host_adjoint(self, U, lam_new, dt):
        out = [np.zeros_like(u) for u in U]
        dg = np.zeros(1)
        xs = (ctypes.POINTER(ctypes.c_double) * 3)(*[_p(x) for x in self.nodes])
        bcs = (ctypes.c_int * 6)(*[orc.BCS[b] for b in self.bc] + [0] * (6 - len(self.bc)))
        rc = host_lib().adjh_step(self.ndim, orc.GEOMS[self.geom], orc.SOLVERS[self.riemann], orc.LIMITERS[self.limiter],
                                  (ctypes.c_int * 3)(*self.n), self.ng, xs, bcs, self.gamma, _p(np.array(self.g)), dt,
                                  *[_p(a) for a in (*U, *lam_new, *out)], _p(dg))
        assert rc == 0
        return out, float(dg[0])

    def adjoints(self, seed):
        """Random adjoints of the step's output, zero outside the interior."""
        rng = np.random.default_rng(seed)
        out = []
        for lead in ((), (self.ndim,), ()):
            a = np.zeros(lead + self.o.shape3)
            sub = a[(Ellipsis,) + self.interior()]
            sub[...] = rng.standard_normal(sub.shape)
            out.append(a)
        return out


THIN = [
    ([5], 3, "VanLeer", "HLLC", MIXED),
    ([4], 4, "Minmod", "HLL", PERIODIC),
    ([3, 6], 2, "VanAlbada", "HLLC", REFLEXIVE + CLAMP),
    ([7, 4], 4, "VanLeer", "HLL", MIXED + PERIODIC),
    ([3, 3, 4], 3, "Minmod", "HLLC", PERIODIC + REFLEXIVE + MIXED),
]


@pytest.mark.parametrize("n,ng,lim,rs,bc", THIN)
def test_host_adjoint_of_short_dims_matches_fd(n, ng, lim, rs, bc):
    p = _Ghosts(n, ng, lim, rs, bc, (0.1, -0.2, 0.05))
    U = p.random_state(5)
    dt = p.stable_dt(*U)
    lam_new = p.adjoints(6)
    lam, _ = p.host_adjoint(U, lam_new, dt)
    it, h = p.interior(), 1e-6
    for a, u in enumerate(U):
        for idx in np.ndindex(u[(Ellipsis,) + it].shape):
            ends = []
            for s in (h, -h):
                W = [w.copy() for w in U]
                W[a][(Ellipsis,) + it][idx] += s
                ends.append(sum(np.sum(x * y) for x, y in zip(lam_new, p.step(*W, dt))))
            fd, ad = (ends[0] - ends[1]) / (2 * h), lam[a][(Ellipsis,) + it][idx]
            assert abs(fd - ad) <= 1e-7 * max(1.0, abs(fd)), (a, idx, fd, ad)


LARGE = [
    ("mixed", (52, 51, 50), 2, "VanLeer", "HLLC", PERIODIC + MIXED + ["NullGradient", "Reflexive"], {}),
    ("thin_z", (220, 200, 3), 2, "Minmod", "HLLC", CLAMP + PERIODIC + REFLEXIVE, {}),
    ("thin_x", (3, 211, 210), 2, "VanAlbada", "HLL", PERIODIC + REFLEXIVE + CLAMP, {}),
    ("thin_y_two_cells", (200, 2, 340), 2, "Constant", "HLLC", MIXED + REFLEXIVE + PERIODIC, {}),
    ("three_ghosts", (56, 50, 47), 3, "VanLeer", "HLL", REFLEXIVE + PERIODIC + MIXED, {}),
    ("four_ghosts_thin", (75, 5, 352), 4, "Minmod", "HLLC", PERIODIC + MIXED + REFLEXIVE, {}),
    ("spherical", (64, 47, 45), 2, "VanLeer", "HLLC", MIXED + REFLEXIVE + PERIODIC, SPH),
]


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("name,n,ng,lim,rs,bc,geom", LARGE, ids=[c[0] for c in LARGE])
def test_gather_apart_matches_host_build(cuda, name, n, ng, lim, rs, bc, geom, steps):
    import torch

    assert np.prod(n) >= 1 << 17
    print(f"[adjoint ghosts] {name}, {steps} steps", flush=True)
    g = (-0.1, 0.0, 0.0) if geom else (0.1, -0.2, 0.05)
    p = _Ghosts(list(n), ng, lim, rs, bc, g, **geom)
    states = [p.random_state(20 + k) for k in range(steps)]
    dts = [p.stable_dt(*U) for U in states]
    lam = p.adjoints(30)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    ctx = H.Grid(3, n, ng, p.geom, p.xmin, p.xmax).context(H.PerfectGas(p.gamma, 1.0), H.UniformGravity(g), bc, None, 0, lim, rs, "fp64")
    U = [[dev(a) for a in s] for s in states]
    lams = [[torch.zeros_like(dev(a)) for a in lam] for _ in range(steps)] + [[dev(a) for a in lam]]
    dg = torch.zeros(1, dtype=torch.float64, device="cuda")
    table = lambda rows, v: (ctypes.c_void_p * len(rows))(*[r[v].data_ptr() for r in rows])  # noqa: E731
    ptr = ctypes.c_void_p(dg.data_ptr())
    L = _lib.lib()
    if steps == 1:
        _lib.check(L.hclpp_step_adjoint(ctx.handle, dts[0], *[ctypes.c_void_p(t.data_ptr()) for t in U[0] + lams[1] + lams[0]], ptr))
    else:
        _lib.check(L.hclpp_steps_adjoint(ctx.handle, steps, (ctypes.c_double * steps)(*dts), *[table(U, v) for v in range(3)],
                                         *[table(lams, v) for v in range(3)], ptr))
    torch.cuda.synchronize()
    it, total = p.interior(), 0.0
    for k in range(steps - 1, -1, -1):
        lam, one = p.host_adjoint(states[k], lam, dts[k])
        total += one
        for v, (a, b) in enumerate(zip(lams[k], lam)):
            np.testing.assert_array_equal(a.cpu().numpy()[(Ellipsis,) + it], b[(Ellipsis,) + it], err_msg=f"step {k}, array {v}")
    assert abs(float(dg.cpu()[0]) - total) <= 1e-12 * max(abs(total), steps * np.sqrt(np.prod(n)))
