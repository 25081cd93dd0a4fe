"""The conversions of grids whose outputs exceed the last-level cache, which are stored past the caches,
against the oracle, bit for bit: ragged rows, over the interior and over all ghosts, nothing written
outside the range."""

import ctypes

import numpy as np
import pytest
import torch

from heraclespp_amd import Grid, PerfectGas, _lib
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd,n", [(1, (16_800_005, 1, 1)), (2, (3361, 3337, 1)), (3, (209, 203, 199))])
def test_streaming_conversions(cuda, nd, n):
    nodes = [np.linspace(0.0, 1.0, n[d] + (5 if d < nd else 1)) for d in range(3)]
    g = Grid(nd, n, 2, nodes=nodes)
    assert (nd + 1) * 8 * np.prod(g.shape3) > 256 << 20
    o = orc.Oracle(nd, n, gamma=1.4, mmw=0.7, nodes=nodes)
    ctx = g.context(PerfectGas(1.4, 0.7))
    gen = torch.Generator(device="cuda").manual_seed(nd)
    rnd = lambda *lead: torch.rand(*lead, *g.shape3, generator=gen, dtype=torch.float64, device="cuda")  # noqa: E731
    rho, u, P = 0.1 + rnd(), rnd(nd) - 0.5, 0.1 + rnd()
    host = [t.cpu().numpy() for t in (rho, u, P)]
    L, p = _lib.lib(), lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    for ngeff in (0, 2):
        r = g.range.with_ghosts(ngeff)._c()
        m, E = torch.full_like(u, -7.0), torch.full_like(P, -7.0)
        _lib.check(L.hclpp_conv_prim_to_cons(ctx.handle, ctypes.byref(r), p(rho), p(u), p(P), p(m), p(E)))
        want = [np.full(t.shape, -7.0) for t in (u, P)]
        o.conv_prim_to_cons(ngeff, *host, *want)
        for name, a, b in zip(("rhou", "E"), (m, E), want):
            assert np.array_equal(a.cpu().numpy(), b), (name, ngeff)
        u2, P2 = torch.full_like(u, -7.0), torch.full_like(P, -7.0)
        _lib.check(L.hclpp_conv_cons_to_prim(ctx.handle, ctypes.byref(r), p(rho), p(m), p(E), p(u2), p(P2)))
        back = [np.full(t.shape, -7.0) for t in (u, P)]
        o.conv_cons_to_prim(ngeff, host[0], *want, *back)
        for name, a, b in zip(("u", "P"), (u2, P2), back):
            assert np.array_equal(a.cpu().numpy(), b), (name, ngeff)
