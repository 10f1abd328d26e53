"""Momenta whose squares overflow in the resident FP64 push: gamma is infinite,
the velocity zero, the particle stays where it is and its momentum takes half
of the electric kick each side, as the reference's quotients have it
(particle.f90:131-161).  Lanes beside such a particle are as exact as ever.

Orders, counts and IDs exact, particles to 1e-12 (_same), fields to 1e-12 of
their largest value."""
import numpy as np
import pytest

from oracle import BC_RECONNECTION, Oracle
from test_gpu_order import _same
from wmhelpers import make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


def _some_huge(up, np2, nsp, every):
    n = 0
    for s in range(nsp):
        for jl in range(up.shape[2]):
            k = np.arange(0, np2[jl, s], every)
            up[2, k, jl, s] = 1e160 * np.where(k % 2, 1, -1)
            up[3, k[::2], jl, s] = -3e200
            up[4, k[::3], jl, s] = 2e155
            n += k.size
    return n


@pytest.mark.parametrize("nx,ny,ppc,nsp", [(16, 3, 21, 2), (250, 140, 3, 1)])
def test_huge_momenta(nx, ny, ppc, nsp):
    p, up, np2, cc, uf = state(nx, ny, ppc, 93, vth=0.3, nsp=nsp)
    random_fields(uf, 93, amp=0.05)
    assert _some_huge(up, np2, nsp, 5) > 0
    ctx = make_ctx(p)
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    for _ in range(2):
        orc.step(up, gp, uf, cc, np2)
        assert np.isfinite(up[:5, :np2.min()]).all() and np.isfinite(uf).all()
        ctx.step(1)
        ctx.state_download(uf=guf)
        assert np.abs(guf - uf).max() <= 1e-12 * np.abs(uf).max()
    _same(p, ctx, up, np2, cc)


def test_huge_momenta_between_walls():
    p, up, np2, cc, uf = wall_state(BC_RECONNECTION, 24, 3, 30, 94, vth=0.2)
    inner = up[0] > p["nxs"] + 2
    up[3][inner & (np.arange(up.shape[1])[:, None, None] % 7 == 0)] = 1e170
    ctx = make_wall_ctx(p)
    ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    orc.step(up, gp, uf, cc, np2)
    ctx.step(1)
    ctx.state_download(uf=guf)
    assert np.isfinite(uf).all()
    s = slice(p["nxs"] - p["nxgs"] + 2, p["nxe"] - p["nxgs"] + 3)
    assert np.abs(guf - uf)[:, s, 2:-2].max() <= 1e-12 * np.abs(uf[:, s]).max()
    n = np.zeros_like(np2)
    ctx.state_download(np2=n)
    assert np.array_equal(n, np2)
