"""Moments of a resident FP64 run between steps, while the rows' order is an
index: read through it, bit for bit what the rows put in order give, and that
order is still there for the next step.  Cells of none to many rounds of sixteen
particles, rows and columns one short of and over the 16 x 4 tiles, one to three
species, walls."""
import numpy as np
import pytest

from oracle import BC_RECONNECTION, BC_SHOCK
from wmhelpers import grid_args, make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc,nx,ny,ppc,vth,nsp", [
    (None, 4, 1, 1, 0.3, 1), (None, 15, 3, 15, 0.3, 2), (None, 16, 4, 16, 0.5, 3),
    (None, 17, 5, 33, 0.5, 2), (None, 33, 9, 120, 0.4, 2), (None, 64, 7, 1, 0.5, 3),
    (BC_SHOCK, 20, 5, 30, 0.2, 2), (BC_RECONNECTION, 31, 6, 30, 0.2, 2),
])
def test_moments_through_the_order(bc, nx, ny, ppc, vth, nsp):
    if bc is None:
        p, up, np2, cc, uf = state(nx, ny, ppc, 97, vth=vth, nsp=nsp)
        random_fields(uf, 97, amp=0.05)
        ctx = make_ctx(p)
    else:
        p, up, np2, cc, uf = wall_state(bc, nx, ny, ppc, 97, vth=vth, extra=6)
        ctx = make_wall_ctx(p)
        ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
    ctx.mom_calc__init(*grid_args(p), p["delx"], p["delt"], p["c"], p["q"], p["r"])
    ctx.state_upload(up, np2, cc, uf)
    for _ in range(2):
        ctx.step(1)
        a = ctx.moments()
        b = ctx.moments()
        ctx.state_download(up=np.zeros_like(up))     # the rows in order
        c = ctx.moments()
        assert np.isfinite(a).all() and a[0].max() > 0
        assert np.array_equal(a, b) and np.array_equal(a, c)
