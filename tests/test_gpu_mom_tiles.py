"""The fused moment pass at the edges of its tiles (16 cells x 4 rows) and of a
cell's rounds of sixteen particles, both forms, against the oracle on the same
state.

Bar: 1e-12 of each moment's largest magnitude.  A node takes at most 4 cells of
40 particles; each term's weight, velocity and gathered field carry a few
roundings of 1.1e-16, and 160 additions of positive weights add at most as many
units in the last place of the sum, so the difference stays below 1e-13 of it.
"""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from oracle import Oracle
from wmhelpers import grid_args, make_ctx, state

pytestmark = pytest.mark.gpu


def _ragged(nx, ny, ppc, seed):
    """Cells of 0 to ppc particles, some rows empty, rows sorted by cell."""
    p, up, np2, cc, uf = state(nx, ny, ppc, seed, vth=0.3, np_cap=nx * (2 * ppc + 16))
    rng = np.random.default_rng(seed)
    uf += rng.normal(scale=0.1, size=uf.shape)
    for s in range(p["nsp"]):
        for jl in range(ny):
            keep = []
            for i in range(nx):
                lo, hi = cc[i, jl, s], cc[i + 1, jl, s]
                n = 0 if jl % 5 == 4 else int(rng.integers(0, hi - lo + 1))
                keep.extend(range(lo, lo + n))
            new = np.array([sum(k < cc[i, jl, s] for k in keep) for i in range(nx + 1)])
            up[:, :len(keep), jl, s] = up[:, keep, jl, s]
            np2[jl, s] = len(keep)
            cc[:, jl, s] = new
    return p, up, np2, cc, uf


@pytest.mark.parametrize("form", [wm.FORM_FP64, wm.FORM_FP32])
@pytest.mark.parametrize("nx,ny,ppc", [(15, 3, 1), (16, 4, 16), (17, 5, 17), (33, 9, 40),
                                       (4, 1, 15)])
def test_moments_at_tile_edges(form, nx, ny, ppc):
    p, up, np2, cc, uf = _ragged(nx, ny, ppc, 31 + nx)
    if form == wm.FORM_FP64:
        ctx = make_ctx(p)
    else:
        ctx = wm.Context(0)
        ctx.set_form(form)
        g = grid_args(p)
        ctx.boundary_periodic__init(*g, 0, 0, 0, 0, 0, 0, [0], p["delx"], p["delt"], p["c"])
        ctx.particle__init(*g, p["delx"], p["delt"], p["c"], p["q"], p["r"])
        ctx.field__init(*g, 0, 0, 0, 0, p["delx"], p["delt"], p["c"], p["q"], p["r"], p["gfac"])
        ctx.sort__init(*g)
    ctx.mom_calc__init(*grid_args(p), p["delx"], p["delt"], p["c"], p["q"], p["r"])
    ctx.state_upload(up, np2, cc, uf)
    got = ctx.moments()
    gup, gnp2 = np.zeros_like(up), np.zeros_like(np2)
    gcc, guf = np.zeros_like(cc), np.zeros_like(uf)
    ctx.state_download(up=gup, np2=gnp2, cumcnt=gcc, uf=guf)
    assert np.array_equal(gnp2, np2)
    orc = Oracle(p)
    gp = np.zeros_like(up)
    orc.mom_calc_accl(gp, gup, guf, gcc)
    want = np.zeros((7, nx + 2, ny + 2, p["nsp"]), order="F")
    orc.mom_calc_nvt(want, gp, gnp2)
    orc.bc_mom(want)
    for s in range(p["nsp"]):
        for k in range(7):
            scale = max(np.abs(want[k, ..., s]).max(), 1e-300)
            assert np.abs(got[k, ..., s] - want[k, ..., s]).max() <= 1e-12 * scale, (s, k)
