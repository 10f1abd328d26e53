"""Current folding, implicit solve and field update against the oracle, at the
sizes where their tilings can go wrong: the smallest grids, one tile of each
shape exactly full and one cell over, last tiles one row or two columns thick,
each tile height and each number of components solved side by side, and a grid
with more tiles than the chip holds at once, which streams.

The same iterations, and fields to 1e-12 of the largest value, the bar of the
other field tests: the solve stops at a relative residual of 1e-6 after the
same iterates, whose rounding differs by sums of at most 1.3e6 terms in
another order (sqrt(1.3e6) * 1.1e-16 = 1.3e-13)."""
import numpy as np
import pytest

from oracle import BC_RECONNECTION, BC_SHOCK, Oracle
from wmhelpers import make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [
    (4, 1), (4, 2), (5, 3), (7, 5),
    (128, 16), (128, 17), (128, 64), (128, 65),       # one tile of 128 columns, then more
    (129, 8), (256, 32), (256, 33), (130, 33),        # 256 columns
    (257, 4), (512, 16), (512, 17), (513, 4),         # 512 columns
    (250, 61), (1024, 250), (1030, 500),              # 4, 8 and 16 rows a lane
    (2050, 300), (2050, 600),                         # two components at a time, one
    (4, 16400),                                       # 257 tiles: streamed
])
def test_fdtd_i_over_tile_edges(nx, ny):
    p, up, np2, cc, uf = state(nx, ny, 1, 51, vth=0.3)
    random_fields(uf, 51, amp=0.02)
    orc = Oracle(p)
    gp = np.zeros_like(up)
    orc.particle__solv(gp, up, uf, cc)
    a, b = uf.copy(order="F"), uf.copy(order="F")
    ctx = make_ctx(p)
    for it in range(2):                    # the second starts from the first's change
        orc.field__fdtd_i(a, up, gp, cc)
        ctx.field__fdtd_i(b, up, gp, cc, p["nxgs"], p["nxge"])
        assert np.array_equal(orc.cg_iters(), ctx.cg_iters()), it
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max(), it


@pytest.mark.parametrize("bc", [BC_SHOCK, BC_RECONNECTION])
@pytest.mark.parametrize("nx,ny", [(24, 2), (127, 64), (140, 40), (520, 9), (260, 130)])
def test_wall_steps_over_tile_edges(bc, nx, ny):
    p, up, np2, cc, uf = wall_state(bc, nx, ny, 2, 52, vth=0.15, extra=6)
    uf[2] = np.random.default_rng(52).normal(0, 0.05, uf.shape[1:])
    orc = Oracle(p)
    ctx = make_wall_ctx(p)
    ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
    ctx.state_upload(up, np2, cc, uf)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    for it in range(2):
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        ctx.state_download(uf=guf)
        assert np.array_equal(orc.cg_iters(), ctx.cg_iters()), it
        s = slice(p["nxs"] - p["nxgs"] + 2, p["nxe"] - p["nxgs"] + 3)
        assert np.abs(guf - uf)[:, s, 2:-2].max() <= 1e-12 * np.abs(uf[:, s]).max(), it
