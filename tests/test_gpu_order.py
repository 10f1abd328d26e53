"""The resident FP64 step's row order (particle_y and the sort as an index the
next push reads through) against the oracle, where it can go wrong: the
smallest grids, rows that are no multiple of the kernels' 16 cells, 32-cell
chunks, 64-lane wavefronts or 512-slot chunks, cells with more movers than a
list holds and more displaced particles than a group has lanes, one to three
species, and the state read back after every step or only at the end.

Orders, counts and IDs are exact.  Positions and momenta to 1e-12 of the
oracle's, the bar of the other resident tests: the push contracts FMAs."""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from oracle import Oracle
from wmhelpers import active, bits, make_ctx, random_fields, state

pytestmark = pytest.mark.gpu


def _same(p, ctx, up, np2, cc):
    g = [np.zeros_like(a) for a in (up, np2, cc)]
    ctx.state_download(up=g[0], np2=g[1], cumcnt=g[2])
    assert np.array_equal(g[1], np2) and np.array_equal(g[2], cc)
    for s in range(p["nsp"]):
        for jl in range(p["ny"]):
            n = np2[jl, s]
            assert np.array_equal(bits(up[5, :n, jl, s]), bits(g[0][5, :n, jl, s])), (s, jl)
            assert np.allclose(active(g[0], np2, jl, s), active(up, np2, jl, s), rtol=1e-12,
                               atol=1e-13), (s, jl)


@pytest.mark.parametrize("nx,ny,ppc,vth,nsp,every", [
    (4, 2, 9, 0.5, 2, 1),        # every cell neighbours every other
    (5, 3, 40, 1.0, 1, 1),
    (16, 4, 7, 0.3, 2, 2),
    (17, 2, 120, 1.0, 2, 1),     # many movers a cell: lists flushed, long displaced lists
    (33, 5, 24, 0.4, 3, 3),
    (66, 4, 300, 0.6, 1, 2),     # cells of several windows, rows of 20000 particles
    (250, 3, 11, 0.2, 2, 4),
    (64, 7, 1, 0.5, 2, 4),       # empty cells
])
def test_row_order_matches_oracle(nx, ny, ppc, vth, nsp, every):
    p, up, np2, cc, uf = state(nx, ny, ppc, 71, vth=vth, nsp=nsp)
    random_fields(uf, 71, amp=0.05)
    ctx = make_ctx(p)
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp = up.copy(order="F")
    for it in range(4):
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        if (it + 1) % every == 0:
            _same(p, ctx, up, np2, cc)
            e = ctx.energy()
            assert np.allclose(e, orc.energy(up, uf, np2), rtol=1e-11, atol=1e-18)


def test_moments_and_energy_read_the_pending_order():
    """Energies before the rows are put in order, moments after, then the run
    goes on."""
    p, up, np2, cc, uf = state(40, 9, 20, 72, vth=0.4)
    random_fields(uf, 72, amp=0.05)
    ctx = make_ctx(p)
    g = (p["ndim"], p["np"], p["nsp"], p["nxgs"], p["nxge"], p["nygs"], p["nyge"], p["nys"], p["nye"])
    ctx.mom_calc__init(*g, p["delx"], p["delt"], p["c"], p["q"], p["r"])
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp = up.copy(order="F")
    for _ in range(3):
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        assert np.allclose(ctx.energy(), orc.energy(up, uf, np2), rtol=1e-11, atol=1e-18)
        mom = np.zeros((7, p["nx"] + 2, p["ny"] + 2, p["nsp"]), order="F")
        orc.mom_calc_accl(gp, up, uf, cc)
        orc.mom_calc_nvt(mom, gp, np2)
        orc.bc_mom(mom)
        got = ctx.moments()
        assert np.abs(got - mom).max() <= 1e-12 * np.abs(mom).max()
        assert np.allclose(ctx.energy(), orc.energy(up, uf, np2), rtol=1e-11, atol=1e-18)
    _same(p, ctx, up, np2, cc)
