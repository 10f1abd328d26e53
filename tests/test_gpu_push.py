"""The resident FP64 push, its movers' sums and the row order at the sizes
where their splits can go wrong: rows one cell short of and over the push's
8-cell tiles, one to three species, cells with no, one, and many more movers
than a list holds at a time (47) or a round takes (16), odd and even numbers of
16-particle steps, cells longer than the order's tables (512 slots), and cells
that receive more displaced particles than are ranked at a time (64).

Orders, counts and IDs are exact; particles to 1e-12 as in the other resident
tests, fields to 1e-12 of their largest value: a cell's current sums at most
a few thousand terms of its size in another order (5e3 * 1.1e-16 = 6e-13)."""
import numpy as np
import pytest

from oracle import BC_RECONNECTION, BC_SHOCK, Oracle
from test_gpu_order import _same
from wmhelpers import make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ppc,vth,nsp", [
    (4, 2, 1, 0.5, 1), (7, 3, 15, 0.05, 2), (8, 2, 16, 0.3, 2), (9, 2, 17, 1.0, 1),
    (15, 3, 31, 0.3, 3), (16, 2, 33, 2.0, 2), (17, 2, 48, 0.0, 2), (23, 2, 130, 1.0, 1),
    (6, 3, 700, 0.8, 1), (5, 2, 1100, 3.0, 2),
])
def test_push_and_order_over_tile_edges(nx, ny, ppc, vth, nsp):
    p, up, np2, cc, uf = state(nx, ny, ppc, 81, vth=vth, nsp=nsp)
    random_fields(uf, 81, amp=0.05)
    ctx = make_ctx(p)
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    for _ in range(3):                       # from slots, then through the order
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        ctx.state_download(uf=guf)
        assert np.abs(guf - uf).max() <= 1e-12 * np.abs(uf).max()
    _same(p, ctx, up, np2, cc)


@pytest.mark.parametrize("bc", [BC_SHOCK, BC_RECONNECTION])
@pytest.mark.parametrize("nx,ny,ppc,vth", [(9, 2, 33, 0.6), (24, 3, 80, 0.3)])
def test_walled_push_over_tile_edges(bc, nx, ny, ppc, vth):
    p, up, np2, cc, uf = wall_state(bc, nx, ny, ppc, 82, vth=vth, extra=6)
    ctx = make_wall_ctx(p)
    ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    s = slice(p["nxs"] - p["nxgs"] + 2, p["nxe"] - p["nxgs"] + 3)
    for _ in range(2):
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        ctx.state_download(uf=guf)
        assert np.abs(guf - uf)[:, s, 2:-2].max() <= 1e-12 * np.abs(uf[:, s]).max()
    n = np.zeros_like(np2)
    ctx.state_download(np2=n)
    assert np.array_equal(n, np2)


@pytest.mark.parametrize("nx,ny,ppc,vth,nsp,bc", [
    (4099, 9, 30, 1.0, 1, None),            # lists filled over and over, three wraps of 8 cells
    (193, 170, 1, 0.5, 3, None),            # odd and even cells of a row, empty ones
    (250, 132, 3, 0.4, 2, BC_SHOCK), (259, 127, 2, 0.6, 2, BC_RECONNECTION),
])
def test_push_with_eight_lanes_a_cell(nx, ny, ppc, vth, nsp, bc):
    """More than 32768 cells of at most 36 particles a species: eight lanes a
    cell, two cells' movers in each row of sixteen."""
    if bc is None:
        p, up, np2, cc, uf = state(nx, ny, ppc, 83, vth=vth, nsp=nsp)
        random_fields(uf, 83, amp=0.05)
        ctx = make_ctx(p)
        s = slice(2, -2)
    else:
        p, up, np2, cc, uf = wall_state(bc, nx, ny, ppc, 83, vth=vth, extra=6)
        ctx = make_wall_ctx(p)
        ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
        s = slice(p["nxs"] - p["nxgs"] + 2, p["nxe"] - p["nxgs"] + 3)
    assert p["nx"] * ny > 32768
    ctx.state_upload(up, np2, cc, uf)
    orc = Oracle(p)
    gp, guf = up.copy(order="F"), np.zeros_like(uf)
    for _ in range(2):
        orc.step(up, gp, uf, cc, np2)
        ctx.step(1)
        ctx.state_download(uf=guf)
        assert np.abs(guf - uf)[:, s, 2:-2].max() <= 1e-12 * np.abs(uf[:, s]).max()
    if bc is None:
        _same(p, ctx, up, np2, cc)
