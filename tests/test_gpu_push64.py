"""The FP64 push that reads its particles through 64-bit offsets, as for species
planes of 4 GB an array and more (2^29 slots): forced on small grids, with
sixteen and eight lanes a cell, periodic and between walls, bit for bit what the
32-bit offsets give."""
import numpy as np
import pytest

from oracle import BC_RECONNECTION, BC_SHOCK, Oracle
from test_gpu_order import _same
from wmdebug import PLANE32, debug
from wmhelpers import make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc,nx,ny,ppc,vth,nsp", [
    (None, 4, 2, 1, 0.5, 1), (None, 9, 2, 17, 1.0, 1), (None, 23, 3, 130, 0.8, 2),
    (None, 66, 4, 40, 0.4, 3), (None, 259, 130, 4, 0.5, 2),
    (BC_SHOCK, 24, 3, 80, 0.3, 2), (BC_RECONNECTION, 24, 3, 80, 0.3, 2),
    (BC_SHOCK, 250, 132, 3, 0.4, 2), (BC_RECONNECTION, 259, 127, 2, 0.6, 2),
])
def test_push_through_64_bit_offsets(bc, nx, ny, ppc, vth, nsp):
    out = []
    for wide in (False, True):
        if bc is None:
            p, up, np2, cc, uf = state(nx, ny, ppc, 95, vth=vth, nsp=nsp)
            random_fields(uf, 95, amp=0.05)
            ctx = make_ctx(p)
        else:
            p, up, np2, cc, uf = wall_state(bc, nx, ny, ppc, 95, vth=vth, extra=6)
            ctx = make_wall_ctx(p)
            ctx.set_walls(p["nxs"], p["nxe"], p["u0"])
        if wide:
            assert debug(ctx, PLANE32, 1) == 1
        else:
            assert debug(ctx, PLANE32) == 1 << 29
        ctx.state_upload(up, np2, cc, uf)
        ctx.step(2)                          # from the slots, then through the order
        orc = Oracle(p)
        gp = up.copy(order="F")
        for _ in range(2):
            orc.step(up, gp, uf, cc, np2)
        if bc is None:
            _same(p, ctx, up, np2, cc)
        g = [np.zeros_like(a) for a in (up, np2, cc, uf)]
        ctx.state_download(*g)
        assert np.array_equal(g[1], np2)
        out.append(g)
    for a, b in zip(*out):
        a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))   # (IDs are no numbers)
