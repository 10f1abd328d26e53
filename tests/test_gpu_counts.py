"""A resident FP64 state whose row counts and cell index do not belong together:
the push visits the particles of cumcnt's cells, so a row's particles beyond its
last cell (or before its first) get no code for the row order.  The step says so
(WM_ERR_RANGE), every index it forms stays inside the row, and the context goes
on with the next state."""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from oracle import Oracle
from test_gpu_order import _same
from wmhelpers import make_ctx, random_fields, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ppc", [(4, 2, 9), (40, 6, 20), (130, 3, 70)])
@pytest.mark.parametrize("where", ["behind", "before"])
def test_particles_outside_the_cells_are_an_error(nx, ny, ppc, where):
    p, up, np2, cc, uf = state(nx, ny, ppc, 91, vth=0.3)
    random_fields(uf, 91, amp=0.05)
    ctx = make_ctx(p)
    jl, s = ny - 1, 1
    bad = cc.copy(order="F")
    if where == "behind":
        bad[-1, jl, s] -= 3                  # the last cell three short of np2
    else:
        bad[0, jl, s] += 3                   # the first begins three late
    ctx.state_upload(up, np2, bad, uf)
    with pytest.raises(wm.WmError) as e:
        ctx.step(1)
    assert e.value.code == wm.WM_ERR_RANGE
    # a state with the right index steps as ever
    ctx.state_upload(up, np2, cc, uf)
    gp = up.copy(order="F")
    Oracle(p).step(up, gp, uf, cc, np2)
    ctx.step(1)
    _same(p, ctx, up, np2, cc)
