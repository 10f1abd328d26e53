"""A field solve on chip whose workgroups do not meet gives up: the update behind
it is skipped, the host solves again by the streaming solver, the solves after
it stream, a thousand the first time and twice as many each further time, and
then the chip is used again.  Forced from the host: the waits' bound is zero, so
every workgroup ends at once or comes to its end.

The second solve may start from a part of the first's result, so fields agree as
far as both are solved: to a relative residual of 1e-13.  The operator's
eigenvalues lie in [t^2, t^2 + 8], t^2 = (1 / (0.5 * 0.501))^2 = 15.9, so a
solution is off by at most 1e-13 * 23.9 / 15.9 of its 2-norm, two of them by
3e-13, the largest cell by sqrt(n) of that, a change by at most twice the largest
field; delta E takes at most four of delta B's cells times 0.25.  With 1e-12 for
rounding, per step: (6e-13 sqrt(n) + 1e-12) of the largest value."""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from oracle import BC_RECONNECTION, BC_SHOCK, Oracle
from wmdebug import SOLVE_GIVES_UP, SOLVE_REST, SOLVE_SLOTS, debug
from wmhelpers import make_ctx, make_wall_ctx, random_fields, state, wall_state

pytestmark = pytest.mark.gpu


class _Run:
    def __init__(self, bc, nx, ny, fcg=False):
        if bc is None:
            self.p, self.up, self.np2, self.cc, self.uf = state(nx, ny, 4, 66, vth=0.2)
            random_fields(self.uf, 66, amp=0.05)
            self.ctx = make_ctx(self.p)
            self.cols = slice(2, -2)
        else:
            self.p, self.up, self.np2, self.cc, self.uf = wall_state(bc, nx, ny, 4, 66, vth=0.15,
                                                                     extra=6)
            self.uf[2] = np.random.default_rng(66).normal(0, 0.05, self.uf.shape[1:])
            self.ctx = make_wall_ctx(self.p)
            self.ctx.set_walls(self.p["nxs"], self.p["nxe"], self.p["u0"])
            self.cols = slice(self.p["nxs"] - self.p["nxgs"] + 2, self.p["nxe"] - self.p["nxgs"] + 3)
        self.ctx.set_cg_tolerance(1e-13)
        self.orc = Oracle(self.p)
        self.orc.set_cg_err(1e-13)
        self.ctx.state_upload(self.up, self.np2, self.cc, self.uf)
        if fcg:
            self.ctx.pc_init(0)
            self.ctx.set_solver(wm.SOLVER_FCG)
        self.gp, self.guf, self.steps = self.up.copy(order="F"), np.zeros_like(self.uf), 0

    def step(self, gives_up=False, counts=False):
        self.orc.step(self.up, self.gp, self.uf, self.cc, self.np2)
        if gives_up:
            debug(self.ctx, SOLVE_GIVES_UP, 1)
        self.ctx.step(1)
        self.steps += 1
        assert debug(self.ctx, SOLVE_SLOTS) == 0
        self.ctx.state_download(uf=self.guf)
        a, b = self.guf[:, self.cols, 2:-2], self.uf[:, self.cols, 2:-2]
        n = self.p["nx"] * self.p["ny"]
        assert np.abs(a - b).max() <= self.steps * (6e-13 * n ** 0.5 + 1e-12) * np.abs(b).max()

    def rest(self, value=0):
        return debug(self.ctx, SOLVE_REST, value)


@pytest.mark.parametrize("bc,nx,ny,fcg", [
    (None, 130, 33, False), (None, 600, 40, False),      # workgroups side by side
    (None, 64, 12, False),                               # one a component
    (None, 600, 1, False), (None, 60, 1, False),         # one row: the separate update
    (None, 136, 40, True),
    (BC_SHOCK, 140, 40, False), (BC_RECONNECTION, 140, 40, False), (BC_RECONNECTION, 24, 5, False),
])
def test_a_solve_that_gives_up_is_streamed(bc, nx, ny, fcg):
    r = _Run(bc, nx, ny, fcg)
    r.step()
    assert r.rest() == 0
    r.step(gives_up=True)
    assert r.rest() == 1000
    for k in range(3):
        r.step()
        assert r.rest() == 999 - k
    r.rest(-1)                               # the chip again
    r.step()
    assert r.rest() == 0
    r.step(gives_up=True)
    assert r.rest() == 2000
    r.rest(-1)
    r.step()
    n = np.zeros_like(r.np2)
    r.ctx.state_download(np2=n)
    assert np.array_equal(n, r.np2)


def test_the_host_array_solve_gives_up():
    p, up, np2, cc, uf = state(130, 33, 1, 67, vth=0.3)
    random_fields(uf, 67, amp=0.02)
    orc = Oracle(p)
    orc.set_cg_err(1e-13)
    gp = np.zeros_like(up)
    orc.particle__solv(gp, up, uf, cc)
    a, b = uf.copy(order="F"), uf.copy(order="F")
    ctx = make_ctx(p)
    ctx.set_cg_tolerance(1e-13)
    for it in range(3):
        orc.field__fdtd_i(a, up, gp, cc)
        debug(ctx, SOLVE_GIVES_UP, int(it == 1))
        ctx.field__fdtd_i(b, up, gp, cc, p["nxgs"], p["nxge"])
        assert np.abs(a - b).max() <= (it + 1) * (6e-13 * 4290 ** 0.5 + 1e-12) * np.abs(a).max()
    assert debug(ctx, SOLVE_REST) == 999 and debug(ctx, SOLVE_SLOTS) == 0


@pytest.mark.parametrize("nx,ny", [(130, 33), (64, 12)])
def test_an_unsolved_step_leaves_the_fields(nx, ny):
    """ite_max reached on chip: the error the streaming solver gives, and the
    fields as they were."""
    p, up, np2, cc, uf = state(nx, ny, 4, 68, vth=0.2)
    random_fields(uf, 68)
    ctx = make_ctx(p)
    ctx.set_cg_tolerance(1e-300)
    ctx.state_upload(up, np2, cc, uf)
    with pytest.raises(wm.WmError) as e:
        ctx.step(1)
    assert e.value.code == wm.WM_ERR_CG_ITEMAX and debug(ctx, SOLVE_SLOTS) == 0
    got = np.zeros_like(uf)
    ctx.state_download(uf=got)
    assert np.array_equal(got, uf)
