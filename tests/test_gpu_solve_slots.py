"""The contexts of a process share the device's CUs for the field solves on
chip: a solve that finds too many taken streams instead of waiting for ever, one
that fails to launch gives back what it took, and contexts of several threads
step side by side.  Fields to 1e-12 of the largest value, the bar of the other
field tests; the same iterations."""
import threading
import time

import numpy as np
import pytest

import wumingpic2d_amd as wm
from oracle import Oracle
from wmdebug import SOLVE_FAILS, SOLVE_SLOTS, debug
from wmhelpers import make_ctx, random_fields, state

pytestmark = pytest.mark.gpu


def _solver(nx, ny, seed):
    p, up, np2, cc, uf = state(nx, ny, 1, seed, vth=0.3)
    random_fields(uf, seed, amp=0.02)
    orc = Oracle(p)
    gp = np.zeros_like(up)
    orc.particle__solv(gp, up, uf, cc)
    a, b = uf.copy(order="F"), uf.copy(order="F")
    ctx = make_ctx(p)

    def same():
        orc.field__fdtd_i(a, up, gp, cc)
        ctx.field__fdtd_i(b, up, gp, cc, p["nxgs"], p["nxge"])
        assert np.array_equal(orc.cg_iters(), ctx.cg_iters())
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()

    def fails():
        with pytest.raises(wm.WmError) as e:
            ctx.field__fdtd_i(b.copy(order="F"), up, gp, cc, p["nxgs"], p["nxge"])
        assert e.value.code == wm.WM_ERR_HIP

    return ctx, same, fails


@pytest.mark.parametrize("nx,ny", [(130, 33), (64, 12)])
def test_a_solve_that_finds_no_room_streams(nx, ny):
    ctx, same, _ = _solver(nx, ny, 61)
    same()
    assert debug(ctx, SOLVE_SLOTS) == 0
    debug(ctx, SOLVE_SLOTS, 4096)
    t = time.monotonic()
    try:
        same()
    finally:
        assert debug(ctx, SOLVE_SLOTS, -4096) == 0
    assert time.monotonic() - t < 20.0
    same()
    assert debug(ctx, SOLVE_SLOTS) == 0


def test_a_failed_launch_holds_nothing():
    ctx, same, fails = _solver(130, 33, 62)
    same()
    debug(ctx, SOLVE_FAILS, 1)
    fails()
    assert debug(ctx, SOLVE_SLOTS) == 0
    same()


def test_a_failed_step_holds_nothing():
    p, up, np2, cc, uf = state(40, 9, 6, 63, vth=0.3)
    random_fields(uf, 63)
    ctx = make_ctx(p)
    ctx.state_upload(up, np2, cc, uf)
    debug(ctx, SOLVE_FAILS, 1)
    with pytest.raises(wm.WmError) as e:
        ctx.step(1)
    assert e.value.code == wm.WM_ERR_HIP and debug(ctx, SOLVE_SLOTS) == 0


def test_two_contexts_step_in_two_threads():
    """1024 x 250: 192 of the 256 CUs each, so they take turns."""
    runs = []
    for seed in (64, 65):
        p, up, np2, cc, uf = state(1024, 250, 1, seed, vth=0.3)
        random_fields(uf, seed, amp=0.02)
        ctx = make_ctx(p)
        ctx.state_upload(up, np2, cc, uf)
        runs.append((p, up, np2, cc, uf, ctx))
    out = [None, None]

    def go(k):
        try:
            for _ in range(10):
                runs[k][5].step(2)
        except Exception as e:              # noqa: BLE001 (handed to the test)
            out[k] = e

    t = [threading.Thread(target=go, args=(k,)) for k in range(2)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert out == [None, None]
    for p, up, np2, cc, uf, ctx in runs:
        alone = make_ctx(p)
        alone.state_upload(up, np2, cc, uf)
        alone.step(20)
        a, b = np.zeros_like(uf), np.zeros_like(uf)
        alone.state_download(uf=a)
        ctx.state_download(uf=b)
        assert np.array_equal(a, b)
        assert debug(ctx, SOLVE_SLOTS) == 0
