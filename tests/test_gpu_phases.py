"""What the step's phases enclose, by bounds from the bytes a phase cannot do
without: cell-centred fields no shorter than their kernel's bytes at 20 TB/s,
more than any memory of the card gives; and the first stream's phases no further
short of the time of the call than the field update's least time, its bytes at 8
TB/s."""
import time

import numpy as np
import pytest

import wumingpic2d_amd as wm
from wumingpic2d_amd import weibel
from wmhelpers import make_ctx

pytestmark = pytest.mark.gpu


def _run(form, n, ppc, tol, steps):
    p = weibel.grid_params(n, n, ppc)
    ctx = make_ctx(p, form=form)
    ctx.init_weibel(98, ppc, 0.05, 0.5)
    ctx.set_cg_tolerance(tol)
    ctx.step(3)
    ctx.step(steps)
    return ctx


@pytest.mark.parametrize("form,write", [(wm.FORM_FP64, 8), (wm.FORM_FP32, 4)])
def test_the_first_phase_holds_the_cell_fields(form, write):
    """1925 workgroups, all on the chip at once: the phase ends with the kernel,
    not with the start of its last workgroup."""
    n, steps = 700, 10
    ctx = _run(form, n, 8, 1e-6, steps)
    ms = ctx.phase_times()[0] / steps
    assert ms * 1e-3 >= 6 * n * n * (8 + write) / 20e12


def test_the_field_phase_holds_the_update():
    """FP32, few particles, a solve that is content with what it begins with: the
    update reads and writes 12 planes and reads 6 more."""
    n, steps = 2048, 10
    ctx = _run(wm.FORM_FP32, n, 8, 1e10, steps)
    assert not ctx.cg_iters().any()
    short = []
    for _ in range(20):
        t = time.perf_counter()
        ctx.step(steps)
        short.append(((time.perf_counter() - t) - ctx.phase_times()[:4].sum() * 1e-3) / steps)
    assert 0.0 < min(short) < 18 * 8 * n * n / 8e12


def test_the_field_phase_of_one_row():
    """One row: the update is a chain of kernels, with nothing to solve."""
    p = weibel.grid_params(256, 1, 16)
    ctx = make_ctx(p)
    ctx.init_weibel(98, 16, 0.05, 0.5)
    ctx.set_cg_tolerance(1e10)
    ctx.step(3)
    ctx.step(10)
    a = ctx.phase_times()
    # the solve's two launches (12 us), six kernels no shorter than 1 us each
    assert (a[:6] >= 0).all() and 0.06 <= a[3] < 10.0
