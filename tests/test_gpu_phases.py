"""What the step's phases enclose, by bounds from the bytes a phase cannot do
without: cell-centred fields no shorter than their kernel's bytes at 20 TB/s,
more than any memory of the card gives."""
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
