"""The words that the workgroups of a solve on chip exchange carry a 32-bit tag,
which begins again at 1 when it has been used up.  Words of an earlier solve
that carry the same tags must not pass for the new ones: after a solve of weak
fields that ends in its first exchange, one that begins with the same tag is bit
for bit the one that goes on counting."""
import numpy as np
import pytest

from wmdebug import SOLVE_TAG, debug
from wmhelpers import make_ctx, random_fields, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(256, 64), (600, 40), (1024, 250)])
def test_tags_begin_again(nx, ny):
    p, up, np2, cc, uf = state(nx, ny, 1, 69, vth=0.2)
    random_fields(uf, 69, amp=0.05)
    out = []
    for again in (False, True):
        ctx = make_ctx(p)
        weak = 1e-9 * uf
        ctx.set_cg_tolerance(1e10)
        # nothing moves: no current
        ctx.field__fdtd_i(weak, up, up, cc, p["nxgs"], p["nxge"])
        assert not ctx.cg_iters().any()
        ctx.set_cg_tolerance(1e-6)
        if again:
            assert debug(ctx, SOLVE_TAG) > 1
            debug(ctx, SOLVE_TAG, 0xFFFFFFFF)
        got = uf.copy(order="F")
        ctx.field__fdtd_i(got, up, up, cc, p["nxgs"], p["nxge"])
        out.append((got, ctx.cg_iters().copy()))
    assert np.array_equal(out[0][1], out[1][1]) and out[0][1].all()
    assert np.array_equal(out[0][0], out[1][0])
