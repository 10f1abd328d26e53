"""A context's first copies make two pinned buffers, or four on the way down (from
16 MB on one for each 4 MB beyond 8 MB, if that is more), later ones of such arrays
more until eight threads have one each; what they copy is right at every number of
them."""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from wmdebug import XFER_BUFFERS, debug
from wmhelpers import bits, make_ctx, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ppc,first,end", [
    (512, 8, 12, 2, 2),          # 4.5 MB of particles: one thread
    (250, 24, 20, 2, 4),         # 11 MB of particles, then small arrays
    (600, 500, 1, 4, 8),         # 27.5 MB of particles, 14 MB of fields
    (1500, 1203, 1, 8, 8),       # 165 MB
])
def test_buffers_grow_with_the_calls(nx, ny, ppc, first, end):
    p, up, np2, cc, uf = state(nx, ny, ppc, 96, vth=0.2)
    uf[...] = np.random.default_rng(96).normal(size=uf.shape)
    ctx = make_ctx(p, form=wm.FORM_FP64)
    last = 0
    for call in range(5):
        ctx.state_upload(up, np2, cc, uf)
        n = debug(ctx, XFER_BUFFERS)
        assert last <= n <= 8
        if call == 0:
            assert n == first
        last = n
        got = [np.zeros_like(a) for a in (up, np2, cc, uf)]
        ctx.state_download(*got)
        assert np.array_equal(bits(got[3]), bits(uf)) and np.array_equal(got[2], cc)
        for s in range(p["nsp"]):
            for jl in range(0, ny, 7):
                m = np2[jl, s]
                assert np.array_equal(bits(up[:, :m, jl, s]), bits(got[0][:, :m, jl, s]))
    assert last == end
