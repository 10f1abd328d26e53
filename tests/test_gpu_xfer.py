"""Host arrays to and from the device at the sizes where the copies' split can
go wrong: states below and above one piece, rows longer than a piece (4 MB),
rows without particles, and rows of one particle.  What comes back is what
went in, bit for bit, and nothing else in the arrays changes."""
import numpy as np
import pytest

import wumingpic2d_amd as wm
from wmhelpers import bits, make_ctx, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ppc,form", [
    (4, 2, 1, wm.FORM_FP64), (64, 37, 9, wm.FORM_FP64), (300, 50, 40, wm.FORM_FP64),
    (64, 2, 1500, wm.FORM_FP64), (301, 51, 40, wm.FORM_FP32),
])
def test_states_come_back_as_they_went(nx, ny, ppc, form):
    p, up, np2, cc, uf = state(nx, ny, ppc, 91)
    if ny > 2:                               # a row without particles, one of a single one
        np2[1, 0], np2[2, 0] = 0, 1
        cc[:, 1, 0] = 0
        cc[:, 2, 0] = np.arange(nx + 1) > int(up[0, 0, 2, 0]) - p["nxgs"]
    uf[...] = np.random.default_rng(91).normal(size=uf.shape)
    ctx = make_ctx(p, form=form)
    ctx.state_upload(up, np2, cc, uf)
    got = [np.full_like(a, 7) for a in (up, np2, cc, uf)]
    ctx.state_download(*got)
    assert np.array_equal(got[1], np2) and np.array_equal(got[2], cc)
    assert np.array_equal(bits(got[3]), bits(uf))
    for s in range(p["nsp"]):
        for jl in range(ny):
            n = np2[jl, s]
            a, b = up[:, :n, jl, s], got[0][:, :n, jl, s]
            if form == wm.FORM_FP64:
                assert np.array_equal(bits(a), bits(b)), (s, jl)
            else:
                assert np.array_equal(bits(a[5]), bits(b[5])) and (np.abs(a[:5] - b[:5]) < 2e-6).all(), (s, jl)
            assert (got[0][:, n:, jl, s] == 7).all(), (s, jl)


def test_ids_of_the_whole_capacity_follow_the_push():
    """particle__solv copies component 6 beyond the rows' counts too, and
    writes nothing else there."""
    p, up, np2, cc, uf = state(200, 40, 12, 92)
    rng = np.random.default_rng(92)
    for s in range(p["nsp"]):
        for jl in range(p["ny"]):
            up[5, np2[jl, s]:, jl, s] = rng.normal(size=p["np"] - np2[jl, s])
    gp = np.full_like(up, 7)
    ctx = make_ctx(p)
    ctx.particle__solv(gp, up, uf, cc, p["nxgs"], p["nxge"])
    assert np.array_equal(bits(gp[5]), bits(up[5]))
    for s in range(p["nsp"]):
        for jl in range(p["ny"]):
            assert (gp[:5, np2[jl, s]:, jl, s] == 7).all()
