"""The IDs' sum and xor of a resident FP64 run between steps, while the IDs lie
as they did when the rows' order became an index: the same as of the IDs handed
in, before and after the rows are put in order, for rows that gain and lose
particles and up to three species."""
import numpy as np
import pytest

from wmhelpers import bits, make_ctx, random_fields, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ppc,vth,nsp", [
    (4, 2, 1, 0.5, 1), (17, 5, 30, 1.0, 2), (66, 4, 90, 0.6, 3), (250, 9, 11, 0.4, 2),
])
def test_ids_are_the_same_set_between_steps(nx, ny, ppc, vth, nsp):
    p, up, np2, cc, uf = state(nx, ny, ppc, 99, vth=vth, nsp=nsp)
    random_fields(uf, 99, amp=0.05)
    # an ID of its own for every slot, so that a wrong one shows
    up[5] = np.random.default_rng(99).integers(1, 2**62, up[5].shape).view(np.float64)
    ids = np.concatenate([bits(up[5, :np2[j, s], j, s]) for s in range(nsp) for j in range(ny)])
    want = (int(np.add.reduce(ids.view(np.uint64))), int(np.bitwise_xor.reduce(ids.view(np.uint64))))
    ctx = make_ctx(p)
    ctx.state_upload(up, np2, cc, uf)
    assert tuple(int(v) for v in ctx.id_checksum()) == want
    for _ in range(3):
        ctx.step(1)
        assert tuple(int(v) for v in ctx.id_checksum()) == want
    n = np.zeros_like(np2)
    ctx.state_download(np2=n)
    assert n.sum() == np2.sum()
    ctx.state_download(up=np.zeros_like(up))
    assert tuple(int(v) for v in ctx.id_checksum()) == want
    ctx.step(2)
    assert tuple(int(v) for v in ctx.id_checksum()) == want
