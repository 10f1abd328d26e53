"""Rows whose cell bins are laid out anew (blocks of cells, then whole rows)
against the same run with room to spare: a row of more particles than a
workgroup holds in registers (12288) and one around that number, blocks above
and below theirs (3072), cells of more than one thread's share of a row, rows
one cell short of a block.

Bins move whole, so each particle's orbit is the same but for the order in
which the deposit's sums run over the bins' lanes: 2e-5, the bar of the other
FP32 tests, for particles matched by ID."""
import numpy as np
import pytest

from test_gpu_fp32 import _by_id, _ctx32
from wmhelpers import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ppc,tight", [(1000, 13, 1.4), (512, 24, 1.2), (100, 60, 1.2),
                                          (1025, 10, 1.5), (63, 20, 1.3)])
def test_relaid_rows_keep_every_particle(nx, ppc, tight):
    p, up, np2, cc, uf = state(nx, 2, ppc, 50, vth=0.2)
    runs = []
    for cap in (int(tight * nx * ppc) // 8 * 8, 5 * nx * ppc):
        ctx = _ctx32(p)
        ctx.set_capacity(cap)
        ctx.state_upload(up, np2, cc, uf)
        ctx.step(5)
        st = ctx.capacity_stats()
        o, n, f = np.zeros_like(up), np.zeros_like(np2), np.zeros_like(uf)
        ctx.state_download(up=o, np2=n, uf=f)
        runs.append((st, _by_id(o, n), f))
        ctx.close()
    (st, a, fa), (_, b, fb) = runs
    assert st["relayouts"] > 0 and st["segment_relayouts"] > 0, st
    assert a.keys() == b.keys() and len(a) == np2.sum()
    assert max(np.abs(a[k] - b[k]).max() for k in a) < 2e-5
    assert np.abs(fa - fb).max() < 1e-3 * np.abs(fb).max()
