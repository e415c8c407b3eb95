"""The fused 3D step's one-pass exchange and sort where its lists change place: columns whose share
fits a wave's registers, columns with too many stayers or too many arrivals for that, and more leavers
than wait in LDS.  Every cell then holds the oracle's particles, bit for bit as a set."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states3d as S
from test_gpu_parity3d import _cells_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, ppc, u", [(20, 40, 0.3), (20, 100, 1.0), (20, 150, 3.0), (32, 150, 0.1), (30, 220, 2.0)])
def test_columns_match_the_oracle(nx, ppc, u):
    from wumingpic_amd import MODE_FAST
    from wumingpic_amd.pic3d import Pic3D
    rng = np.random.default_rng(11)
    q, r = S.weibel_consts(ppc)
    p = po.make_params3d(nx, 4, 3, np_cap=4 * ppc * nx, delt=0.5, q=q, r=r)
    cnt = rng.poisson(ppc, (2, nx, 4, 3))
    up, cc, np2 = S.sorted_particles3d(p, ppc, rng, u_scale=(u, u), drift=(0.0, 0.3), colocate=False,
                                       counts=list(cnt))
    uf = S.periodic_fill_fields3d(p, S.random_fields3d(p, rng, scale=0.02))
    print(nx, ppc, u, flush=True)
    with Pic3D(nx, 4, 3, list(p.q)[:2], list(p.r)[:2], delt=0.5, mode=MODE_FAST,
               capacity=int(np2.sum(axis=(0, 1)).max())) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        sim.step(1)
        u_dev, n2, c2 = sim.download_up(p.np)
    o = po.Oracle3D(p)
    o.step(up, np.zeros_like(up, order="F"), uf, cc, np2, 1)
    assert np.array_equal(n2, np2) and np.array_equal(c2, cc)
    ok, info = _cells_equal(u_dev, up, np2, cc)
    assert ok, info
