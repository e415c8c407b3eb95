"""Field values that no particle's gather reads never reach the current: a cell that holds no particle
adds nothing, whatever its fields are. A node of empty cells, or the column beyond the right wall that
no routine writes, is NaN in one run and 0 in the other; one step of either gives the same current.

Tolerance: the two runs add the same numbers in an order of their own, at most a few thousand terms a
node: 1e-12 of the largest current value, and in the mixed form (FP32 sums of a cell in a fixed order,
FP64 between cells) the same."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states2d as S
import states3d as S3

pytestmark = pytest.mark.gpu


def _same_current(make, up, np2, cc, uf, at, cells):
    """one step with uf[at] NaN and 0: the currents, and the fields in `cells`"""
    got = []
    for v in (np.nan, 0.0):
        w = uf.copy(order="F")
        w[at] = v
        with make() as sim:
            sim.upload_up(up, np2, cc)
            sim.upload_fields(w)
            sim.step(1)
            got.append((sim.download_current(), sim.download_fields()[cells]))
    (j0, f0), (j1, f1) = got
    assert np.isfinite(j0).all()
    assert np.abs(j0 - j1).max() <= 1e-12 * np.abs(j1).max()
    if f0.size:
        assert np.abs(f0 - f1).max() <= 1e-12 * np.abs(f1).max()


# tiles of 8, 16 and 32 columns; 8 and 16 lanes a cell; the walls leave cells 0, nx-2 and nx-1 empty
@pytest.mark.parametrize("form", ["fast", "mixed"])
@pytest.mark.parametrize("nx, ny, ppc, walls", [(46, 9, 3, True), (47, 5, 70, True), (300, 190, 2, True),
                                                (606, 130, 1, True), (40, 9, 3, False), (40, 5, 120, False)])
def test_empty_cells_2d(nx, ny, ppc, walls, form):
    from wumingpic_amd import MODE_FAST, MODE_MIXED
    from wumingpic_amd.pic2d import Pic2D
    print(nx, ny, ppc, walls, form, flush=True)
    rng = np.random.default_rng(2)
    q, r = S.weibel_consts(ppc)
    p = po.make_params(nx, ny, np_cap=ppc * nx, delt=0.5, q=q, r=r, bc=po.BC_WALLX if walls else po.BC_PERIODIC)
    cnt = np.full((nx, ny), ppc)
    if walls:
        cnt[0] = cnt[-2:] = 0
        at, cells = np.s_[:, nx + 3], np.s_[:, :nx + 3]
    else:
        cnt[17:30] = 0
        at, cells = np.s_[:, 2 + 20], np.s_[:0]
    up, cc, np2 = S.sorted_particles(p, ppc, rng, counts=[cnt, cnt])
    uf = np.asfortranarray(S.random_fields(p, rng, scale=0.02))
    if not walls:
        uf = S.periodic_fill_fields(p, uf)
    _same_current(lambda: Pic2D(nx, ny, list(q), list(r), delt=0.5, bc=p.bc, capacity=int(cnt.sum()),
                                mode=MODE_MIXED if form == "mixed" else MODE_FAST), up, np2, cc, uf, at, cells)


def test_empty_cells_beyond_the_shock_s_edge():
    """the box's active part ends at nxe: what lies in the storage beyond stays there"""
    from wumingpic_amd import MODE_FAST
    from wumingpic_amd.pic2d import Pic2D
    nx, ny, ppc, nxe = 46, 9, 4, 2 + 28
    rng = np.random.default_rng(2)
    q, r = S.weibel_consts(ppc)
    p = po.make_params(nx, ny, np_cap=ppc * nx, delt=0.5, q=q, r=r, bc=po.BC_SHOCK)
    cnt = np.zeros((nx, ny), dtype=int)
    cnt[1:nxe - 3] = ppc
    up, cc, np2 = S.sorted_particles(p, ppc, rng, counts=[cnt, cnt])
    uf = np.asfortranarray(S.random_fields(p, rng, scale=0.02))

    def make():
        sim = Pic2D(nx, ny, list(q), list(r), delt=0.5, bc=p.bc, mode=MODE_FAST, capacity=int(cnt.sum()))
        sim.nxe = nxe
        return sim
    _same_current(make, up, np2, cc, uf, np.s_[:, nxe + 2:], np.s_[:, :nxe])


@pytest.mark.parametrize("form", ["fast", "mixed"])
@pytest.mark.parametrize("ppc", [1, 9])
def test_empty_cells_3d(ppc, form):
    from wumingpic_amd import MODE_FAST, MODE_MIXED
    from wumingpic_amd.pic3d import Pic3D
    nx, ny, nz = 40, 6, 5
    print(ppc, form, flush=True)
    rng = np.random.default_rng(2)
    q, r = S.weibel_consts(ppc)
    p = po.make_params3d(nx, ny, nz, np_cap=ppc * nx, delt=0.5, q=q, r=r)
    cnt = np.full((nx, ny, nz), ppc)
    cnt[17:30] = 0
    up, cc, np2 = S3.sorted_particles3d(p, ppc, rng, counts=[cnt, cnt])
    uf = S3.periodic_fill_fields3d(p, S3.random_fields3d(p, rng, scale=0.02))
    _same_current(lambda: Pic3D(nx, ny, nz, list(q), list(r), delt=0.5, capacity=int(cnt.sum()),
                                mode=MODE_MIXED if form == "mixed" else MODE_FAST),
                  up, np2, cc, uf, np.s_[:, 2 + 20], np.s_[:0])
