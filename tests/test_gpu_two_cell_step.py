"""Steps at c delt = delx, the longest a context accepts: a particle near c can round across two cell
faces at once (x = 4 - 2^-51 to 5 in FP64; an offset of 1 - 2^-24 by 1 in FP32). Its current is the
reference's weights for that step (field.f90:244-266, smo with |inc| = 2), as for any other.

The FP64 push has the oracle's bits, so the oracle's own push gives the same crossings; in the mixed
form the oracle deposits the positions that the step left. Tolerances: 1e-12 of the largest current
(sums in another order), 1e-5 in the mixed form (every term rounded to FP32)."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states2d as S
import states3d as S3

pytestmark = pytest.mark.gpu

U = np.array([3e4, 1e6, 3e8, 1e9, 4e12])


def _state(dim, n, ppc, mixed, seed=9):
    rng = np.random.default_rng(seed)
    q, r = S.weibel_consts(ppc)
    if dim == 2:
        p = po.make_params(*n, np_cap=2 * ppc * n[0], delt=1.0, q=q, r=r)
        up, cc, np2 = S.sorted_particles(p, ppc, rng, u_scale=(0.3, 0.3), colocate=False)
        uf, o = np.zeros((6, n[0] + 4, n[1] + 4), order="F"), po.Oracle2D(p)
    else:
        p = po.make_params3d(*n, np_cap=2 * ppc * n[0], delt=1.0, q=q, r=r)
        up, cc, np2 = S3.sorted_particles3d(p, ppc, rng, u_scale=(0.3, 0.3), colocate=False)
        uf, o = np.zeros((6, *(m + 4 for m in n)), order="F"), po.Oracle3D(p)
    flat = up.reshape(up.shape[0], -1, order="F")
    cell = np.floor(flat[0])
    # half of them at the cell's right edge and near c along x; they start and end inside the box
    fast = (rng.random(cell.size) < 0.5) & (cell >= 3) & (cell < n[0] - 3)
    edge = cell + np.float64(np.float32(1) - np.float32(2.0 ** -24)) if mixed else np.nextafter(cell + 1, 0)
    if mixed:  # positions that an FP32 offset holds
        flat[:dim] = np.floor(flat[:dim]) + np.float32(0.25)
    flat[0] = np.where(fast, edge, flat[0])
    u = rng.choice(U, cell.size) * (1 + 0.1 * rng.random(cell.size))
    for d, v in enumerate((u, 0 * u, 0 * u + 1)):
        flat[dim + d] = np.where(fast, v, 0.3 * flat[dim + d])
    up[:] = flat.reshape(up.shape, order="F")
    return p, q, r, up, cc, np2, uf, o


# (the 3D mixed form reports such a step instead, test below)
@pytest.mark.parametrize("dim, n, ppc, form", [
    *((2, (40, 6), ppc, form) for ppc in (5, 120) for form in ("fast", "vay", "mixed")),
    (3, (40, 6, 5), 5, "fast"), (3, (40, 6, 5), 5, "vay")])
def test_current_of_a_step_over_two_cells(dim, n, ppc, form):
    from wumingpic_amd import MODE_FAST, MODE_MIXED
    from wumingpic_amd._lib import PUSHER_VAY
    from wumingpic_amd.pic2d import Pic2D
    from wumingpic_amd.pic3d import Pic3D
    print(dim, n, ppc, form, flush=True)
    mixed = form == "mixed"
    p, q, r, up, cc, np2, uf, o = _state(dim, n, ppc, mixed)
    gp = np.zeros_like(up, order="F")
    if form == "vay":
        o.particle_solv_vay(gp, up, uf, cc)
    else:
        o.particle_solv(gp, up, uf, cc)
    with (Pic2D if dim == 2 else Pic3D)(*n, list(q), list(r), delt=1.0, capacity=int(np2.sum()),
                                        mode=MODE_MIXED if mixed else MODE_FAST) as sim:
        if form == "vay":
            sim.set_pusher(PUSHER_VAY)
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        sim.step(1)
        got = sim.download_current()
        if mixed:  # gp as the step left it, back in the old slots, y unwrapped
            new, _, _ = sim.download_up(p.np)
            a, b = (v.reshape(6, -1, order="F") for v in (up, new))
            ia, ib = (np.argsort(v[5].view(np.int64), kind="stable") for v in (a, b))
            g = gp.reshape(6, -1, order="F")
            g[:, ia] = b[:, ib]
            g[1] -= n[1] * np.rint((g[1] - a[1]) / n[1])
            g[0] -= n[0] * np.rint((g[0] - a[0]) / n[0])
            gp = np.asfortranarray(g.reshape(up.shape, order="F"))
    inc = np.trunc(gp[0]) - np.trunc(up[0])
    assert (inc == 2).sum() >= 3, np.unique(inc, return_counts=True)
    uj = np.zeros_like(got, order="F")
    o.ele_cur(uj, up, gp, cc)
    o.bc_curre(uj)
    assert np.abs(got - uj).max() <= (1e-5 if mixed else 1e-12) * np.abs(uj).max()


def test_3d_mixed_reports_a_step_over_two_cells():
    from wumingpic_amd import MODE_MIXED
    from wumingpic_amd._lib import WpicError
    from wumingpic_amd.pic3d import Pic3D
    n = (40, 6, 5)
    p, q, r, up, cc, np2, uf, o = _state(3, n, 5, True)
    with Pic3D(*n, list(q), list(r), delt=1.0, capacity=int(np2.sum()), mode=MODE_MIXED) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        with pytest.raises(WpicError):
            sim.step(1)
