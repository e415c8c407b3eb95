"""The fast 3D push and deposit over the shapes that tell its tiles apart: whole and ragged 8x4x4
tiles, cells with fewer particles than lanes, empty and crowded ones, one to four species, momenta that
send many particles across faces, edges and corners, the FP64 form, the mixed one and the push alone,
against the oracle after one step.

Tolerances: the FP64 current is the oracle's sums in another order, at most a few thousand terms a
node, so 1e-12 of the largest field value; the mixed form rounds its inputs and every term to FP32
(6e-8 each), 1e-5 of the largest."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states3d as S

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, nz, particles per cell and species, species
    (4, 4, 4, 3, 2), (9, 5, 5, 9, 1), (17, 6, 4, 20, 2), (8, 4, 9, 40, 4), (13, 11, 10, 2, 3),
]


def _state(nx, ny, nz, ppc, nsp, seed=7):
    rng = np.random.default_rng(seed)
    q, r = S.weibel_consts(ppc)
    q, r = np.resize(q, nsp), np.resize(r, nsp)
    p = po.make_params3d(nx, ny, nz, nsp=nsp, np_cap=4 * ppc * nx + 64, delt=0.5, q=q, r=r)
    cnt = rng.poisson(ppc, (nsp, nx, ny, nz))
    cnt[:, rng.random((nx, ny, nz)) < 0.1] = 0
    up, cc, np2 = S.sorted_particles3d(p, ppc, rng, u_scale=(0.3,) * nsp, drift=(0.4,) * nsp, colocate=False,
                                       counts=list(cnt))
    return p, up, cc, np2, S.periodic_fill_fields3d(p, S.random_fields3d(p, rng, scale=0.05))


@pytest.mark.parametrize("form", ["fast", "mixed", "push"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
def test_one_step_matches_the_oracle(case, form):
    from wumingpic_amd import MODE_FAST, MODE_MIXED
    from wumingpic_amd.pic3d import Pic3D
    nx, ny, nz, _, nsp = case
    p, up, cc, np2, uf = _state(*case)
    print(case, form, flush=True)
    mode = MODE_MIXED if form == "mixed" else MODE_FAST
    o = po.Oracle3D(p)
    gp = np.zeros_like(up, order="F")
    with Pic3D(nx, ny, nz, list(p.q)[:nsp], list(p.r)[:nsp], nsp=nsp, delt=0.5, mode=mode,
               capacity=max(1, int(np2.sum(axis=(0, 1)).max()))) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        if form == "push":
            sim.particle_solv()
            got, n2 = sim.download_gp(p.np)
            o.particle_solv(gp, up, uf, cc)
            assert np.array_equal(n2, np2)
            for s in range(nsp):
                for k in range(nz):
                    for j in range(ny):
                        n = np2[j, k, s]
                        assert np.array_equal(got[:, :n, j, k, s].view(np.int64), gp[:, :n, j, k, s].view(np.int64))
            return
        sim.step(1)
        got = sim.download_fields()
        _, n2, c2 = sim.download_up(p.np)
    o.step(up, gp, uf, cc, np2, 1)
    tol = 1e-5 if form == "mixed" else 1e-12
    assert np.abs(got - uf).max() <= tol * np.abs(uf).max()
    if form != "mixed":  # FP32 rounding may move a particle across a cell edge
        assert np.array_equal(n2, np2) and np.array_equal(c2, cc)
