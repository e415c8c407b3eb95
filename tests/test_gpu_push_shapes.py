"""The fast 2D push and deposit over the shapes its launch rules tell apart: tiles of 32, 16 and 8
columns with ragged edges, 8 and 16 lanes a cell, empty and crowded cells, one to four species, each
boundary kind, the two fused forms and the separate routines, against the oracle after one step.

Tolerances: the FP64 current is the oracle's sums in another order, at most a few thousand terms a
node, so 1e-12 of the largest field value; the mixed form rounds its inputs and every term to FP32
(6e-8 each), 1e-5 of the largest."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states2d as S

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, particles per cell and species, species, walls
    (4, 4, 3, 2, False), (9, 5, 1, 1, False), (33, 6, 70, 2, False), (65, 43, 5, 2, True), (47, 4, 30, 4, False),
    (40, 21, 60, 2, True), (300, 190, 3, 2, False), (601, 40, 2, 3, True),
]


def _state(nx, ny, ppc, nsp, walls, seed=5):
    rng = np.random.default_rng(seed)
    q, r = S.weibel_consts(ppc)
    q, r = np.resize(q, nsp), np.resize(r, nsp)
    p = po.make_params(nx, ny, nsp=nsp, np_cap=4 * ppc * nx + 64, delt=0.5, q=q, r=r,
                       bc=po.BC_WALLX if walls else po.BC_PERIODIC)
    cnt = rng.poisson(ppc, (nsp, nx, ny))
    cnt[:, rng.random((nx, ny)) < 0.1] = 0
    if walls:
        cnt[:, 0] = cnt[:, -2:] = 0
    up, cc, np2 = S.sorted_particles(p, ppc, rng, u_scale=(0.3,) * nsp, drift=(0.4,) * nsp, colocate=False,
                                     counts=list(cnt))
    uf = S.random_fields(p, rng, scale=0.05)
    if not walls:
        uf = S.periodic_fill_fields(p, uf)
    return p, up, np2, cc, np.asfortranarray(uf)


@pytest.mark.parametrize("form", ["fast", "mixed", "routines"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(int(v)) for v in c))
def test_one_step_matches_the_oracle(case, form):
    from wumingpic_amd import MODE_FAST, MODE_MIXED
    from wumingpic_amd.pic2d import Pic2D
    nx, ny, _, nsp, walls = case
    p, up, np2, cc, uf = _state(*case)
    print(case, form, flush=True)
    mode = MODE_MIXED if form == "mixed" else MODE_FAST
    with Pic2D(nx, ny, list(p.q)[:nsp], list(p.r)[:nsp], nsp=nsp, delt=0.5, bc=p.bc, mode=mode,
               capacity=max(1, int(np2.sum(axis=0).max()))) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        if form == "routines":
            sim.particle_solv()
            if walls:
                sim.bc_particle_x()
            sim.field_fdtd_i()
            if not walls:
                sim.bc_particle_x()
            sim.bc_particle_y()
            sim.sort_bucket()
        else:
            sim.step(1)
        got = sim.download_fields()
        _, n2, c2 = sim.download_up(p.np)
    o = po.Oracle2D(p)
    gp = np.zeros_like(up, order="F")
    o.step(up, gp, uf, cc, np2, 1)
    tol = 1e-5 if form == "mixed" else 1e-12
    assert np.abs(got - uf).max() <= tol * np.abs(uf).max()
    if form != "mixed":  # FP32 rounding may move a particle across a cell edge
        assert np.array_equal(n2, np2) and np.array_equal(c2, cc)
