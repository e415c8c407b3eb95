"""The fast field solve over the shapes its kernels' work splits tell apart: strips of 64 columns (2D)
and tiles of 32x8 columns (3D), whole, ragged and narrower than one; one row or level a unit and
several; the periodic box and the walls, against the oracle.

Tolerance: the device adds the same numbers as the oracle in another order, at most 2e5 terms a dot
product, which moves the solution by a few 1e-15 an iteration: 1e-12 of the largest value."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states2d as S
import states3d as S3

pytestmark = pytest.mark.gpu


def _check(sim, o, p, up, cc, np2, uf):
    gp = np.zeros_like(up, order="F")
    o.particle_solv(gp, up, uf, cc)
    with sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        for _ in range(2):  # the second solve starts from the first one's increments and iteration count
            sim.particle_solv()
            got_it = sim.field_fdtd_i()
            it = o.field_fdtd_i(uf, up, gp, cc)
            assert tuple(got_it) == tuple(it)
            got = sim.download_fields()
            assert np.abs(got - uf).max() <= 1e-12 * np.abs(uf).max()
            assert np.abs(sim.download_dfield() - o.df).max() <= 1e-12 * np.abs(o.df).max()
            o.particle_solv(gp, up, uf, cc)


@pytest.mark.parametrize("nx, ny, walls", [(4, 4, False), (63, 5, False), (64, 7, True), (65, 6, False),
                                           (129, 31, True), (130, 1500, False), (70, 2100, True)])
def test_field_solve_2d(nx, ny, walls):
    from wumingpic_amd import MODE_FAST
    from wumingpic_amd.pic2d import Pic2D
    rng = np.random.default_rng(3)
    q, r = S.weibel_consts(1)
    p = po.make_params(nx, ny, np_cap=4 * nx + 16, delt=0.5, q=q, r=r, bc=po.BC_WALLX if walls else po.BC_PERIODIC)
    cnt = np.ones((nx, ny), dtype=int)
    cnt[0] = cnt[-2:] = 0
    up, cc, np2 = S.sorted_particles(p, 1, rng, counts=[cnt, cnt])
    uf = S.random_fields(p, rng, scale=0.02)
    if not walls:
        uf = S.periodic_fill_fields(p, uf)
    print(nx, ny, walls, flush=True)
    sim = Pic2D(nx, ny, list(p.q)[:2], list(p.r)[:2], delt=0.5, bc=p.bc, mode=MODE_FAST, capacity=nx * ny)
    _check(sim, po.Oracle2D(p), p, up, cc, np2, np.asfortranarray(uf))


@pytest.mark.parametrize("nx, ny, nz", [(4, 3, 3), (32, 8, 5), (33, 9, 6), (31, 17, 4), (33, 130, 64)])
def test_field_solve_3d(nx, ny, nz):
    from wumingpic_amd import MODE_FAST
    from wumingpic_amd.pic3d import Pic3D
    rng = np.random.default_rng(4)
    q, r = S.weibel_consts(1)
    p = po.make_params3d(nx, ny, nz, np_cap=4 * nx + 16, delt=0.5, q=q, r=r)
    up, cc, np2 = S3.sorted_particles3d(p, 1, rng)
    uf = S3.periodic_fill_fields3d(p, S3.random_fields3d(p, rng, scale=0.02))
    print(nx, ny, nz, flush=True)
    sim = Pic3D(nx, ny, nz, list(p.q)[:2], list(p.r)[:2], delt=0.5, mode=MODE_FAST, capacity=nx * ny * nz)
    _check(sim, po.Oracle3D(p), p, up, cc, np2, uf)


@pytest.mark.parametrize("n", [(64, 66000), (1056, 520, 3)], ids=["4125 strips", "2145 tiles"])
def test_field_solve_with_more_work_units_than_blocks(n):
    """each block (2D: wave) takes several units; no particles, so the fields alone drive the solve.
    The oracle adds 4.2e6 terms one after another, about sqrt(4.2e6) 1e-16 off per dot product and
    some ten iterations of two: 1e-11 of the largest value."""
    from wumingpic_amd import MODE_FAST
    from wumingpic_amd.pic2d import Pic2D
    from wumingpic_amd.pic3d import Pic3D
    rng = np.random.default_rng(5)
    q, r = S.weibel_consts(1)
    print(n, flush=True)
    if len(n) == 2:
        p = po.make_params(*n, np_cap=1, delt=0.5, q=q, r=r)
        o, (up, gp, _, cc, np2) = po.Oracle2D(p), po.alloc_state(p)
        uf = np.asfortranarray(S.periodic_fill_fields(p, S.random_fields(p, rng, scale=0.02)))
    else:
        p = po.make_params3d(*n, np_cap=1, delt=0.5, q=q, r=r)
        o, (up, gp, _, cc, np2) = po.Oracle3D(p), po.alloc_state3d(p)
        uf = S3.periodic_fill_fields3d(p, S3.random_fields3d(p, rng, scale=0.02))
    with (Pic2D if len(n) == 2 else Pic3D)(*n, list(q), list(r), delt=0.5, mode=MODE_FAST, capacity=1) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        for _ in range(2):
            sim.particle_solv()
            assert tuple(sim.field_fdtd_i()) == tuple(o.field_fdtd_i(uf, up, gp, cc))
            got = sim.download_dfield()
            assert np.abs(got - o.df).max() <= 1e-11 * np.abs(o.df).max()
            assert np.abs(sim.download_fields() - uf).max() <= 1e-11 * np.abs(uf).max()


@pytest.mark.parametrize("n", [(4, 4), (8, 8), (5, 13), (15, 17), (16, 16), (4, 65), (37, 31), (4, 4, 4), (5, 5, 5),
                               (4, 8, 8), (7, 9, 11)], ids=lambda n: "x".join(map(str, n)))
def test_parity_solve_is_bit_exact(n):
    """the parity mode's serial sums, taken 256 elements at a time: fewer than 64, whole chunks, remainders"""
    from wumingpic_amd import MODE_PARITY
    from wumingpic_amd.pic2d import Pic2D
    from wumingpic_amd.pic3d import Pic3D
    rng = np.random.default_rng(6)
    q, r = S.weibel_consts(2)
    if len(n) == 2:
        p = po.make_params(*n, np_cap=8 * n[0], delt=0.5, q=q, r=r)
        o, (up, cc, np2) = po.Oracle2D(p), S.sorted_particles(p, 2, rng)
        uf = np.asfortranarray(S.periodic_fill_fields(p, S.random_fields(p, rng, scale=0.02)))
    else:
        p = po.make_params3d(*n, np_cap=8 * n[0], delt=0.5, q=q, r=r)
        o, (up, cc, np2) = po.Oracle3D(p), S3.sorted_particles3d(p, 2, rng)
        uf = S3.periodic_fill_fields3d(p, S3.random_fields3d(p, rng, scale=0.02))
    gp = np.zeros_like(up, order="F")
    o.particle_solv(gp, up, uf, cc)
    print(n, flush=True)
    with (Pic2D if len(n) == 2 else Pic3D)(*n, list(q), list(r), delt=0.5, mode=MODE_PARITY,
                                           capacity=int(np2.sum())) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        sim.particle_solv()
        assert tuple(sim.field_fdtd_i()) == tuple(o.field_fdtd_i(uf, up, gp, cc))
        assert np.array_equal(sim.download_dfield().view(np.int64), o.df.copy(order="F").view(np.int64))
        assert np.array_equal(sim.download_fields().view(np.int64), uf.view(np.int64))
