"""Momenta whose Lorentz factor has a significand of all ones (u = sqrt(3): 1 + u*u = 4 - 2^-51, root
2 - 2^-52), where 1/gamma lies just above the middle of two doubles: the pushes keep the reference's
bits there. With B = 0 the final 1/gamma is such a number, with E = 0 and B not also the kick's own."""
import numpy as np
import pytest

from oracle import pyoracle as po
import states2d as S
import states3d as S3

pytestmark = pytest.mark.gpu


def _corner_momenta():
    """doubles u with the significand of sqrt(fl(1 + fl(u u))) all ones"""
    out = []
    for n in range(2, 12):
        u = np.sqrt(4.0 ** n - 1.0) if n > 1 else np.sqrt(3.0)
        v = u.view(np.int64) + np.arange(-40, 41)
        out.append(v.view(np.float64))
    out.append((np.sqrt(3.0).view(np.int64) + np.arange(-40, 41)).view(np.float64))
    u = np.concatenate(out)
    root = np.sqrt(1.0 + u * u)
    u = u[(root.view(np.int64) & 0xFFFFFFFFFFFFF) == 0xFFFFFFFFFFFFF]
    assert u.size and np.any(np.abs(u - np.sqrt(3.0)) < 1e-15)
    return u


def _bits(a, dim, n):
    """positions and momenta (mom_calc__accl writes no ids)"""
    return np.ascontiguousarray(a[:dim + 3, :n]).view(np.int64)


@pytest.mark.parametrize("b", [0.0, 0.3])
@pytest.mark.parametrize("dim", [2, 3])
def test_push_keeps_the_reference_s_bits(dim, b):
    u = _corner_momenta()
    rng = np.random.default_rng(6)
    print(dim, b, u.size, flush=True)
    ppc, n = 6, (12, 5) if dim == 2 else (12, 5, 4)
    if dim == 2:
        from wumingpic_amd.pic2d import Pic2D as Pic
        q, r = S.weibel_consts(ppc)
        p = po.make_params(*n, np_cap=ppc * n[0], delt=0.5, q=q, r=r)
        up, cc, np2 = S.sorted_particles(p, ppc, rng)
        o, uf = po.Oracle2D(p), np.zeros((6, n[0] + 4, n[1] + 4), order="F")
    else:
        from wumingpic_amd.pic3d import Pic3D as Pic
        q, r = S.weibel_consts(ppc)
        p = po.make_params3d(*n, np_cap=ppc * n[0], delt=0.5, q=q, r=r)
        up, cc, np2 = S3.sorted_particles3d(p, ppc, rng)
        o, uf = po.Oracle3D(p), np.zeros((6, n[0] + 4, n[1] + 4, n[2] + 4), order="F")
    axis = rng.integers(0, 3, up.shape[1:])
    for d in range(3):
        v = rng.choice(u, up.shape[1:]) * rng.choice([-1.0, 1.0], up.shape[1:])
        up[dim + d] = np.where(axis == d, v, 0.0)
    uf[:3] = b
    gp = np.zeros_like(up, order="F")
    o.particle_solv(gp, up, uf, cc)
    acc = np.zeros_like(up, order="F")
    o.mom_accl(acc, up, uf, cc)
    with Pic(*n, list(q), list(r), delt=0.5, capacity=int(np2.sum())) as sim:
        sim.upload_up(up, np2, cc)
        sim.upload_fields(uf)
        sim.particle_solv()
        got, _ = sim.download_gp(p.np)
        assert np.array_equal(_bits(got, dim, ppc * n[0]), _bits(gp, dim, ppc * n[0]))
        sim.upload_up(up, np2, cc)
        sim.mom_accl()
        got, _ = sim.download_gp(p.np)
        assert np.array_equal(_bits(got, dim, ppc * n[0]), _bits(acc, dim, ppc * n[0]))
