"""A row of more than 2^31 / 6 particles (its words no longer fit an int) arrives whole: its kinetic
energy is that of the last particle, the only one that moves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_row_of_360_million_particles_is_uploaded_whole():
    from wumingpic_amd.pic2d import Pic2D
    n, u = 360_000_000, 3.0
    up = np.zeros((6, n, 4, 1), order="F")  # 69 GB of address space, pages of zeros but for two records
    up[:, n - 1, 0, 0] = 2.5, 2.5, u, 0.0, 0.0, 0.0
    np2 = np.zeros((4, 1), dtype=np.int32)
    cumcnt = np.zeros((5, 4, 1), dtype=np.int32, order="F")
    np2[0], cumcnt[1:, 0] = n, n
    print("upload", flush=True)
    with Pic2D(4, 4, [1.0], [1.0], nsp=1, capacity=n) as sim:
        sim.upload_up(up, np2, cumcnt)
        print("energy", flush=True)
        e = sim.energy()
    want = np.sqrt(1 + u * u) - 1  # r c^2 (gamma - 1), app.f90:505-519
    assert abs(e[0] - want) <= 1e-12 * want, e
