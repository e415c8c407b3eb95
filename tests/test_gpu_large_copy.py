"""Downloads on both sides of the size from which several threads move them, with a last chunk that is
not full: every value comes back as it was uploaded, into a new array and again into another."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(500, 300), (900, 1001), (64, 50, 40), (101, 90, 80)], ids=str)
def test_download_returns_what_was_uploaded(shape):
    from wumingpic_amd.pic2d import Pic2D
    from wumingpic_amd.pic3d import Pic3D
    print(shape, flush=True)
    rng = np.random.default_rng(1)
    make = Pic2D if len(shape) == 2 else Pic3D
    with make(*shape, [1.0, -1.0], [25.0, 1.0], capacity=16) as sim:
        uf = np.asfortranarray(rng.standard_normal((6, *(n + 4 for n in shape))))
        sim.upload_fields(uf)
        for _ in range(2):
            assert np.array_equal(sim.download_fields(), uf)
        mom = np.asfortranarray(rng.standard_normal((7, *(n + 2 for n in shape), 2)))
        sim.upload_mom(mom)
        assert np.array_equal(sim.download_mom(), mom)
