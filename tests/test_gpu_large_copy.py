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


def test_download_into_pinned_memory_goes_straight_there():
    """an array the link can write to itself needs no slots and no threads"""
    import ctypes as C
    import os
    import threading

    from wumingpic_amd._lib import check, lib
    from wumingpic_amd.pic3d import Pic3D
    shape = (160, 144, 128)
    n = tuple(v + 4 for v in shape)
    uf = np.asfortranarray(np.random.default_rng(2).standard_normal((6, *n)))
    pinned = C.c_void_p()  # from the HIP runtime that the library itself uses
    assert lib().hipHostMalloc(C.byref(pinned), C.c_size_t(uf.nbytes), C.c_uint(0)) == 0
    a = np.ctypeslib.as_array((C.c_double * uf.size).from_address(pinned.value)).reshape(uf.shape, order="F")
    a[:] = 0.0
    most, done = [0], threading.Event()

    def watch():
        while not done.is_set():
            most[0] = max(most[0], len(os.listdir("/proc/self/task")))

    with Pic3D(*shape, [1.0, -1.0], [25.0, 1.0], capacity=16) as sim:
        sim.upload_fields(uf)
        check(sim._L.wpic_download_fields3d(sim._h, a))
        assert np.array_equal(a, uf)
        before = len(os.listdir("/proc/self/task"))
        t = threading.Thread(target=watch)
        t.start()
        for _ in range(5):
            a[:] = 0.0
            check(sim._L.wpic_download_fields3d(sim._h, a))
            assert np.array_equal(a, uf)
        done.set()
        t.join()
    del a
    assert lib().hipHostFree(pinned) == 0
    assert most[0] <= before + 1  # the watcher
