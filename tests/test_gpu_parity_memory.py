"""The vectors that only the parity mode's solve uses (A p; in 3D also b) are made with its first
step, like its per-cell current blocks: a context of another mode holds none of them."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def _free_bytes(L):
    free, total = C.c_size_t(), C.c_size_t()
    assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


# cells; doubles a cell: the deposit's blocks, then the solve's vectors
@pytest.mark.parametrize("n, block, vectors", [((1024, 1024), 65, 3), ((128, 128, 64), 300, 6)], ids=["2d", "3d"])
def test_parity_mode_s_own_memory(n, block, vectors):
    from wumingpic_amd import MODE_FAST, MODE_PARITY
    from wumingpic_amd._lib import lib
    from wumingpic_amd.pic2d import Pic2D
    from wumingpic_amd.pic3d import Pic3D
    cells = 1024 * 1024
    with (Pic2D if len(n) == 2 else Pic3D)(*n, [1.0, -1.0], [25.0, 1.0], capacity=16, mode=MODE_FAST) as sim:
        sim.step(1)
        fast = _free_bytes(lib())
        sim.set_mode(MODE_PARITY)
        sim.step(1)
        got = fast - _free_bytes(lib())
        want = 8 * cells * (block + vectors)
        assert abs(got - want) <= 8 << 20, (got, want)  # the allocator's granularity
        sim.set_mode(MODE_FAST)
        sim.step(1)
