"""Launch shapes of the sweeps: the one that is reported, and what a search may
choose."""
import pytest

from bamrex_amd.level import Level, make_params

from conftest import announce
from test_gpu_shapes import smooth_level

pytestmark = pytest.mark.gpu


def level(n, box):
    lay, U = smooth_level((n, n), box)
    lev = Level(make_params(2, 1.4, 1.0, limiter="minbee"), lay, [0, 0], [n - 1, n - 1],
                ["periodic"] * 2, ["periodic"] * 2)
    lev.set_state(U)
    return lev


@pytest.mark.parametrize("n,box", [(64, 32), (256, 64)])
def test_reported_shape_is_the_one_in_use(n, box):
    """A level without a shape of its own sweeps in segments chosen by its
    size, short ones while SIMDs would be idle; what is read is that length, so
    that a caller who changes another field keeps it."""
    announce("reported shape %d^2" % n)
    lev = level(n, box)
    try:
        t = lev.get_tuning()
        assert t["seg_k"] < 8
        lev.set_tuning(block_x=128)
        assert lev.get_tuning() == dict(t, block_x=128)
        lev.set_tuning(seg_k=24)
        assert lev.get_tuning() == dict(t, block_x=128, seg_k=24)
    finally:
        lev.close()


def test_autotune_of_a_small_level_finds_short_segments():
    """256^2 cells: one cell per lane (the length used without a shape) sweeps
    in 9.7 us against 21.4 for 8, once the shortest length that was searched."""
    announce("autotune 256^2")
    lev = level(256, 64)
    try:
        lev.autotune([1 / 256, 1 / 256], 1e-4)
        assert lev.get_tuning()["seg_k"] < 8
    finally:
        lev.close()
