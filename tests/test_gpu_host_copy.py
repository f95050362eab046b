"""State vectors to the device and back through the ring of pinned blocks
(host_copy.cpp): sizes below the direct limit of 8 MB, past it within and beyond the ring of 12
blocks of 1 MB (converted by the calling thread), and past 32 MB (by worker
threads), none a whole number of blocks.
FP64 comes back bit for bit, FP32 as the rounded values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import dgtd_amd as D  # noqa: E402


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("cells", [4, 19, 20, 23, 27, 31, 40])  # 144 cells^3 unknowns: 0.07 to 74 MB on the host
def test_state_round_trip(cells, precision):
    vx, E, bc = D.cube_mesh(cells, 1.0, "pec")
    op = D.HesthavenEvolution(vx, E, bc, 1, precision=precision, kernel="valu")
    rng = np.random.default_rng(cells)
    for _ in range(2):  # the second transfer reuses the ring
        x = rng.standard_normal(op.ndofs)
        op.set_state(x)
        want = x if precision == 64 else x.astype(np.float32).astype(np.float64)
        assert np.array_equal(op.get_state(), want)


def test_batch_instance_state():
    vx, E, bc = D.cube_mesh(24, 1.0, "pec")
    b = D.Batch(precision=32, max_instances=1)
    x = np.random.default_rng(1).standard_normal(24 * E.shape[0])
    i = b.add(vx, E, bc, 1, x0=x, final_time=1.0)
    assert np.array_equal(b.get_state(i), x.astype(np.float32).astype(np.float64))
    b.close()
