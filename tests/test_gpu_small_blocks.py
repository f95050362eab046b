"""The per-node stage's small element blocks (meshes of at most one such block
per compute unit) against the oracle and the matrix-core stage: one element, a
block and its neighbours, the last mesh that takes them and the first that does
not.

Bars as in test_gpu_parity.py: FP64 1e-12 of the largest entry (another order
of the same sums), FP32 1e-5 relative L2.
"""
import numpy as np
import pytest

import meshgen as MG
from oracle import oracle as O

pytestmark = pytest.mark.gpu

import dgtd_amd as D  # noqa: E402


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("edge", ["one", "block", "block+1", "last", "first"])
def test_small_blocks(order, edge):
    nodes = (order + 1) * (order + 2) * (order + 3) // 6
    block = 128 // nodes
    most = block * 256  # compute units
    K = {"one": 1, "block": block, "block+1": block + 1, "last": most, "first": most + 1}[edge]
    n = int(np.ceil((K / 6) ** (1 / 3)))
    vx, E, fbc = MG.cube_mesh(n, 1.0, ["pec", "pmc", "sma", "pec", "pmc", "sma"])
    E, fbc = E[:K], fbc[:K]
    eps = np.random.default_rng(order).uniform(1, 4, K)
    ref = O.Operator(vx, E, fbc, order, eps=eps)
    x = np.random.default_rng(K).standard_normal(ref.ndofs)
    yr = ref.mult(x)
    gpu = D.HesthavenEvolution(vx, E, fbc, order, eps=eps, precision=64, kernel="valu")
    assert np.abs(gpu.mult(x) - yr).max() <= 1e-12 * np.abs(yr).max()
    f32 = D.HesthavenEvolution(vx, E, fbc, order, eps=eps, precision=32, kernel="valu")
    assert np.linalg.norm(f32.mult(x) - yr) <= 1e-5 * np.linalg.norm(yr)
    dt = 0.1 * np.abs(x).max() / np.abs(yr).max()
    for integrator in ("lserk4", "rk4"):
        ends = []
        for kernel in ("valu", "mfma"):
            op = D.HesthavenEvolution(vx, E, fbc, order, eps=eps, precision=64, kernel=kernel, integrator=integrator)
            op.set_state(x)
            op.advance(dt, 2)
            ends.append(op.get_state())
        assert np.abs(ends[0] - ends[1]).max() <= 1e-12 * np.abs(ends[1]).max()
