"""Time steps of operators above 12 MB per state buffer, where LSERK4's first
stage reads no residual and its last leaves none, and where the stage output
is kept in the Infinity Cache up to 250 MB in all: the step composed on the host in
FP64 from the operator's own Mult (2N-storage recurrence with
test_rk_tableau's coefficients, classic RK4 in MFEM's order), every shape,
kernel and precision, plane waves at the stage times included.  Mult itself is
pinned to the oracle by the other tests; here the kernels of one shape are
compared with each other at these sizes.

Bars: FP64 1e-12 of the largest entry (other orders of the same sums), FP32
1e-5 relative L2.
"""
import numpy as np
import pytest

from test_global_assembly import csr_matvec
from test_rk_tableau import A, B, lserk_polynomials
from test_tfsf import MEAN, SPREAD

pytestmark = pytest.mark.gpu

import dgtd_amd as D  # noqa: E402

C = lserk_polynomials()[1]
ORDER = {"tet": 3, "triangle": 4, "quad": 3, "hex": 2}
NODES = {"tet": 20, "triangle": 15, "quad": 16, "hex": 27}
FACES = {"tet": [(1, 2, 3), (0, 2, 3), (0, 1, 3), (0, 1, 2)], "triangle": [(0, 1), (1, 2), (2, 0)],
         "quad": [(0, 1), (1, 2), (2, 3), (3, 0)],
         "hex": [(3, 2, 1, 0), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (3, 0, 4, 7), (4, 5, 6, 7)]}
CASES = [("tet", "valu"), ("tet", "mfma"), ("tet", "csr"), ("triangle", "valu"), ("triangle", "mfma"),
         ("triangle", "csr"), ("quad", "csr"), ("hex", "valu"), ("hex", "csr")]


def mesh(shape, megabytes, precision, tfsf=False):
    """A sheared box of just more than that many megabytes per state buffer;
    with tfsf its faces in the middle plane carry TF/SF."""
    per_cell = {"tet": 6, "triangle": 2}.get(shape, 1) * NODES[shape] * 6 * precision // 8
    cells = int(megabytes * 1e6 / per_cell) + 1
    dim = 2 if shape in ("triangle", "quad") else 3
    n = int(cells ** (1 / dim)) // 2 * 2
    m = -(-cells // n ** (dim - 1))
    bc = ["pec", "sma", "pmc", "sma", "pec", "sma"][:2 * dim]
    vx, E, fbc = D.cartesian_2d(n, m, shape, bc=bc) if dim == 2 else D.cartesian_3d(n, n, m, shape, bc=bc)
    fbc = fbc.copy()
    if tfsf:
        for f, v in enumerate(FACES[shape]):
            fbc[(np.abs(vx[E[:, v], 0] - 0.5) < 1e-9).all(axis=1), f] = 7
        assert (fbc == 7).any()
    vx = vx + 0.2 * vx[:, [1, 0, 2]] * np.array([1, 1, 0])
    assert 6 * NODES[shape] * E.shape[0] * precision // 8 > megabytes * 1e6
    return vx, E, fbc


def operator(shape, kernel, precision, m, integrator="lserk4"):
    K = m[1].shape[0]
    rng = np.random.default_rng(1)
    eps, sigma = rng.uniform(1, 4, K), rng.uniform(0, 3, K)
    return D.HesthavenEvolution(*m, ORDER[shape], alpha=0.5, eps=eps, precision=precision, integrator=integrator,
                                kernel=kernel, sigma=sigma if kernel == "csr" or shape == "hex" else None,
                                quads=shape == "quad")


def composed(op, x, t, dt, steps, integrator):
    def rhs(q, time):
        op.SetTime(time)
        return op.mult(q)

    q = x.copy()
    for _ in range(steps):
        if integrator == "lserk4":
            res = np.zeros_like(q)
            for s in range(5):
                res = A[s] * res + dt * rhs(q, t + C[s] * dt)
                q = q + B[s] * res
        else:
            k1 = rhs(q, t)
            k2 = rhs(q + dt / 2 * k1, t + dt / 2)
            k3 = rhs(q + dt / 2 * k2, t + dt / 2)
            k4 = rhs(q + dt * k3, t + dt)
            q = q + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        t += dt
    return q


def agree(got, want, precision):
    if precision == 64:
        return np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
    return np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


def check_steps(op, precision, integrator, x, t, dt):
    want = composed(op, x, t, dt, 2, integrator)
    op.set_state(x, t)
    op.advance(dt, 1)
    op.advance(dt, 1)
    got = op.get_state()
    assert agree(got, want, precision)
    return got


@pytest.mark.parametrize("integrator", ["lserk4", "rk4"])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape,kernel", CASES)
def test_steps(shape, kernel, precision, integrator):
    m = mesh(shape, 12, precision)
    op = operator(shape, kernel, precision, m, integrator)
    x = np.random.default_rng(2).standard_normal(op.ndofs)
    y = op.mult(x)
    dt = 0.2 * np.linalg.norm(x) / np.linalg.norm(y)
    got = check_steps(op, precision, integrator, x, 0.0, dt)
    op.set_graphs(True)
    op.set_state(x)
    for _ in range(2):
        op.advance(dt, 1)
    assert np.array_equal(op.get_state(), got)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape", ["tet", "triangle", "quad", "hex"])
def test_kernels_agree(shape, precision):
    m = mesh(shape, 12, precision)
    kernels = [k for s, k in CASES if s == shape and (k != "csr" or shape == "hex")]
    ops = [operator(shape, k, precision, m) for k in kernels]
    x = np.random.default_rng(3).standard_normal(6 * NODES[shape] * m[1].shape[0])
    if shape == "quad":  # one kernel: against the matrix
        K = m[1].shape[0]
        rng = np.random.default_rng(1)
        eps, sigma = rng.uniform(1, 4, K), rng.uniform(0, 3, K)
        M = D.global_assemble(*m, ORDER[shape], alpha=0.5, eps=eps, sigma=sigma, quads=True)
        assert agree(operator(shape, "csr", precision, m).mult(x), csr_matvec(M, x), precision)
        return
    ys = [op.mult(x) for op in ops]
    for y in ys[1:]:
        assert agree(y, ys[0], precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("shape,kernel", CASES)
def test_plane_wave_steps(shape, kernel, precision):
    """From rest, so that every entry stems from the injection."""
    m = mesh(shape, 12, precision, tfsf=True)
    op = operator(shape, kernel, precision, m)
    op.set_planewaves([D.planewave((0, 0, 1), (1, 0, 0), SPREAD, MEAN)])
    x = np.random.default_rng(2).standard_normal(op.ndofs)
    dt = 0.2 * np.linalg.norm(x) / np.linalg.norm(op.mult(x))
    zero = np.zeros(op.ndofs)
    op.SetTime(1.0)
    assert np.abs(op.mult(zero)).max() > 0
    check_steps(op, precision, "lserk4", zero, 1.0, dt)


@pytest.mark.parametrize("shape,kernel", [("tet", "valu"), ("tet", "mfma"), ("triangle", "valu"), ("triangle", "mfma")])
def test_steps_past_the_infinity_cache(shape, kernel):
    op = operator(shape, kernel, 64, mesh(shape, 125, 64))
    x = np.random.default_rng(2).standard_normal(op.ndofs)
    dt = 0.2 * np.linalg.norm(x) / np.linalg.norm(op.mult(x))
    check_steps(op, 64, "lserk4", x, 0.0, dt)


@pytest.mark.parametrize("shape,kernel", CASES)
def test_bytes_per_stage(shape, kernel):
    """A step of five stages moves 18 passes over the six components above 12
    MB per state buffer and 20 below it (always 20 with the assembled matrix;
    RK4: 16 in four stages)."""
    records = {"tet": 27 * 8 + 32, "triangle": 15 * 8 + 24, "quad": 19 * 8 + 32, "hex": 36 * 8 + 48}[shape]
    for megabytes, integrator, passes in ((12, "lserk4", 18 / 5), (0.1, "lserk4", 4), (12, "rk4", 4)):
        op = operator(shape, kernel, 64, mesh(shape, megabytes, 64), integrator)
        b = op.work_per_element()[0]
        if (shape, kernel) == ("hex", "csr"):
            assert b > 4 * 6 * NODES[shape] * 8
        else:
            assert b == pytest.approx(passes * 6 * NODES[shape] * 8 + records, rel=1e-14)
