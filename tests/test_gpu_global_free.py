"""The Global operator applied without a matrix against the matrix itself
(dgtd_global_assemble, FP64 on the host, pinned to the oracle in
tests/test_global_assembly.py): element counts around one block of the stage
kernels, every order, face orientations, every boundary and interior face code, conductivity, and
upwind weights where SMA faces differ from the hesthaven operator.

Bars: FP64 1e-12 of the largest entry, as the Global operator's other tests
(row sums of a few hundred products); FP32 1e-5 relative L2.
"""
import numpy as np
import pytest

from test_global_assembly import csr_matvec

pytestmark = pytest.mark.gpu

import dgtd_amd as D  # noqa: E402


def mesh(shape, K, seed):
    """K elements of a box with random wall codes, a third of the interior
    faces carrying an interior condition, random materials."""
    rng = np.random.default_rng(seed)
    if shape in ("tet", "hex"):
        n = 3 if shape == "tet" else 6
        vx, E, bc = D.cartesian_3d(n, n, n, shape, sx=1.1, sy=0.9, sz=1.0)
        if shape == "tet":  # the six of a cell in a row, so that the first K share faces
            cell = np.arange(E.shape[0]).reshape(6, -1).T.ravel()
            E, bc = E[cell], bc[cell]
    else:
        n = 8 if shape == "triangle" else 15
        vx, E, bc = D.cartesian_2d(n, n, shape, sx=1.2, sy=0.8)
    vx = vx + 0.2 * vx[:, [1, 0, 2]] * (shape != "tet")  # sheared
    E, bc = E[:K].copy(), bc[:K].copy()
    if shape == "hex":  # every element in its own rotation about z
        for e in range(E.shape[0]):
            r = int(rng.integers(0, 4))
            E[e] = E[e][[(r + i) % 4 for i in range(4)] + [4 + (r + i) % 4 for i in range(4)]]
            bc[e] = bc[e][[0] + [1 + (r + i) % 4 for i in range(4)] + [5]]
    if shape == "quad":
        for e in range(E.shape[0]):
            r = int(rng.integers(0, 4))
            E[e], bc[e] = np.roll(E[e], -r), np.roll(bc[e], -r)
    walls = bc != 0
    bc[walls] = rng.integers(0, 4, int(walls.sum()))
    # a face is interior when its vertices occur twice
    nf = E.shape[1]
    if shape == "tet":
        verts = [[v for v in range(4) if v != f] for f in range(4)]
    elif shape == "hex":
        verts, nf = [(3, 2, 1, 0), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (3, 0, 4, 7), (4, 5, 6, 7)], 6
    else:
        verts = [(f, (f + 1) % nf) for f in range(nf)]
    faces = [np.sort(E[:, v], axis=1) for v in verts]
    seen = {}
    for f in range(nf):
        for e in range(E.shape[0]):
            seen.setdefault(tuple(faces[f][e]), []).append((e, f))
    for pair in seen.values():
        if len(pair) == 2 and rng.random() < 0.33:
            bc[pair[0]] = rng.integers(4, 7)
    K = E.shape[0]
    return vx, E, bc, rng.uniform(1, 4, K), rng.uniform(1, 2, K), rng.uniform(0, 3, K)


@pytest.mark.parametrize("shape,order", [(s, p) for s in ("tet", "triangle", "quad", "hex") for p in range(1, 6)])
def test_matches_the_matrix(shape, order):
    p1 = order + 1
    npe = {"tet": p1 * (p1 + 1) * (p1 + 2) // 6, "triangle": p1 * (p1 + 1) // 2, "quad": p1 ** 2, "hex": p1 ** 3}[shape]
    block = 256 // npe
    make = lambda mesh, **kw: (D.HesthavenEvolution(*mesh, kernel="valu", **kw) if shape == "hex"  # noqa: E731
                               else D.GlobalEvolution(*mesh, quads=shape == "quad", **kw))
    for K, alpha in ((1, 1.0), (max(1, block - 1), 0.0), (block, 0.5), (block + 1, 0.5), (3 * block + 2, 1.0)):
        vx, E, bc, eps, mu, sigma = mesh(shape, K, 10 * order + K)
        A = D.global_assemble(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu, sigma=sigma, quads=shape == "quad")
        kw = dict(alpha=alpha, eps=eps, mu=mu, sigma=sigma)
        x = np.random.default_rng(K).standard_normal(A[0].size - 1)
        y = csr_matvec(A, x)
        g = make((vx, E, bc, order), precision=64, **kw)
        assert np.abs(g.mult(x) - y).max() <= 1e-12 * np.abs(y).max()
        g32 = make((vx, E, bc, order), precision=32, **kw)
        assert np.linalg.norm(g32.mult(x) - y) <= 1e-5 * np.linalg.norm(y)
        # one classic RK4 step is the Taylor polynomial of the matrix
        dt = 0.02
        z, k = x.copy(), x.copy()
        for m in range(1, 5):
            k = csr_matvec(A, k) * (dt / m)
            z += k
        r = make((vx, E, bc, order), precision=64, integrator="rk4", **kw)
        r.set_state(x)
        r.advance(dt, 1)
        assert np.abs(r.get_state() - z).max() <= 1e-12 * max(np.abs(z).max(), np.abs(k).max())
