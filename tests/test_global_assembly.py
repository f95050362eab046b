"""The operator of the "csr" kernel, assembled (the Global operator's matrix,
DGOperatorFactory::buildGlobalOperator, DGOperatorFactory.h:1428-1600),
checked on the host.

- Without conductivity A x equals the oracle's Mult (tetrahedra:
  oracle/dgtd_oracle.cpp; triangles: oracle/oracle2d.py) for every face code,
  to 1e-12 relative: only the summation order differs.  SMA boundary faces
  follow the Global operator, which weights their upwind terms by 1 whatever
  alpha (DGOperatorFactory.h:485-495, 521-531, 557-567): the expected product
  is the oracle's with those faces' contribution taken at alpha = 1, isolated
  by linearity (the same faces with zero jump contribute nothing).
- Bulk conductivity (collectGlobalConductiveOperator, DGOperatorFactory.h:
  1351-1361, -M_eps^-1 M_sigma on the E blocks) is pinned through the energy
  balance of the semi-discrete system: with the energy inner product
  B(x, y) = sum_e J_e (eps E_x^T M E_y + mu H_x^T M H_y), the centred operator
  on PEC walls is skew (B(x, A x) = 0) and conductivity adds exactly
  -sum_e J_e sigma_e E^T M E (Poynting's theorem: d/dt W = -int sigma |E|^2).
  A wrong sign, a missing 1/eps or a term on the H rows fails it.
"""
import numpy as np
import pytest

import meshgen as MG
from oracle import oracle as O
from oracle import oracle2d as O2

import dgtd_amd as D


def csr_matvec(A, x):
    rowptr, col, val = A
    out = np.zeros(rowptr.size - 1)
    prod = val * x[col]
    nz = np.diff(rowptr) > 0
    out[nz] = np.add.reduceat(prod, rowptr[:-1][nz])
    return out


def bform(energy, x, y):
    """B(x, y) from the quadratic form energy(x) = B(x, x) / 2."""
    return 0.5 * (energy(x + y) - energy(x - y))


def global_expected(make, fbc, x, alpha):
    """Global-operator product from the hesthaven oracle: make(fbc, alpha)
    builds an oracle operator; SMA boundary faces (code 3) are taken at
    alpha = 1 by linearity (the face's contribution isolated as the
    difference of the operator with and without it, both at alpha = 1)."""
    fbc = np.asarray(fbc)
    zero = fbc.copy()
    zero[fbc == 3] = 0
    y = make(zero, alpha).mult(x)
    if (fbc == 3).any():
        y = y + make(fbc, 1.0).mult(x) - make(zero, 1.0).mult(x)
    return y


def test_oracle_global_sma_switch_equals_linearity():
    """The oracle's Global-operator SMA weighting (global_sma) against the
    linearity construction on boundary SMA faces, and against the plain
    oracle when no SMA face is present or alpha = 1."""
    vx, E, fbc, eps, mu = cube_case(2, 7)
    x = np.random.default_rng(7).standard_normal(6 * O.np_of(3) * E.shape[0])
    for alpha in (0.5, 0.0):
        mk = lambda b, a, g=False: O.Operator(vx, E, b, 3, alpha=a, eps=eps, mu=mu, global_sma=g)
        yl = global_expected(lambda b, a: mk(b, a), fbc, x, alpha)
        yg = mk(fbc, alpha, True).mult(x)
        assert np.abs(yg - yl).max() <= 1e-12 * np.abs(yl).max()
    nosma = np.where(np.asarray(fbc) == 3, 1, fbc)
    for g in (False, True):
        y = O.Operator(vx, E, nosma, 3, alpha=0.5, global_sma=g).mult(x)
        if not g:
            y0 = y
    assert np.array_equal(y, y0)
    y1 = O.Operator(vx, E, fbc, 3, alpha=1.0, eps=eps, mu=mu).mult(x)
    assert np.array_equal(O.Operator(vx, E, fbc, 3, alpha=1.0, eps=eps, mu=mu, global_sma=True).mult(x), y1)


def cube_case(n, seed, bc=("pec", "pmc", "sma", "pec", "pmc", "sma")):
    rng = np.random.default_rng(seed)
    vx, E, fbc = MG.cube_mesh(n, 1.0, list(bc))
    K = E.shape[0]
    return vx, E, fbc, rng.uniform(1, 4, K), rng.uniform(1, 2, K)


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("alpha", [1.0, 0.5, 0.0])
def test_tet_matrix_equals_oracle_mult(order, alpha):
    """alpha = 0 with SMA faces: the centred Global operator, which the
    hesthaven operator refuses (driver.cpp:1596-1598)."""
    vx, E, fbc, eps, mu = cube_case(2, order)
    A = D.global_assemble(vx, E, fbc, order, alpha=alpha, eps=eps, mu=mu)
    x = np.random.default_rng(order).standard_normal(A[0].size - 1)
    yr = global_expected(lambda b, a: O.Operator(vx, E, b, order, alpha=a, eps=eps, mu=mu), fbc, x, alpha)
    y = csr_matvec(A, x)
    assert np.abs(y - yr).max() <= 1e-12 * np.abs(yr).max()
    if alpha == 0.5:  # and the SMA faces do differ from the hesthaven operator's
        ref = O.Operator(vx, E, fbc, order, alpha=alpha, eps=eps, mu=mu)
        assert np.abs(y - ref.mult(x)).max() > 1e-6 * np.abs(yr).max()
    rowptr, col, val = A
    assert rowptr[0] == 0 and np.all(np.diff(rowptr) > 0)
    assert col.min() >= 0 and col.max() < x.size and np.all(val != 0.0)
    for r in range(0, x.size, 97):  # columns unique within a row
        seg = col[rowptr[r]:rowptr[r + 1]]
        assert np.unique(seg).size == seg.size


@pytest.mark.parametrize("cond", [4, 5, 6, 7])
def test_tet_interior_and_tfsf_faces_equal_oracle_mult(cond):
    vx, E, fbc = MG.cube_mesh(2, 1.0, "pec")
    fbc = fbc.astype(np.int32)
    fbc[MG.plane_faces(vx, E, 0, 0.5)] = cond
    A = D.global_assemble(vx, E, fbc, 3, alpha=0.7)
    ref = O.Operator(vx, E, fbc, 3, alpha=0.7, global_sma=True)
    x = np.random.default_rng(cond).standard_normal(ref.ndofs)
    yr = ref.mult(x)  # TF/SF faces without plane waves: plain interior faces
    assert np.abs(csr_matvec(A, x) - yr).max() <= 1e-12 * np.abs(yr).max()
    if cond == 6:  # interior SMA at upwind weight 1: differs from the hesthaven weighting
        yh = O.Operator(vx, E, fbc, 3, alpha=0.7).mult(x)
        assert np.abs(csr_matvec(A, x) - yh).max() > 1e-6 * np.abs(yr).max()


def _tri_line_edges(vx, E, x0):
    on = np.zeros(E.shape, dtype=bool)
    for f, (p, q) in enumerate(MG.TRI_EDGES):
        on[:, f] = (np.abs(vx[E[:, p], 0] - x0) < 1e-12) & (np.abs(vx[E[:, q], 0] - x0) < 1e-12)
    return on


def _tri_cut_at_x(vx, E, x0):
    on = np.where(np.abs(vx[:, 0] - x0) < 1e-12)[0]
    dup = {int(v): vx.shape[0] + i for i, v in enumerate(on)}
    vx2 = np.vstack([vx, vx[on]])
    E2 = E.copy()
    for e in range(E.shape[0]):
        if vx[E[e], 0].mean() > x0:
            E2[e] = [dup.get(int(v), int(v)) for v in E[e]]
    return vx2, E2


@pytest.mark.parametrize("alpha", [0.5, 0.0])
@pytest.mark.parametrize("dim", [3, 2])
def test_interior_sma_weighted_as_global_operator(dim, alpha):
    """Interior SMA faces (code 6) take upwind weight 1 in the Global
    operator whatever alpha (DGOperatorFactory.h:587-591, 655-659), centred
    flux included; SMA boundary faces as well.  The oracle's weighting is
    pinned first: the flux is linear in the jump and in the face's upwind
    weight, so an interior SMA face at weight 1 equals the mean of the mesh
    cut along that surface with SMA boundaries (jump -1, weight 1) and of the
    cut mesh with zero jump there."""
    if dim == 3:
        vx, E, fbc = MG.cube_mesh(2, 1.0, ["pec", "sma", "pmc", "sma", "pec", "pec"])
        fbc = np.asarray(fbc, dtype=np.int32)
        on = MG.plane_faces(vx, E, 0, 0.5)
        vx2, E2 = MG.cut_along_plane(vx, E, 0, 0.5)
        make = lambda v, e, b: O.Operator(v, e, b, 3, alpha=alpha, global_sma=True)
    else:
        vx, E, fbc = MG.square_mesh(4, bc=["pec", "sma", "pmc", "pec"], jitter=0.0, seed=1)
        fbc = np.asarray(fbc, dtype=np.int32)
        on = _tri_line_edges(vx, E, 0.5)
        vx2, E2 = _tri_cut_at_x(vx, E, 0.5)
        make = lambda v, e, b: O2.Operator2D(v, e, b, 3, alpha=alpha, global_sma=True)
    assert on.any()
    fbc6 = np.where(on, 6, fbc)
    ref = make(vx, E, fbc6)
    A = D.global_assemble(vx, E, fbc6, 3, alpha=alpha)
    x = np.random.default_rng(11).standard_normal(A[0].size - 1)
    yr = ref.mult(x)
    ycut = 0.5 * (make(vx2, E2, np.where(on, 3, fbc)).mult(x) + make(vx2, E2, np.where(on, 0, fbc)).mult(x))
    assert np.abs(yr - ycut).max() <= 1e-12 * np.abs(yr).max()
    assert np.abs(csr_matvec(A, x) - yr).max() <= 1e-12 * np.abs(yr).max()


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
def test_tri_matrix_equals_oracle_mult(order):
    vx, E, bc = MG.square_mesh(4, bc=["pec", "pmc", "sma", "pec"], jitter=0.2, seed=order)
    rng = np.random.default_rng(order)
    eps, mu = rng.uniform(1, 4, E.shape[0]), rng.uniform(1, 2, E.shape[0])
    for alpha in (1.0, 0.5):
        A = D.global_assemble(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu)
        x = rng.standard_normal(A[0].size - 1)
        yr = global_expected(lambda b, a: O2.Operator2D(vx, E, b, order, alpha=a, eps=eps, mu=mu), bc, x, alpha)
        assert np.abs(csr_matvec(A, x) - yr).max() <= 1e-12 * np.abs(yr).max()


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
def test_quad_matrix_equals_oracle_mult(order):
    """Quadrilaterals (parallelograms of unequal sizes, sheared): boundary
    PEC/PMC/SMA, interior PEC/PMC/SMA and TF/SF edges (without plane waves a
    TF/SF edge is a plain interior edge), SMA at upwind weight 1 whatever
    alpha, as the Global operator assembles it."""
    vx, E, bc = MG.quad_mesh(4, 3, Lx=2.0, bc=["pec", "pmc", "sma", "pec"], stretch=0.3, shear=0.3, seed=order)
    bc = bc.copy()
    bc[5, 1], bc[6, 3] = 4, 4   # interior PEC edge between elements 5 and 6
    bc[1, 2], bc[5, 0] = 5, 5   # interior PMC edge between elements 1 and 5
    bc[6, 2], bc[10, 0] = 6, 6  # interior SMA edge between elements 6 and 10
    bc[2, 1], bc[3, 3] = 7, 7   # TF/SF edge between elements 2 and 3
    rng = np.random.default_rng(order)
    eps, mu = rng.uniform(1, 4, E.shape[0]), rng.uniform(1, 2, E.shape[0])
    for alpha in (1.0, 0.5, 0.0):
        A = D.global_assemble(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu, quads=True)
        x = rng.standard_normal(A[0].size - 1)
        yr = O2.Operator2D(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu, global_sma=True, quads=True).mult(x)
        assert np.abs(csr_matvec(A, x) - yr).max() <= 1e-12 * np.abs(yr).max()


@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_hex_matrix_equals_oracle_mult(order):
    """Hexahedra (sheared parallelepipeds): boundary PEC/PMC/SMA, interior
    PEC/PMC/SMA and TF/SF faces, SMA at upwind weight 1 whatever alpha, every
    neighbour orientation the shear leaves; against oracle/oracle_hex.py."""
    from oracle import oracle_hex as OH
    from test_oracle_hex import sheared_hexes

    vx, E, bc = sheared_hexes(3, 2, 2, bc=("pec", "pmc", "sma", "pec", "pmc", "sma"), sx=1.5)
    bc = bc.copy()
    bc[0, 2], bc[1, 4] = 4, 4   # interior PEC between elements 0 and 1 (x faces)
    bc[1, 3], bc[4, 1] = 7, 7   # TF/SF between elements 1 and 4 (y faces)
    bc[4, 5], bc[10, 0] = 5, 5  # interior PMC between elements 4 and 10 (z faces)
    bc[2, 3], bc[5, 1] = 6, 6   # interior SMA between elements 2 and 5
    rng = np.random.default_rng(order)
    eps, mu = rng.uniform(1, 4, E.shape[0]), rng.uniform(1, 2, E.shape[0])
    for alpha in (1.0, 0.5, 0.0):
        A = D.global_assemble(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu)
        x = rng.standard_normal(A[0].size - 1)
        yr = OH.OperatorHex(vx, E, bc, order, alpha=alpha, eps=eps, mu=mu).mult(x)
        assert np.abs(csr_matvec(A, x) - yr).max() <= 1e-12 * np.abs(yr).max()


def test_hex_neighbour_orientations():
    """The second hexahedron of a 2 x 1 x 1 pair takes each of the cube's 24
    rotations of its vertex list (still a positively oriented parallelepiped
    in MFEM order): the shared face is then each of its six faces, entered at
    each of the four corners (two positively oriented neighbours always
    traverse a shared face in opposite directions).  The host matrix and the
    oracle agree, and the product is unchanged up to the node relabelling
    (the physics does not depend on the local vertex order)."""
    from oracle import oracle_hex as OH

    vx, E, bc = D.cartesian_3d(2, 1, 1, "hex", bc="pec")
    x = np.random.default_rng(3).standard_normal(6 * 27 * 2)
    ref = OH.OperatorHex(vx, E, bc, 2)
    y0 = ref.mult(x)
    # the cube's 24 proper rotations as vertex permutations of MFEM's hexahedron
    C = OH.HEX_CORNERS
    lookup = {tuple(c): i for i, c in enumerate(C)}
    perms = set()
    for mat in _rotations():
        img = [lookup[tuple(np.rint(mat @ (c - 0.5) + 0.5).astype(int))] for c in C]
        perms.add(tuple(img))
    assert len(perms) == 24
    R = OH.RefHex(2)
    for perm in sorted(perms):
        E2 = E.copy()
        E2[1] = E[1][list(perm)]
        # face codes follow the faces: boundary everywhere except the shared face
        op2 = OH.OperatorHex(vx, E2, np.where(_shared(E2), 0, 1), 2)
        A = D.global_assemble(vx, E2, np.where(_shared(E2), 0, 1), 2)
        # same node set per element: map the oracle's state by node position
        pos1, pos2 = ref.pos.reshape(-1, 3), op2.pos.reshape(-1, 3)
        key = lambda p: np.round(p, 9).view([("", p.dtype)] * 3).ravel()
        i1, i2 = np.argsort(key(pos1), kind="stable"), np.argsort(key(pos2), kind="stable")
        m = np.empty(pos1.shape[0], dtype=np.int64)
        m[i2] = i1
        x2 = x.reshape(6, -1)[:, m].reshape(-1)
        y2 = csr_matvec(A, x2)
        np.testing.assert_allclose(y2, op2.mult(x2), atol=1e-12 * np.abs(y0).max())
        np.testing.assert_allclose(y2.reshape(6, -1), y0.reshape(6, -1)[:, m], atol=1e-11 * np.abs(y0).max())
    assert R.Np == 27


def _rotations():
    import itertools
    out = []
    for perm in itertools.permutations(range(3)):
        for signs in itertools.product((1, -1), repeat=3):
            M = np.zeros((3, 3))
            for r, (c, s) in enumerate(zip(perm, signs)):
                M[r, c] = s
            if np.linalg.det(M) > 0:
                out.append(M)
    return out


def _shared(E2):
    """(2, 6) mask of the faces the two hexahedra share."""
    from oracle import oracle_hex as OH

    keys = [[tuple(sorted(E2[e][list(f)])) for f in OH.HEX_FACES] for e in range(2)]
    common = set(keys[0]) & set(keys[1])
    return np.array([[k in common for k in keys[e]] for e in range(2)])


@pytest.mark.parametrize("dim", [3, 2, 4, 8])
def test_conductivity_energy_balance(dim):
    """dim 4: quadrilaterals, 8: hexahedra."""
    rng = np.random.default_rng(dim)
    if dim == 3:
        vx, E, fbc = MG.cube_mesh(2, 1.0, "pec")
        order = 3
    elif dim == 2:
        vx, E, fbc = MG.square_mesh(5, bc="pec", jitter=0.2, seed=1)
        order = 4
    elif dim == 4:
        vx, E, fbc = MG.quad_mesh(3, 4, bc="pec", stretch=0.3, shear=-0.2, seed=2)
        order = 3
    else:
        from test_oracle_hex import sheared_hexes

        vx, E, fbc = sheared_hexes(2, 2, 2, bc="pec")
        order = 2
    K = E.shape[0]
    eps, mu, sigma = rng.uniform(1, 4, K), rng.uniform(1, 2, K), rng.uniform(0.5, 3.0, K)

    def oracle(eps_, mu_):
        if dim == 8:
            from oracle import oracle_hex as OH

            return OH.OperatorHex(vx, E, fbc, order, alpha=0.0, eps=eps_, mu=mu_)
        return (O.Operator(vx, E, fbc, order, alpha=0.0, eps=eps_, mu=mu_) if dim == 3
                else O2.Operator2D(vx, E, fbc, order, alpha=0.0, eps=eps_, mu=mu_, quads=dim == 4))

    W = oracle(eps, mu)
    Ws = oracle(sigma, np.ones(K))  # energy with eps -> sigma: (1/2) sum J sigma E^T M E + ...
    A0 = D.global_assemble(vx, E, fbc, order, alpha=0.0, eps=eps, mu=mu)
    As = D.global_assemble(vx, E, fbc, order, alpha=0.0, eps=eps, mu=mu, sigma=sigma)
    x = rng.standard_normal(A0[0].size - 1)
    y0, ys = csr_matvec(A0, x), csr_matvec(As, x)
    scale = np.linalg.norm(x) * np.linalg.norm(y0) * eps.max()
    # centred flux with PEC walls: skew in the energy inner product
    assert abs(bform(W.energy, x, y0)) <= 1e-12 * scale
    # conductivity: B(x, A_sigma x) = -sum_e J_e sigma_e E^T M E
    xe = x.copy()
    xe[xe.size // 2:] = 0.0
    want = -2.0 * Ws.energy(xe)
    assert bform(W.energy, x, ys) == pytest.approx(want, rel=1e-11)
    # and it only touches the E rows
    half = x.size // 2
    assert np.array_equal(ys[half:], y0[half:])


def test_conductivity_needs_the_assembled_operator():
    vx, E, fbc = MG.cube_mesh(1, 1.0, "pec")
    sig = np.ones(E.shape[0])
    with pytest.raises(D.DgtdError, match="DGTD_KERNEL_CSR"):
        D.HesthavenEvolution(vx, E, fbc, 2, sigma=sig, kernel="valu")
    with pytest.raises(D.DgtdError, match="conductivity"):
        D.global_assemble(vx, E, fbc, 2, sigma=-sig)
