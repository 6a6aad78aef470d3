"""GPU test of the base factors on the device, at the sizes around its tiles and
its limit of 128 rows: a multigrid whose base level is its top level applies the
inverse of the assembled matrix (dense solve in numpy; error at most 64 m eps
cond). Large coefficients make the columns of Dirichlet DoFs swap rows; a
vanishing coefficient is singular."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


@pytest.mark.parametrize("kind,refs,rows", [(0, 0, 8), (0, 1, 27), (0, 2, 125), (1, 0, 4), (1, 2, 25), (1, 3, 81),
                                            (1, 4, 289), (2, 0, 64)])
@pytest.mark.parametrize("shift", [0.0, 6.0])
def test_base_solve_is_the_inverse(kind, refs, rows, shift):
    print(f"case base lu kind={kind} refs={refs} shift={shift}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(10 * kind + refs)
    d = u.DomainDiscretization(kind, refs)
    if kind != 1:
        d.set_theta(shift + rng.normal(size=d.n_fine ** d.dim))
    if kind == 2:
        d.set_velocity((2000.0, 10.0, -500.0))
        d.set_jitter(3, 0.2 / np.sqrt(3.0))
    N = d.num_dofs()
    assert N == rows
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    rp, cl, vl = A.download_csr()
    M = np.zeros((N, N))
    np.add.at(M, (np.repeat(np.arange(N), np.diff(rp)), cl), vl)
    for transposed in ((False, True) if kind != 1 else (False,)):
        g = u.GeometricMultiGrid(d, base_level=refs, transposed=transposed)
        g.init(A)
        dv = rng.normal(size=N)
        dv[d.num_inner():] = 0.0
        c = u.Vector(N)
        g.apply(c, u.Vector(values=dv))
        E = M
        if transposed:
            # the transposed operator: Dirichlet rows stay identity rows
            E = M.T.copy()
            E[d.num_inner():] = 0.0
            E[np.arange(d.num_inner(), N), np.arange(d.num_inner(), N)] = 1.0
        ref = np.linalg.solve(E, dv)
        assert np.abs(c.numpy() - ref).max() <= 64 * N * 2.0 ** -52 * np.linalg.cond(E) * np.abs(ref).max()


@pytest.mark.parametrize("refs", [1, 2])
def test_singular_base_matrix(refs):
    print(f"case base lu singular refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    d = u.DomainDiscretization(0, refs)
    d.set_theta(np.full(8 ** refs, -60.0))
    A, b = u.SparseMatrix(), u.Vector(d.num_dofs())
    d.assemble_linear(A, b)
    g = u.GeometricMultiGrid(d, base_level=refs)
    with pytest.raises(u.UGError, match="singular"):
        g.init(A)
