"""GPU test of the CG whose scalars are formed by the kernels that use them, on
both sides of the line up to which the update sums the operator's partial sums
itself (65^3 and 129^3) and at one workgroup: solution, defects and returned
defect against the same CG on the surface operator, and the breakdown lambda = 0
of a zero operator direction."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


@pytest.mark.parametrize("kind,refs,precision", [(0, 1, "f64"), (0, 2, "f32"), (0, 5, "f32"), (0, 6, "f64"),
                                                 (0, 7, "f32"), (1, 3, "f64"), (1, 6, "f32")])
def test_lattice_cg_equals_surface_cg(kind, refs, precision):
    print(f"case cg scalars kind={kind} refs={refs} {precision}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(refs)
    d = u.DomainDiscretization(kind, refs)
    if kind == 0:
        d.set_theta(0.5 * rng.normal(size=8 ** refs))
    N, ni = d.num_dofs(), d.num_inner()
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    x0, rhs = rng.normal(size=N), rng.normal(size=N)
    x0[ni:] = rhs[ni:] = 0.0
    for start in (np.zeros(N), x0):
        got = []
        for on in (True, False):
            S = u.CG(u.GeometricMultiGrid(d, base_level=min(refs, 1), precision=precision), max_steps=100, reduction=1e-10)
            S.set_lattice_path(on)
            S.init(A)
            x, r = u.Vector(values=start), u.Vector(values=rhs)
            assert S.apply_return_defect(x, r)
            assert S.used_lattice_path() == on
            assert np.linalg.norm(r.numpy()) == pytest.approx(S.defects()[-1], rel=1e-10)
            got.append((x.numpy(), S.defects()))
        (xl, dl), (xs, ds) = got
        assert abs(len(dl) - len(ds)) <= 1
        n = min(len(dl), len(ds)) - 1
        # the two operators differ by the quadrature's rounding, which the steps amplify
        assert np.allclose(dl[:n], ds[:n], rtol=1e-2)
        assert np.linalg.norm(xl - xs) <= 1e-8 * np.linalg.norm(xs)


def test_breakdown_leaves_the_solution():
    print("case cg breakdown", flush=True)
    sys.stdout.flush()
    u = U()
    n = 300
    A = u.SparseMatrix()
    # p^T A p = 0 for p = b: the entries of +1 and -1 cancel
    A.upload_csr(np.arange(n + 1), np.arange(n), np.where(np.arange(n) % 2 == 0, 1.0, -1.0))
    S = u.CG(None, max_steps=10, reduction=1e-10)
    S.init(A)
    x = u.Vector(n)
    assert not S.apply(x, u.Vector(values=np.ones(n)))
    assert not x.numpy().any()


@pytest.mark.parametrize("rows,cols", [(40, 70), (40, 41)])
def test_rectangular_operator_is_refused(rows, cols):
    """a Jacobi-preconditioned CG on a matrix with more columns than rows: the
    product z.r of vectors of different lengths is an error"""
    print(f"case cg rectangular {rows}x{cols}", flush=True)
    import ugcore_amd as u
    rng = np.random.default_rng(rows)
    M = np.zeros((rows, cols))
    M[np.arange(rows), np.arange(rows)] = 4.0
    M[np.arange(rows), (np.arange(rows) + 1) % cols] = -1.0
    c = np.argsort(M == 0, axis=1, kind="stable")[:, :2]
    c.sort(axis=1)
    A = u.SparseMatrix()
    A.upload_csr(2 * np.arange(rows + 1), c.reshape(-1), np.take_along_axis(M, c, 1).reshape(-1), n_cols=cols)
    S = u.CG(u.Jacobi(1.0), max_steps=20)
    S.init(A)
    x = u.Vector(cols)
    with pytest.raises(u.UGError):
        S.apply(x, u.Vector(values=rng.normal(size=rows)))
    assert not x.numpy().any()
