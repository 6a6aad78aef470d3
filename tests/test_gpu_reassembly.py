"""GPU test of the re-assembly of the Q1 lattice operator in one pass: values,
load vector and products equal those of a fresh assembly bit for bit at every
small width (blocks of four points cut by the lattice's end), in both
numberings, for a matrix whose layout was switched or given slices of the
caller's own, and for k = 1; and of the multigrid's level operators set up in one
pass: every level against the ones of an hierarchy with Galerkin products off and
the stored form read back."""
import sys

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


@pytest.mark.parametrize("refs", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("ordering", ["reference", "lex"])
def test_reassembly_equals_fresh_assembly(refs, ordering):
    print(f"case re-assembly refs={refs} {ordering}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(refs)
    d = u.DomainDiscretization(0, refs, ordering=ordering)
    N = d.num_dofs()
    x = u.Vector(values=rng.normal(size=N))
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)                      # k = 1
    for k in range(5):
        if k == 2:
            A.set_spmv_layout("sell")
        if k == 3:
            A.set_spmv_layout("dict")
        if k == 4:                               # slices in DoF order: they may not fit a dictionary
            order = np.full((N + 63) // 64 * 64, -1, np.int32)
            order[:N] = rng.permutation(N)
            A.set_slice_order(order)
        if k:
            d.set_theta(rng.normal(size=8 ** refs))
        d.set_source(1.0 + k)
        d.assemble_linear(A, b)
        F, f = u.SparseMatrix(), u.Vector(N)
        d.assemble_linear(F, f)
        assert all(np.array_equal(p, q) for p, q in zip(A.download_csr(), F.download_csr()))
        assert np.array_equal(b.numpy(), f.numpy())
        y, z = u.Vector(N), u.Vector(N)
        A.apply(y, x)
        F.apply(z, x)
        assert np.allclose(y.numpy(), z.numpy(), rtol=0, atol=1e-14 * np.abs(z.numpy()).max())
        # the fresh matrix took the pattern over: the next assembly into A renews it
        d.assemble_linear(A, b)


@pytest.mark.parametrize("refs", [1, 2, 3, 4])
def test_levels_match_oracle(refs):
    print(f"case level operators refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    theta = O.make_theta(2 ** refs, 3, 2)
    p = O.Problem(0, refs)
    p.set_theta(theta)
    p.assemble_all()
    d = u.DomainDiscretization(0, refs)
    d.set_theta(theta)
    A, b = u.SparseMatrix(), u.Vector(d.num_dofs())
    d.assemble_linear(A, b)
    for precision, tol in (("f64", 1e-12), ("f32", 2.0 ** -23)):
        for mf in (True, False):
            g = u.GeometricMultiGrid(d, base_level=0, precision=precision, matrix_free=mf)
            g.init(A)
            for lev in range(1, refs + 1):
                W = 2 ** lev + 1
                dia = g.level_dia(lev)
                dol = d.dof_of_lattice(lev)
                R = p.A(lev).to_scipy().toarray()[np.ix_(dol, dol)]
                bnd = np.array([x in (0, W - 1) or y in (0, W - 1) or z in (0, W - 1)
                                for z in range(W) for y in range(W) for x in range(W)])
                E = R.copy()
                E[np.ix_(~bnd, bnd)] = 0.0       # Dirichlet columns eliminated
                got = np.zeros_like(E)
                for k in range(27):
                    off = k % 3 - 1 + (k // 3 % 3 - 1) * W + (k // 9 - 1) * W * W
                    for i in range(W ** 3):
                        if dia[k, i] != 0.0:
                            got[i, i + off] += dia[k, i]
                assert np.abs(got - E).max() <= tol * np.abs(E).max(), (precision, mf, lev)
