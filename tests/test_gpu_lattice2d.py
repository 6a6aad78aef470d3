"""GPU test of the triangular hierarchy's lattice kernels at widths around a
workgroup of 256 points: one cycle against the oracle's (transfers with and
without the folded correction update), and CG, whose first smoothing step reads
the FP64 defect and whose product leaves its partial sums, against the CG on the
surface operator, with and without pre-smoothing."""
import sys

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


@pytest.mark.parametrize("refs", [1, 2, 3, 4, 5])
def test_cycle_matches_oracle(refs):
    print(f"case 2d cycle refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(refs)
    p = O.Problem(1, refs)
    p.assemble_all()
    d = u.DomainDiscretization(1, refs)
    N = d.num_dofs()
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    dv = rng.normal(size=N)
    dv[d.num_inner():] = 0.0
    for cycle in (1, 2):
        for nu1, nu2 in ((2, 2), (0, 1), (1, 3), (2, 0)):
            ref = p.gmg_apply(dv, base_lev=0, nu1=nu1, nu2=nu2, cycle=cycle, omega=0.66)
            for precision, tol in (("f64", 1e-12), ("f32", 100 * 2.0 ** -24)):
                g = u.GeometricMultiGrid(d, base_level=0, nu1=nu1, nu2=nu2, cycle=cycle, precision=precision)
                g.init(A)
                c = u.Vector(N)
                g.apply(c, u.Vector(values=dv))
                assert np.linalg.norm(c.numpy() - ref) <= tol * np.linalg.norm(ref), (cycle, nu1, nu2, precision)


@pytest.mark.parametrize("refs", [1, 2, 4, 5, 7])
@pytest.mark.parametrize("nu1,nu2", [(2, 2), (0, 2), (1, 1)])
def test_cg_equals_surface_cg(refs, nu1, nu2):
    print(f"case 2d cg refs={refs} nu={nu1},{nu2}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(refs)
    d = u.DomainDiscretization(1, refs)
    N, ni = d.num_dofs(), d.num_inner()
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    rhs = rng.normal(size=N)
    rhs[ni:] = 0.0
    for precision in ("f64", "f32"):
        for graphs in (True, False):
            got = []
            for on in (True, False):
                g = u.GeometricMultiGrid(d, base_level=0, nu1=nu1, nu2=nu2, precision=precision, graphs=graphs)
                S = u.CG(g, max_steps=200, reduction=1e-11)
                S.set_lattice_path(on)
                S.init(A)
                x = u.Vector(N)
                assert S.apply(x, u.Vector(values=rhs))
                assert S.used_lattice_path() == on
                got.append(x.numpy())
            assert np.linalg.norm(got[0] - got[1]) <= 1e-8 * np.linalg.norm(got[1])
