"""GPU test of the coarse part of the V-cycle that runs as one kernel: every
domain, hierarchies whose levels end below, at and above what one workgroup
takes, every base level, 0 - 3 smoothing steps before and after, against the
oracle's cycle (1e-12 of the correction's norm in FP64, as the separate kernels
are tested; FP32 levels: 2^-24 times the about 100 roundings of a cycle)."""
import sys

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
VEL = (20.0, 10.0, 5.0)


def problem(kind, refs):
    import ugcore_amd as U
    p = O.Problem(kind, refs)
    d = U.DomainDiscretization(kind, refs)
    if kind != 1:
        theta = O.make_theta(p.n_fine, 7, 3)
        p.set_theta(theta)
        d.set_theta(theta)
    if kind == 2:
        p.set_tet_params(vel=VEL, jitter_seed=11, jitter_amp=0.2 / np.sqrt(3.0))
        d.set_velocity(VEL)
        d.set_jitter(11, 0.2 / np.sqrt(3.0))
    p.assemble_all()
    A, b = U.SparseMatrix(), U.Vector(d.num_dofs())
    d.assemble_linear(A, b)
    return p, d, A


@pytest.mark.parametrize("kind,refs", [(0, 1), (0, 2), (0, 3), (0, 4), (1, 2), (1, 5), (1, 6), (2, 1), (2, 2), (2, 3)])
def test_coarse_cycle_matches_oracle(kind, refs):
    print(f"case coarse cycle kind={kind} refs={refs}", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    p, d, A = problem(kind, refs)
    rng = np.random.default_rng(refs)
    dv = rng.normal(size=p.num_dofs(refs))
    dv[p.dirichlet(refs) == 1] = 0.0
    omega = 0.6 if kind == 2 else 0.66
    for base in range(min(refs, 3 if kind != 2 else 1)):
        for nu1, nu2 in ((2, 2), (1, 1), (0, 2), (2, 0), (3, 1), (1, 3)):
            want = p.gmg_apply(dv, base_lev=base, nu1=nu1, nu2=nu2, omega=omega)
            for precision, tol in (("f64", 1e-12), ("f32", 100 * 2.0 ** -24)):
                g = U.GeometricMultiGrid(d, base_level=base, nu1=nu1, nu2=nu2, omega=omega, precision=precision)
                g.init(A)
                c = U.Vector(len(dv))
                for _ in range(2):              # nothing is left over from the first application
                    g.apply(c, U.Vector(values=dv))
                err = np.linalg.norm(c.numpy() - want) / np.linalg.norm(want)
                assert err <= tol, (base, nu1, nu2, precision, err)
