"""GPU test of BiCGStab on lattice-ordered vectors (tetrahedral problems with the
multigrid of the same assembly) against the same iteration on the surface
operator, which a copy of the matrix selects (the copy is not the
discretisation's assembly): steps +-1, solutions and returned defects to what a
reduction of 1e-12 leaves; several cycles, restarts, starts with entries on the
Dirichlet DoFs, right-hand sides one after another, and an operator renewed in
between. Breakdowns end with false on both paths: with (v, r0) = 0 in the first
step x and the defect are those of the start, with (t, t) = 0 the first half
step stands; a defect that is not finite ends the iteration before x changes."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


def problem(refs, seed):
    u = U()
    d = u.DomainDiscretization(2, refs)
    rng = np.random.default_rng(seed)
    d.set_theta(0.5 * rng.normal(size=d.n_fine ** 3))
    d.set_velocity((20.0, 10.0, 5.0))
    d.set_jitter(11, 0.2 / np.sqrt(3.0))
    d.set_source(1.0)
    A, b = u.SparseMatrix(), u.Vector(d.num_dofs())
    d.assemble_linear(A, b)
    return d, A, b, rng


@pytest.mark.parametrize("refs,precision,cycle,graphs,restart", [
    (0, "f64", "V", True, 0), (1, "f32", "V", True, 0), (2, "f64", "V", True, 5), (2, "f32", "W", True, 0),
    (2, "f64", "F", False, 0), (3, "f32", "V", True, 4), (3, "f64", "V", False, 0)])
def test_lattice_path_equals_surface_path(refs, precision, cycle, graphs, restart):
    print(f"case bicgstab refs={refs} {precision} {cycle} graphs={graphs} restart={restart}", flush=True)
    sys.stdout.flush()
    u = U()
    d, A, b, rng = problem(refs, refs)
    C = u.SparseMatrix()
    C.set_as_copy_of(A)
    N = d.num_dofs()
    sol = {}
    for name, M in (("lattice", A), ("surface", C)):
        g = u.GeometricMultiGrid(d, base_level=0, omega=0.6, cycle=cycle, precision=precision, graphs=graphs)
        S = u.BiCGStab(g, max_steps=200, reduction=1e-12)
        if restart:
            S.set_restart(restart)
        S.init(M)
        sol[name] = (S, g)
    x0 = rng.normal(size=N)                      # entries on the Dirichlet DoFs too
    for start, rhs in ((np.zeros(N), b.numpy()), (x0, b.numpy()), (np.zeros(N), rng.normal(size=N))):
        got = {}
        for name, (S, _) in sol.items():
            x, r = u.Vector(values=start), u.Vector(values=rhs)
            assert S.apply_return_defect(x, r), name
            got[name] = (x.numpy(), r.numpy(), S.steps())
            y = u.Vector(values=start)
            assert S.apply(y, u.Vector(values=rhs))
            assert np.array_equal(y.numpy(), got[name][0])
        (xl, rl, kl), (xs, rs, ks) = got["lattice"], got["surface"]
        assert abs(kl - ks) <= 1
        assert np.linalg.norm(xl - xs) <= 1e-9 * np.linalg.norm(xs)
        # the returned defect is b - A x up to the recursion's rounding
        true = u.Vector(values=rhs)
        A.apply_sub(true, u.Vector(values=xl))
        scale = np.linalg.norm(rhs) + np.abs(A.download_csr()[2]).max() * np.linalg.norm(xl)
        assert np.linalg.norm(true.numpy() - rl) <= 1e-12 * scale
    # a renewed operator
    d.set_theta(0.5 * rng.normal(size=d.n_fine ** 3))
    d.assemble_linear(A, b)
    S, g = sol["lattice"]
    S.init(A)
    x = u.Vector(N)
    assert S.apply(x, b)
    C.set_as_copy_of(A)
    T = u.BiCGStab(g, max_steps=200, reduction=1e-12)
    T.init(C)
    y = u.Vector(N)
    assert T.apply(y, b)
    assert np.linalg.norm(x.numpy() - y.numpy()) <= 1e-9 * np.linalg.norm(y.numpy())


def test_limits_and_non_finite_defects():
    print("case bicgstab limits", flush=True)
    sys.stdout.flush()
    u = U()
    d, A, b, _ = problem(1, 5)
    N = d.num_dofs()
    S = u.BiCGStab(u.GeometricMultiGrid(d, base_level=0, omega=0.6), max_steps=3, reduction=1e-14)
    S.init(A)
    x = u.Vector(N)
    assert not S.apply(x, b) and S.steps() == 3
    zero = u.Vector(N)
    assert S.apply(x := u.Vector(N), zero) and S.steps() == 0 and not x.numpy().any()
    bad = b.numpy()
    bad[3] = np.nan
    assert not S.apply(u.Vector(N), u.Vector(values=bad))
    assert S.steps() <= 1
    x, r = u.Vector(values=np.full(N, 0.5)), u.Vector(values=bad)
    assert not S.apply_return_defect(x, r)
    assert np.all(x.numpy() == 0.5) and np.isnan(r.numpy()).any() and S.steps() == 0


def test_precision_set_after_init():
    """counts from the next init on (the C++ interface's setter)"""
    print("case bicgstab precision set after init", flush=True)
    sys.stdout.flush()
    import os
    import subprocess
    client = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp_client", "_build", "settings_client")
    r = subprocess.run([client, "precision"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count("equal") == 4


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("which,refs,scale", [("v.r0", 1, 1e-170), ("v.r0", 2, 1e-170), ("t.t", 0, 1e-150)])
def test_breakdowns(which, refs, scale, graphs):
    """Right-hand sides so small that a product underflows to an exact zero.
    v.r0: (v, r0) of vectors near 1e-170. t.t: the base level's LU alone is the
    preconditioner, so s = r - alpha A B r is rounding, 1e-16 of r, and
    (t, t) of t = A B s is below 1e-320 where (v, r0) near 1e-300 is not; the
    half step queued before the host has looked writes scratch only."""
    print(f"case bicgstab breakdown {which} refs={refs} graphs={graphs}", flush=True)
    sys.stdout.flush()
    u = U()
    d, A, b, rng = problem(refs, 7)
    C = u.SparseMatrix()
    C.set_as_copy_of(A)
    N = d.num_dofs()
    rhs = scale * rng.uniform(0.5, 1.5, N)
    got = {}
    for name, M in (("lattice", A), ("surface", C)):
        g = u.GeometricMultiGrid(d, base_level=0, omega=0.6, graphs=graphs)
        S = u.BiCGStab(g, max_steps=20, min_defect=0.0, reduction=0.0)
        S.init(M)
        for _ in range(2):                       # also with what the first left behind
            x, r = u.Vector(N), u.Vector(values=rhs)
            assert not S.apply_return_defect(x, r), name
            assert S.steps() == (0 if which == "v.r0" else 1), name
            assert np.array_equal(r.numpy(), rhs), name
        got[name] = x.numpy()
        # the solver is as before: an ordinary problem
        S.set_conv_check(200, 1e-50, 1e-10)
        y = u.Vector(N)
        assert S.apply(y, b), name
    if which == "v.r0":
        assert not got["lattice"].any() and not got["surface"].any()
    else:
        # x = alpha B r solves the system
        Rx = u.Vector(values=rhs)
        A.apply_sub(Rx, u.Vector(values=got["lattice"]))
        assert np.linalg.norm(Rx.numpy() / scale) <= 1e-12 * np.linalg.norm(rhs / scale)
        assert np.linalg.norm((got["lattice"] - got["surface"]) / scale) <= 1e-12 * np.linalg.norm(got["surface"] / scale)
