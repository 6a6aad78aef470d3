"""GPU tests of the Q2 hierarchy against the oracle: the LEVEL numbering of
every level, the level operators (element loop with the coefficient at the
Gauss points), StdTransfer's prolongations and restrictions with their
Dirichlet adjustments, the multigrid over these matrices (V, W and F cycles,
one application and the GMG-preconditioned CG), and the generic Q2 element
loop against the lattice Q2 assembly."""
import sys

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def U():
    import ugcore_amd
    return ugcore_amd


def rows_close(rp, a, b):
    worst = 0.0
    for r in range(len(rp) - 1):
        x, y = a[rp[r]:rp[r + 1]], b[rp[r]:rp[r + 1]]
        if y.size:
            worst = max(worst, np.abs(x - y).max() / max(np.abs(y).max(), 1e-300))
    return worst


def oracle(refs, theta):
    p = O.Problem(0, refs)
    p.enable_q2()
    if theta is not None:
        p.set_theta(theta)
    p.assemble_all()
    return p


@pytest.mark.parametrize("refs", [1, 2, 3])
def test_numbering_matches_oracle(refs):
    say(f"case q2 numbering refs={refs}")
    u = U()
    q = u.Q2Discretization(refs)
    p = O.Problem(0, refs)
    p.enable_q2()
    for lev in range(refs + 1):
        pos, dr = p.q2_dofs(lev)
        X = q.dof_positions(lev)
        assert np.array_equal(np.rint(X * 2 * 2 ** refs).astype(np.int64), pos), lev
        assert np.array_equal(q.dirichlet(lev), dr), lev


@pytest.mark.parametrize("refs,seed", [(2, 3), (3, 4)])
def test_operators_and_transfers_match_oracle(refs, seed):
    say(f"case q2 hierarchy refs={refs}")
    u = U()
    theta = np.random.default_rng(seed).normal(size=8 ** refs) * 0.4
    p = oracle(refs, theta)
    q = u.Q2Discretization(refs)
    q.set_theta(theta)
    q.set_source(1.0)
    A, P, R, b = q.hierarchy()
    for lev in range(refs + 1):
        rp, col, val = A[lev].download_csr()
        o = p.A(lev)
        assert np.array_equal(rp, o.rowptr) and np.array_equal(col, o.col), lev
        assert rows_close(rp, val, o.val) <= 1e-12, lev
        if lev > 0:
            for mine, ref in ((P[lev], p.P(lev)), (R[lev], p.R(lev))):
                rp2, col2, val2 = mine.download_csr()
                assert np.array_equal(rp2, ref.rowptr) and np.array_equal(col2, ref.col), lev
                assert np.array_equal(val2, ref.val), lev
    bo = p.rhs(refs)
    assert np.abs(b.numpy() - bo).max() <= 1e-12 * np.abs(bo).max()


@pytest.mark.parametrize("refs,base,cycle", [(2, 0, 1), (3, 0, 1), (3, 1, 2), (3, 0, -1)])
def test_multigrid_matches_oracle(refs, base, cycle):
    say(f"case q2 multigrid refs={refs} base={base} cycle={cycle}")
    u = U()
    theta = np.random.default_rng(refs + 10).normal(size=8 ** refs) * 0.4
    p = oracle(refs, theta)
    q = u.Q2Discretization(refs)
    q.set_theta(theta)
    q.set_source(1.0)
    A, P, R, b = q.hierarchy()
    N = q.num_dofs(refs)
    dr = q.dirichlet(refs)
    d = np.random.default_rng(1).normal(size=N)
    d[dr == 1] = 0.0
    G = u.MatrixMultiGrid(A, P, R, base_level=base, nu1=2, nu2=2, cycle=cycle, omega=0.66)
    G.init(A[refs])
    c = u.Vector(N)
    G.apply(c, u.Vector(values=d))
    co = p.gmg_apply(d, base_lev=base, nu1=2, nu2=2, cycle=cycle, omega=0.66)
    assert np.abs(c.numpy() - co).max() <= 1e-11 * np.abs(co).max()
    # the preconditioned CG
    ro = p.solve(base_lev=base, cycle=cycle, rel_red=1e-10)
    S = u.CG(G, max_steps=100, reduction=1e-10)
    S.init(A[refs])
    x = u.Vector(N)
    assert S.apply(x, b)
    assert S.steps() == ro["steps"]
    assert np.abs(x.numpy() - ro["x"]).max() <= 1e-9 * np.abs(ro["x"]).max()


def test_generic_q2_element_loop_equals_the_lattice_assembly():
    """ElementDiscretization('hexahedron_q2') fed the lattice connectivity
    (nodes x fastest) gives the lattice Q2 assembly; its defect is A u - b"""
    say("case q2 generic vs lattice")
    u = U()
    n = 4
    W = 2 * n + 1
    theta = np.random.default_rng(7).normal(size=n ** 3) * 0.3
    mi = O.q2_hex_multi_index()
    E = []
    for ez in range(n):
        for ey in range(n):
            for ex in range(n):
                E.append([((2 * ez + m[2]) * W + (2 * ey + m[1])) * W + (2 * ex + m[0]) for m in mi])
    E = np.array(E, np.int32)
    g = np.arange(W) / (2.0 * n)
    X = np.stack(np.meshgrid(g, g, g, indexing="ij")[::-1], -1).reshape(-1, 3)
    bnd = np.flatnonzero(np.any((X == 0) | (X == 1), axis=1)).astype(np.int32)
    e = u.ElementDiscretization("hexahedron_q2", E, X)
    e.set_dirichlet(bnd)
    e.set_diffusion(np.exp(theta))
    e.set_source(1.0)
    A, b = u.SparseMatrix(), u.Vector(W ** 3)
    e.assemble_linear(A, b)
    L, bl = u.q2_assemble_lattice(n, theta, 1.0)
    rp, col, val = A.download_csr()
    rl, cl, vl = L.download_csr()
    assert np.array_equal(rp, rl) and np.array_equal(col, cl)
    assert rows_close(rp, val, vl) <= 1e-12
    assert np.abs(b.numpy() - bl.numpy()).max() <= 1e-12 * np.abs(bl.numpy()).max()
    # the coefficient at the Gauss points (here constant per element) gives the same
    e.set_diffusion_at_points(np.repeat(np.exp(theta), 27))
    A2, b2 = u.SparseMatrix(), u.Vector(W ** 3)
    e.assemble_linear(A2, b2)
    assert rows_close(rp, A2.download_csr()[2], val) <= 1e-15
    # defect
    x = np.random.default_rng(2).normal(size=W ** 3)
    d = u.Vector(W ** 3)
    e.assemble_defect(d, u.Vector(values=x))
    import scipy.sparse as sp
    S = sp.csr_matrix((val, col, rp), shape=(W ** 3, W ** 3))
    ref = S @ x - b.numpy()
    ref[bnd] = 0.0
    assert np.abs(d.numpy() - ref).max() <= 1e-12 * np.abs(ref).max()


def test_pybind_q2_multigrid_solve_equals_the_ctypes_path():
    say("case q2 ug4py")
    u = U()
    from ugcore_amd import ug4py as P
    refs = 2
    theta = np.random.default_rng(9).normal(size=8 ** refs) * 0.3
    P.init()
    q = P.Q2Discretization(refs)
    q.set_theta(theta)
    q.set_source(1.0)
    A, Pm, Rm = [], [None], [None]
    b = None
    for lev in range(refs + 1):
        a, bv = P.SparseMatrix(), P.Vector(q.num_dofs(lev))
        q.assemble_linear(lev, a, bv)
        A.append(a)
        b = bv
        if lev:
            p, r = P.SparseMatrix(), P.SparseMatrix()
            q.prolongation(lev, p)
            q.restriction(lev, p, r)
            Pm.append(p)
            Rm.append(r)
    G = P.MatrixMultiGrid(A, Pm, Rm, base_level=0)
    S = P.CG(G, 100, 1e-10, 1e-50)
    S.init(A[refs])
    x = P.Vector(q.num_dofs(refs))
    assert S.apply(x, b)
    # the ctypes path
    q2 = u.Q2Discretization(refs)
    q2.set_theta(theta)
    q2.set_source(1.0)
    A2, P2, R2, b2 = q2.hierarchy()
    S2 = u.CG(u.MatrixMultiGrid(A2, P2, R2), max_steps=100, reduction=1e-10)
    S2.init(A2[refs])
    x2 = u.Vector(q2.num_dofs(refs))
    assert S2.apply(x2, b2)
    assert S.steps() == S2.steps()
    assert np.array_equal(x.numpy(), x2.numpy())


@pytest.mark.parametrize("cycle", [1, 2])
def test_matrix_multigrid_initialised_again_with_other_sizes(cycle):
    """the same object after its level matrices took larger (then smaller) ones
    of another hierarchy of the same depth: every correction is, bit for bit,
    that of a new object"""
    print(f"case matrix multigrid initialised again cycle={cycle}", flush=True)
    u = U()
    rng = np.random.default_rng(cycle)
    q = u.Q2Discretization(3)
    q.set_theta(0.4 * rng.normal(size=8 ** 3))
    q.set_source(1.0)
    A, P, R, _ = q.hierarchy()
    data = [[(m.download_csr(), m.num_cols()) if m is not None else None for m in ms] for ms in (A, P, R)]
    mats = [[u.SparseMatrix() if l or k == 0 else None for l in range(3)] for k in range(3)]
    G = u.MatrixMultiGrid(*mats, base_level=0, cycle=cycle)
    for first in (0, 1, 0):
        for k in range(3):
            for l in range(3):
                if mats[k][l] is not None:
                    (rp, col, val), cols = data[k][first + l]
                    mats[k][l].upload_csr(rp, col, val, n_cols=cols)
        G.init(mats[0][-1])
        F = u.MatrixMultiGrid(*mats, base_level=0, cycle=cycle)
        F.init(mats[0][-1])
        n = mats[0][-1].num_rows()
        d = u.Vector(values=rng.normal(size=n))
        c, ref = u.Vector(n), u.Vector(n)
        for _ in range(2):
            G.apply(c, d)
            F.apply(ref, d)
            assert np.array_equal(c.numpy(), ref.numpy()), first
        assert np.linalg.norm(ref.numpy()) > 0


def test_matrix_multigrid_base_level_lowered():
    """another base level on the same object (an option of the C++ interface)"""
    print("case matrix multigrid base level lowered", flush=True)
    import os
    import subprocess
    client = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp_client", "_build", "settings_client")
    r = subprocess.run([client, "base_level"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.count("equal") == 6


@pytest.mark.parametrize("which,level", [(0, 1), (0, 2), (1, 2), (2, 2), (1, 1)])
def test_matrix_multigrid_refuses_levels_replaced_after_init(which, level):
    """a level matrix (0: operator, 1: prolongation, 2: restriction) replaced by
    a larger one needs a new init: apply raises and launches nothing"""
    print(f"case matrix multigrid level replaced which={which} level={level}", flush=True)
    u = U()
    rng = np.random.default_rng(level)
    q = u.Q2Discretization(3)
    q.set_source(1.0)
    A, P, R, _ = q.hierarchy()
    mats = [[u.SparseMatrix() if l or k == 0 else None for l in range(3)] for k in range(3)]

    def fill(k, l, shift):
        m = (A, P, R)[k][l + shift]
        rp, col, val = m.download_csr()
        mats[k][l].upload_csr(rp, col, val, n_cols=m.num_cols())

    for k in range(3):
        for l in range(3):
            if mats[k][l] is not None:
                fill(k, l, 0)
    G = u.MatrixMultiGrid(*mats, base_level=0)
    G.init(mats[0][-1])
    n = mats[0][-1].num_rows()
    d, c = u.Vector(values=rng.normal(size=n)), u.Vector(n)
    G.apply(c, d)
    want = c.numpy()
    fill(which, level, 1)
    c.set(-7.0)
    with pytest.raises(u.UGError):
        G.apply(c, d)
    assert np.all(c.numpy() == -7.0)
    fill(which, level, 0)
    G.init(mats[0][-1])
    G.apply(c, d)
    assert np.array_equal(c.numpy(), want)


def test_restriction_with_an_empty_row_adds_nothing():
    """a coarse DoF that nothing is restricted to keeps its level's defect
    (apply_ignore_zero_rows), which is zero after init, whatever the memory of
    that vector held before"""
    print("case matrix multigrid empty restriction row", flush=True)
    u = U()
    import scipy.sparse as sp
    rng = np.random.default_rng(4)
    sizes = [9, 19, 39]
    mats = [[None] * 3 for _ in range(3)]

    def up(M):
        M = M.tocsr()
        M.sort_indices()
        m = u.SparseMatrix()
        m.upload_csr(M.indptr, M.indices, M.data, n_cols=M.shape[1])
        return m

    csr = [sp.diags([-np.ones(n - 1), 2.5 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1]) for n in sizes]
    for l, n in enumerate(sizes):
        mats[0][l] = up(csr[l])
        if l:
            m = sizes[l - 1]
            Pm = sp.lil_matrix((n, m))
            for j in range(m):
                Pm[2 * j + 1, j] = 1.0
                Pm[2 * j, j] = Pm[2 * j + 2, j] = 0.5
            Rm = Pm.T.tocsr()
            Rm.data[Rm.indptr[3]:Rm.indptr[4]] = 0.0
            Rm.eliminate_zeros()
            mats[1][l], mats[2][l] = up(Pm), up(Rm)
    dv = rng.normal(size=sizes[-1])
    got = []
    for layout in ("sell", "csr"):          # the fused and the separate steps
        mats[1][2].set_spmv_layout(layout)
        for value in (0.0, np.nan, 3.0):
            old = [u.Vector(values=np.full(n, value)) for n in sizes for _ in range(8)]
            u.synchronize()
            del old                         # what the next buffers of these sizes hold
            G = u.MatrixMultiGrid(*mats, base_level=0)
            G.init(mats[0][-1])
            c = u.Vector(sizes[-1])
            G.apply(c, u.Vector(values=dv))
            got.append(c.numpy())
    for g in got[1:]:
        assert np.linalg.norm(g - got[0]) <= 1e-13 * np.linalg.norm(got[0])
    assert np.linalg.norm(got[0]) > 0
