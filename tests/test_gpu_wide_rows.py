"""GPU test of the sliced-ELL product where one slice is shared by four waves
(rows of more than 32 entries) at its edges: row counts around 64, widths
around the quarter and the eight entries a wave keeps in flight, empty rows,
alpha / beta / ignore-zero-rows, against numpy in extended precision (a sum of m
products: m + 4 ulp of the sum of the magnitudes); and of the multigrid cycle
over matrices in fused steps against the same cycle in separate steps, which a
level in the CSR layout selects."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


@pytest.mark.parametrize("rows,width", [(1, 33), (63, 35), (64, 36), (65, 63), (130, 125), (1000, 64), (7, 200),
                                        (300, 32), (300, 1)])
def test_wide_rows(rows, width):
    print(f"case wide rows rows={rows} width={width}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(rows + width)
    cols = 400
    ln = np.minimum(rng.integers(0, width + 1, rows), cols)
    ln[rng.integers(rows)] = width
    c = np.concatenate([np.sort(rng.choice(cols, k, replace=False)) for k in ln]) if ln.sum() else np.zeros(0, int)
    rp = np.concatenate([[0], np.cumsum(ln)])
    r = np.repeat(np.arange(rows), ln)
    v = rng.normal(size=c.size)
    A = u.SparseMatrix()
    A.upload_csr(rp, c, v, n_cols=cols)
    assert A.spmv_layout() == "sell"
    x, w = rng.normal(size=cols), rng.normal(size=rows)
    s, mag = np.zeros(rows, np.longdouble), np.zeros(rows)
    np.add.at(s, r, v.astype(np.longdouble) * x[c])
    np.add.at(mag, r, np.abs(v * x[c]))
    for alpha, beta in ((0.0, 1.0), (1.0, -1.0), (0.5, 2.0)):
        y = u.Vector(values=rng.normal(size=rows))
        A.axpy(y, alpha, u.Vector(values=w), beta, u.Vector(values=x))
        ref = (alpha * w.astype(np.longdouble) + beta * s).astype(np.float64)
        assert np.all(np.abs(y.numpy() - ref) <= (ln + 4) * 2.0 ** -52 * (np.abs(alpha * w) + abs(beta) * mag))
    y = u.Vector(values=w)
    assert u.lib().ugx_matrix_apply_ignore_zero_rows(A.h, y.h, 2.0, u.Vector(values=x).h) >= 0
    u.synchronize()
    ref = np.where(ln > 0, (2 * s).astype(np.float64), w)
    assert np.all(np.abs(y.numpy() - ref) <= (ln + 4) * 2.0 ** -52 * 2 * mag)


@pytest.mark.parametrize("refs", [1, 2, 3])
def test_fused_matrix_cycle_equals_separate_steps(refs):
    print(f"case fused matrix cycle refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    rng = np.random.default_rng(refs)
    q = u.Q2Discretization(refs)
    q.set_theta(0.4 * rng.normal(size=8 ** refs))
    q.set_source(1.0)
    A, P, R, b = q.hierarchy()
    N = b.size()
    dv = rng.normal(size=N)
    for base in range(refs):
        for cycle in (1, 2, -1, 3):
            for nu1, nu2 in ((2, 2), (1, 0), (0, 2), (3, 1)):
                got = []
                for layout in ("sell", "csr"):
                    P[refs].set_spmv_layout(layout)
                    G = u.MatrixMultiGrid(A, P, R, base_level=base, nu1=nu1, nu2=nu2, cycle=cycle)
                    G.init(A[-1])
                    c = u.Vector(values=rng.normal(size=N))
                    for _ in range(2):
                        G.apply(c, u.Vector(values=dv))
                    got.append(c.numpy())
                # about 20 sums of up to 125 terms deep, in another order
                assert np.linalg.norm(got[0] - got[1]) <= 1e-12 * np.linalg.norm(got[1]), (base, cycle, nu1, nu2)
    P[refs].set_spmv_layout("sell")


def test_cg_with_device_scalars_on_an_uploaded_matrix():
    print("case cg device scalars", flush=True)
    sys.stdout.flush()
    u = U()
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl
    rng = np.random.default_rng(1)
    n = 700
    B = sp.random(n, n, 0.02, random_state=3, format="csr")
    M = (B @ B.T + sp.identity(n) * 4).tocsr()
    M.sort_indices()
    A = u.SparseMatrix()
    A.upload_csr(M.indptr, M.indices, M.data)
    f = rng.normal(size=n)
    ref = spl.spsolve(M.tocsc(), f)
    for pre in (None, u.Jacobi(1.0)):
        S = u.CG(pre, max_steps=500, reduction=1e-12)
        S.init(A)
        x, r = u.Vector(n), u.Vector(values=f)
        assert S.apply_return_defect(x, r)
        assert np.linalg.norm(x.numpy() - ref) <= 1e-10 * np.linalg.norm(ref)
        assert len(S.defects()) == S.steps() + 1
        assert np.linalg.norm(r.numpy()) == pytest.approx(S.defects()[-1], rel=1e-12)
