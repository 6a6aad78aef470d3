"""GPU test of the transposed product at the edges of its workgroups: row
counts around the 64 rows of a workgroup and the 8-fold block order, empty
transposed rows, a transposed row longer than one staged chunk of 1024 entries,
every alpha case and dest aliasing v1, against numpy in extended precision.
Tolerance per row: a sum of m products in FP64 is off by at most (m + 2) ulp of
the sum of the magnitudes."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,long_row", [(1, 1, False), (3, 63, False), (200, 64, False), (70, 65, False),
                                                (2500, 130, True), (900, 64 * 64 + 1, False), (3000, 5001, True)])
def test_transposed_product_at_workgroup_edges(rows, cols, long_row):
    print(f"case transposed product rows={rows} cols={cols} long={long_row}", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    rng = np.random.default_rng(rows + cols)
    r = rng.integers(0, rows, 6 * max(rows, cols))
    c = rng.integers(0, max(1, cols - cols // 5), r.size)      # the last columns stay empty
    if long_row:
        r = np.concatenate([r, np.arange(rows)])
        c = np.concatenate([c, np.full(rows, cols // 3)])      # one transposed row with every source row
    key = np.unique(r * cols + c)
    r, c = key // cols, key % cols
    v = rng.normal(size=r.size)
    rp = np.zeros(rows + 1, np.int64)
    rp[1:] = np.cumsum(np.bincount(r, minlength=rows))
    A = U.SparseMatrix()
    A.upload_csr(rp, c, v, n_cols=cols)
    w, v1 = rng.normal(size=rows), rng.normal(size=cols)
    m = np.bincount(c, minlength=cols)
    for alpha, beta in ((0.0, 1.0), (1.0, -1.0), (0.5, 2.0)):
        ref = alpha * v1.astype(np.longdouble)
        np.add.at(ref, c, np.longdouble(beta) * v.astype(np.longdouble) * w[r].astype(np.longdouble))
        size = np.abs(alpha * v1)
        np.add.at(size, c, np.abs(beta * v * w[r]))
        for alias in (False, True):
            d = U.Vector(values=v1 if alias else rng.normal(size=cols))
            A.axpy_transposed(d, alpha, d if alias else U.Vector(values=v1), beta, U.Vector(values=w))
            err = np.abs(d.numpy() - ref.astype(np.float64))
            assert np.all(err <= (m + 2) * 2.0 ** -52 * size), (alpha, alias, float(err.max()))
