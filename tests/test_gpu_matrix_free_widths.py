"""GPU test of the matrix-free Q1 kernels at every width of their two schedules
(one row per thread up to 65^3, the march at 129^3): the lattice operator
against the element sum in numpy (43 operations a row: 64 ulp of the sum of the
magnitudes), also for vectors that do not vanish on the boundary, and a V(2,2)
application with matrix-free against stored top level (FP64: the stored entries
carry the quadrature's rounding; FP32: 2^-24 times the about 100 roundings of a
cycle)."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def U():
    import ugcore_amd
    return ugcore_amd


def element_sum(k, x):
    """(A x, sum of magnitudes) of sum_e h k_e K_ref; boundary rows identity"""
    n = k.shape[0]
    m = np.array([[2.0, 1.0], [1.0, 2.0]]) / 6
    s = np.array([[1.0, -1.0], [-1.0, 1.0]])
    K = np.kron(m, np.kron(m, s)) + np.kron(m, np.kron(s, m)) + np.kron(s, np.kron(m, m))
    K[np.abs(K) < 1e-14] = 0.0
    sl = [(slice(c >> 2, n + (c >> 2)), slice((c >> 1) & 1, n + ((c >> 1) & 1)), slice(c & 1, n + (c & 1)))
          for c in range(8)]
    y, a = np.zeros_like(x), np.zeros_like(x)
    for p in range(8):
        for q in range(8):
            if K[p, q] != 0.0:
                t = k / n * K[p, q] * x[sl[q]]
                y[sl[p]] += t
                a[sl[p]] += np.abs(t)
    out, mag = x.copy(), np.abs(x)
    i = (slice(1, n),) * 3
    out[i], mag[i] = y[i], a[i]
    return out, mag


@pytest.mark.parametrize("refs", [1, 2, 3, 4, 5, 6, 7])
def test_lattice_operator(refs):
    print(f"case matrix-free operator refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    n = 2 ** refs
    N = (n + 1) ** 3
    rng = np.random.default_rng(refs)
    d = u.DomainDiscretization(0, refs)
    theta = 0.5 * rng.normal(size=n ** 3)
    d.set_theta(theta)
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    L = u.lib()
    for precision in ("f64", "f32"):
        g = u.GeometricMultiGrid(d, base_level=0, precision=precision)
        g.init(A)
        H = L.ugx_gmg_lattice_halo(g.h)
        for boundary in (False, True):
            x = rng.normal(size=(n + 1,) * 3)
            if not boundary:
                z = np.zeros_like(x)
                z[1:n, 1:n, 1:n] = x[1:n, 1:n, 1:n]
                x = z
            xd = u.DeviceArray(np.concatenate([np.zeros(H), x.ravel(), np.zeros(H)]))
            yd = u.DeviceArray(np.full(N, np.nan))
            assert L.ugx_gmg_surface_apply_lattice(g.h, yd.ptr, xd.ptr + 8 * H) == 0
            u.synchronize()
            want, mag = element_sum(np.exp(theta).reshape(n, n, n), x)
            assert np.all(np.abs(yd.numpy().reshape(want.shape) - want) <= 64 * 2.0 ** -52 * mag)
            # the direction update: p = z + beta p_old, y = A p, (y, p)
            zv = rng.normal(size=x.shape)
            zd = u.DeviceArray(np.concatenate([np.zeros(H), zv.ravel(), np.zeros(H)]))
            pd = u.DeviceArray(np.zeros(N + 2 * H))
            beta, qp, part = u.DeviceArray(np.array([0.75])), u.DeviceArray(np.zeros(1)), u.DeviceArray(np.zeros(65536))
            assert L.ugx_gmg_surface_direction_lattice(g.h, yd.ptr, xd.ptr + 8 * H, zd.ptr + 8 * H, beta.ptr,
                                                       pd.ptr + 8 * H, qp.ptr, part.ptr) == 0
            u.synchronize()
            p = pd.numpy()[H:H + N].reshape(x.shape)
            assert np.all(np.abs(p - (zv + 0.75 * x)) <= 2.0 ** -51 * (np.abs(zv) + np.abs(x)))
            want, mag = element_sum(np.exp(theta).reshape(n, n, n), p)
            assert np.all(np.abs(yd.numpy().reshape(want.shape) - want) <= 64 * 2.0 ** -52 * mag)
            assert abs(qp.numpy()[0] - np.sum(want * p)) <= 128 * 2.0 ** -52 * np.sum(mag * np.abs(p))


@pytest.mark.parametrize("refs", [2, 5, 6, 7, 8])
def test_cycle_with_matrix_free_and_stored_top_level(refs):
    print(f"case matrix-free cycle refs={refs}", flush=True)
    sys.stdout.flush()
    u = U()
    n = 2 ** refs
    rng = np.random.default_rng(refs)
    d = u.DomainDiscretization(0, refs)
    d.set_theta(0.5 * rng.normal(size=n ** 3))
    N = d.num_dofs()
    A, b = u.SparseMatrix(), u.Vector(N)
    d.assemble_linear(A, b)
    dv = rng.normal(size=N)
    dv[d.num_inner():] = 0.0
    for precision, tol in (("f64", 1e-12), ("f32", 100 * 2.0 ** -24)):
        if refs == 8 and precision == "f64":
            continue
        got = []
        for mf in (True, False):
            g = u.GeometricMultiGrid(d, base_level=min(2, refs - 1), precision=precision, matrix_free=mf)
            g.init(A)
            c = u.Vector(N)
            g.apply(c, u.Vector(values=dv))
            got.append(c.numpy())
        assert np.linalg.norm(got[0] - got[1]) <= tol * np.linalg.norm(got[1]), precision


def test_lattice_operator_at_257():
    """The marching width of 257 on planes at its ends and inside: the row sums of
    a plane need the two element layers beside it."""
    print("case matrix-free operator 257", flush=True)
    sys.stdout.flush()
    u = U()
    n = 256
    W = n + 1
    rng = np.random.default_rng(8)
    d = u.DomainDiscretization(0, 8)
    theta = 0.5 * rng.normal(size=n ** 3)
    d.set_theta(theta)
    A, b = u.SparseMatrix(), u.Vector(W ** 3)
    d.assemble_linear(A, b)
    L = u.lib()
    g = u.GeometricMultiGrid(d, base_level=2, precision="f32")
    g.init(A)
    H = L.ugx_gmg_lattice_halo(g.h)
    x = rng.normal(size=(W, W, W))
    xd = u.DeviceArray(np.concatenate([np.zeros(H), x.ravel(), np.zeros(H)]))
    yd = u.DeviceArray(np.full(W ** 3, np.nan))
    assert L.ugx_gmg_surface_apply_lattice(g.h, yd.ptr, xd.ptr + 8 * H) == 0
    u.synchronize()
    y = yd.numpy().reshape(W, W, W)
    k = np.exp(theta).reshape(n, n, n)
    assert np.array_equal(y[[0, n]], x[[0, n]])
    for z in (1, 2, 31, 32, 33, 36, 37, 64, 73, 110, 128, 147, 183, 200, 220, n - 1):
        s, mag = layer_sum(k[z - 1:z + 1], x[z - 1:z + 2])
        assert np.all(np.abs(y[z] - s) <= 64 * 2.0 ** -52 * mag), z


def layer_sum(k, x):
    """rows of the middle of three planes (identity on its boundary) and magnitudes"""
    n = k.shape[1]
    m = np.array([[2.0, 1.0], [1.0, 2.0]]) / 6
    s = np.array([[1.0, -1.0], [-1.0, 1.0]])
    K = np.kron(m, np.kron(m, s)) + np.kron(m, np.kron(s, m)) + np.kron(s, np.kron(m, m))
    K[np.abs(K) < 1e-14] = 0.0
    y, a = np.zeros((n + 1, n + 1)), np.zeros((n + 1, n + 1))
    for lay in (0, 1):
        for p in range(8):
            if lay + (p >> 2) != 1:
                continue
            py, px = (p >> 1) & 1, p & 1
            for q in range(8):
                if K[p, q] != 0.0:
                    qz, qy, qx = q >> 2, (q >> 1) & 1, q & 1
                    t = k[lay] / n * K[p, q] * x[lay + qz, qy:n + qy, qx:n + qx]
                    y[py:n + py, px:n + px] += t
                    a[py:n + py, px:n + px] += np.abs(t)
    out, mag = x[1].copy(), np.abs(x[1])
    out[1:n, 1:n], mag[1:n, 1:n] = y[1:n, 1:n], a[1:n, 1:n]
    return out, mag
