"""GPU test of the Q2 element kernel's pairs of elements: counts around a pair, a
workgroup and a full grid, with and without coefficient and load vector, against
the oracle's contraction over all points (FP64: 64 ulp of the entries' magnitude
|B|^T |C| |B|, bounded here by the largest entry of the element)."""
import sys

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 17, 6145])
def test_pairs_match_oracle(n):
    print(f"case q2 pairs n={n}", flush=True)
    sys.stdout.flush()
    import ugcore_amd as u
    L = u.lib()
    rng = np.random.default_rng(n)
    cube = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]], float)
    X = (cube + 0.05 * rng.normal(size=(n, 8, 3))) * rng.uniform(0.01, 10.0, size=(n, 1, 1))
    k = np.exp(rng.normal(size=n))
    dX, dk = u.DeviceArray(X.reshape(n, 24)), u.DeviceArray(k)
    pick = rng.choice(n, min(n, 40), replace=False)
    pick[-1] = n - 1
    for with_k in (True, False):
        for with_f in (True, False):
            Ke, fe = u.DeviceArray(np.full((n, 729), np.nan)), u.DeviceArray(np.full((n, 27), np.nan))
            assert L.ugx_q2_hex_element_matrices(n, dX.ptr, dk.ptr if with_k else None, 1.5, Ke.ptr,
                                                 fe.ptr if with_f else None) == 0
            u.synchronize()
            got, gf = Ke.numpy().reshape(n, 27, 27), fe.numpy()
            assert np.isfinite(got).all() and np.array_equal(got, got.transpose(0, 2, 1))
            assert np.isfinite(gf).all() == with_f
            for e in pick:
                K, f = O.q2_hex_elements(X[e:e + 1], k[e:e + 1] if with_k else None, 1.5)
                K, f = np.asarray(K).reshape(27, 27), np.asarray(f).reshape(27)
                assert np.abs(got[e] - K).max() <= 64 * 2.0 ** -52 * 27 * np.abs(K).max()
                if with_f:
                    assert np.abs(gf[e] - f).max() <= 64 * 2.0 ** -52 * np.abs(f).max() * 27
