"""GPU test of the element assembly at the sizes where its launches and lists
have edges: element counts around the 128 threads of a workgroup, a DoF shared
by many elements (long lists), DoFs without any element (zero right-hand side
and defect, empty rows), matrix, load vector and defect of random triangles and
tetrahedra against numpy. Tolerance: the local integrals are a few dozen
operations on the inverse of the element's Jacobian, known to cond(J) ulp (64
cond(J) ulp of the entry's magnitude); a list of m terms adds m ulp."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def p1(X, k):
    """P1 stiffness and equal shares of the volume (the box method's matrix and load)"""
    dim = X.shape[2]
    J = (X[:, 1:] - X[:, :1]).transpose(0, 2, 1)
    vol = np.abs(np.linalg.det(J)) / (2.0 if dim == 2 else 6.0)
    g = np.linalg.inv(J)
    g = np.concatenate([-g.sum(1, keepdims=True), g], 1)
    return np.einsum("n,nar,nbr->nab", vol * k, g, g), np.repeat(vol[:, None] / (dim + 1), dim + 1, 1), g, vol


@pytest.mark.parametrize("kind,ne,hub", [("triangle_fv1", 1, 0), ("triangle_fv1", 127, 40), ("triangle_fv1", 128, 0),
                                         ("triangle_fv1", 129, 50), ("triangle_fv1", 3001, 50),
                                         ("tetrahedron_fv1", 1, 0), ("tetrahedron_fv1", 129, 25),
                                         ("tetrahedron_fv1", 1000, 25)])
def test_gathered_assembly(kind, ne, hub):
    print(f"case gathered assembly {kind} ne={ne} hub={hub}", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    dim = 2 if kind == "triangle_fv1" else 3
    nv = dim + 1
    rng = np.random.default_rng(ne)
    n = max(nv + 3, ne // 2 + 3)
    E = np.stack([rng.choice(n - 2, nv, replace=False) for _ in range(4 * ne + 50)]) if n < 400 else \
        np.concatenate([rng.integers(0, n - 2, (4 * ne + 50, nv))])
    E = E[[len(set(e)) == nv for e in E]]
    X = rng.uniform(size=(n, dim))
    vol = np.abs(np.linalg.det(X[E][:, 1:] - X[E][:, :1]))
    E = E[vol > 0.05 if dim == 2 else vol > 0.02][:ne]
    if hub:
        E[:hub, 0] = np.where((E[:hub, 1:] == 0).any(1), E[:hub, 0], 0)
        ok = [len(set(e)) == nv for e in E]
        ok = ok & (np.abs(np.linalg.det(X[E][:, 1:] - X[E][:, :1])) > 1e-3)
        E = E[ok]
    # the reference tetrahedron's orientation
    neg = np.linalg.det((X[E][:, 1:] - X[E][:, :1])) < 0
    E[neg, 1], E[neg, 2] = E[neg, 2].copy(), E[neg, 1].copy()
    ne = E.shape[0]
    assert ne > 0
    k = np.exp(rng.normal(size=ne))
    ed = U.ElementDiscretization(kind, E, X)
    ed.set_diffusion(k)
    ed.set_source(1.5)
    A, b, d = U.SparseMatrix(), U.Vector(n), U.Vector(values=np.full(n, np.nan))
    u = rng.normal(size=n)
    Ke, fe, g, vol = p1(X[E], k)
    fe = 1.5 * fe
    R = np.zeros((n, n))
    S = np.zeros((n, n))
    # an entry adds fluxes |grad phi_b| |n| through the box faces of node a, |n| <= 3 vol max |grad phi|
    gn = np.linalg.norm(g, axis=2)
    scale = np.einsum("n,na,nb->nab", 3.0 * vol * k, np.broadcast_to(gn.max(1, keepdims=True), gn.shape), gn)
    scale *= np.linalg.cond((X[E][:, 1:] - X[E][:, :1]))[:, None, None]
    rb, rd, sd, m = np.zeros(n), np.zeros(n), np.zeros(n), np.zeros(n)
    for a in range(nv):
        for c in range(nv):
            np.add.at(R, (E[:, a], E[:, c]), Ke[:, a, c])
            np.add.at(S, (E[:, a], E[:, c]), scale[:, a, c])
        np.add.at(rb, E[:, a], fe[:, a])
        np.add.at(rd, E[:, a], (Ke[:, a] * u[E]).sum(1) - fe[:, a])
        np.add.at(sd, E[:, a], (scale[:, a] * np.abs(u[E])).sum(1) + np.abs(fe[:, a]))
        np.add.at(m, E[:, a], 1.0)
    eps = 2.0 ** -52
    for _ in range(2):                  # the second time into the kept pattern
        ed.assemble_linear(A, b)
        rp, col, val = A.download_csr()
        row = np.repeat(np.arange(n), np.diff(rp))
        assert np.all(np.abs(val - R[row, col]) <= (64 + m[row]) * eps * S[row, col])
        assert np.count_nonzero(S) == val.size
        assert np.all(np.abs(b.numpy() - rb) <= (64 + m) * eps * np.maximum(rb, 1.0 / n))
        ed.assemble_defect(d, U.Vector(values=u))
        assert np.all(np.abs(d.numpy() - rd) <= (64 + m) * eps * np.maximum(sd, 1e-30))
    assert m[n - 1] == 0 and b.numpy()[n - 1] == 0.0 and d.numpy()[n - 1] == 0.0


def test_local_matrices_are_not_kept():
    """between assemblies the discretisation holds its mesh, its pattern and its
    lists, not the 512 bytes per Q1 hexahedron of the local matrices"""
    print("case element workspace", flush=True)
    sys.stdout.flush()
    import torch
    import ugcore_amd as U
    n = 64
    W, ne = n + 1, n ** 3
    z, y, x = np.meshgrid(*[np.arange(n)] * 3, indexing="ij")
    at = lambda dx, dy, dz: (((z + dz) * W + y + dy) * W + x + dx).reshape(-1)
    E = np.stack([at(*c) for c in ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1),
                                   (0, 1, 1))], 1)
    X = np.stack(np.meshgrid(*[np.arange(W) / n] * 3, indexing="ij")[::-1], -1).reshape(-1, 3)
    keep = U.Vector(8)
    ed = U.ElementDiscretization("hexahedron_q1", E, X)
    A, b, d = U.SparseMatrix(), U.Vector(W ** 3), U.Vector(W ** 3)
    for _ in range(2):
        ed.assemble_linear(A, b)
        ed.assemble_defect(d, b)
    U.synchronize()
    U.trim_memory()
    with_ed = torch.cuda.mem_get_info()[0]
    nnz = ed.nnz()
    del ed
    U.trim_memory()
    held = torch.cuda.mem_get_info()[0] - with_ed
    # element table, list of local entries, vertex lists; pattern and entry
    # pointers; coordinates and pointers; blocks are up to 1/8 larger than asked
    lists = ne * (4 * 8 + 4 * 64 + 4 * 8) + 8 * nnz + 32 * W ** 3
    assert held <= 1.125 * lists + (32 << 20) < lists + 512 * ne, (held, lists)
    assert keep.size() == 8


@pytest.mark.parametrize("m", [40, 64, 65, 300])
def test_any_number_of_elements_may_share_a_dof(m):
    """a fan of m triangles around one DoF: the assembly needs no colours (more
    than 63 of them are an error of num_colours alone)"""
    print(f"case fan of {m} triangles", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    t = 2 * np.pi * np.arange(m) / m
    X = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], 1)])
    E = np.stack([np.zeros(m, int), 1 + np.arange(m), 1 + (np.arange(m) + 1) % m], 1)
    ed = U.ElementDiscretization("triangle_fv1", E, X)
    ed.set_source(2.0)
    A, b = U.SparseMatrix(), U.Vector(m + 1)
    ed.assemble_linear(A, b)
    if m <= 64:
        assert ed.num_colours() == m                    # every two share the centre
    else:
        with pytest.raises(U.UGError, match="63 neighbouring colours"):
            ed.num_colours()
    Ke, fe, _, vol = p1(X[E], np.ones(m))
    R, S, rb = np.zeros((m + 1, m + 1)), np.zeros((m + 1, m + 1)), np.zeros(m + 1)
    for a in range(3):
        np.add.at(rb, E[:, a], 2.0 * fe[:, a])
        for c in range(3):
            np.add.at(R, (E[:, a], E[:, c]), Ke[:, a, c])
            np.add.at(S, (E[:, a], E[:, c]), np.abs(Ke).max(axis=(1, 2)))
    rp, col, val = A.download_csr()
    row = np.repeat(np.arange(m + 1), np.diff(rp))
    # 64 operations at the condition of a fan triangle's Jacobian (about m), then a sum of up to m terms
    assert np.all(np.abs(val - R[row, col]) <= (64 * m + m) * 2.0 ** -52 * S[row, col])
    assert np.all(np.abs(b.numpy() - rb) <= (64 * m + m) * 2.0 ** -52 * rb.max())
