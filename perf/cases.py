"""Performance cases: what programs that use this package ask of it, through
its public entry points, with the outputs they read back from the device.

Families (the "path" of a case):

  solve_hex   CG + geometric multigrid on the Q1 hexahedral hierarchy
              (FP32 or FP64 levels): the package's headline solve
  solve_tri   CG + geometric multigrid on the 2D FV1 hierarchy
  solve_tet   BiCGStab + geometric multigrid, FV1 convection-diffusion
  solve_q2    CG + multigrid over the Q2 level matrices
  adjoint     one step of an inverse problem through torch.autograd
  refresh     a new coefficient field: re-assembly, multigrid set-up and one
              application of the cycle to a right-hand side
  product     A x with an assembled lattice operator
  csr         A x and A^T x with an uploaded matrix of ragged rows
  q2_element  batched Q2 element matrices
  elements    assembly and defect from caller-supplied connectivity
"""
import math

import numpy as np
import torch

import ugcore_amd as U

FAMILIES = ("solve_hex", "solve_tri", "solve_tet", "solve_q2", "adjoint", "refresh", "product", "csr", "q2_element",
            "elements")


# ---- the cases -----------------------------------------------------------------------------------

def listed():
    return [
        # the headline problem of the benchmark: 16,974,593 unknowns, FP32 levels in an FP64 CG
        dict(name="hex 256 f32", path="solve_hex", refs=8, prec="f32", ordering="reference", nu=2, omega=0.66),
        # a medium 3D problem with the all-FP64 multigrid
        dict(name="hex 128 f64", path="solve_hex", refs=7, prec="f64", ordering="lex", nu=2, omega=0.66),
        # a small 3D problem solved over and over (time stepping, sampling): latency counts
        dict(name="hex 32 f32", path="solve_hex", refs=5, prec="f32", ordering="lex", nu=2, omega=0.66),
        # the 2D FV1 Poisson configuration of the benchmark, FP64
        dict(name="tri 128 f64", path="solve_tri", refs=7, prec="f64", ordering="lex", nu=2, omega=0.66),
        # the tetrahedral convection-diffusion configuration of the benchmark: 96^3 x 6 tetrahedra
        dict(name="tet 96 f32", path="solve_tet", refs=5, prec="f32", nu=2, omega=0.6),
        # a quadratic discretisation: 33^3 unknowns, multigrid over matrices
        dict(name="q2 16", path="solve_q2", refs=4, nu=2, omega=0.66),
        # one gradient step on 64^3 parameters with 4096 observations, tensors on the device
        dict(name="adjoint 64 f32", path="adjoint", refs=6, prec="f32", observations=4096),
        # a parameter update at 128^3: everything that has to be renewed before the next solve
        dict(name="refresh 128 f32", path="refresh", refs=7, prec="f32", ordering="lex", nu=2, omega=0.66),
        # the assembled operator of the headline problem applied to a vector
        dict(name="product hex 256", path="product", kind=0, refs=8, ordering="reference"),
        # a matrix that comes from elsewhere, rows of 1 to 40 entries
        dict(name="csr 400003", path="csr", rows=400003, mean=15, band=6000),
        # Q2 element matrices of a 64^3 mesh for a caller's own assembly
        dict(name="q2 elements 64^3", path="q2_element", elements=262144),
        # an unstructured-mesh code handing over its tetrahedra: 264 thousand of them
        dict(name="tets 41x37x29", path="elements", kind="tetrahedron_fv1", nx=41, ny=37, nz=29),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(FAMILIES)
    omega = round(rng.uniform(0.6, 0.8), 4)
    if path == "solve_hex":
        refs = rng.randint(3, 8)
        prec = "f32" if refs == 8 else rng.choice(("f32", "f64"))
        return dict(path=path, refs=refs, prec=prec, ordering="lex" if refs < 8 and rng.random() < 0.5 else "reference",
                    nu=2 if refs == 8 else rng.choice((1, 2, 2, 3)), omega=round(rng.uniform(0.62, 0.7), 4))
    if path == "solve_tri":
        return dict(path=path, refs=rng.randint(3, 10), prec=rng.choice(("f32", "f64")),
                    ordering=rng.choice(("lex", "reference")), nu=rng.choice((1, 2, 2, 3)), omega=omega)
    if path == "solve_tet":
        return dict(path=path, refs=rng.randint(2, 5), prec=rng.choice(("f32", "f64")), nu=rng.choice((2, 2, 3)),
                    omega=round(rng.uniform(0.55, 0.65), 4))
    if path == "solve_q2":
        return dict(path=path, refs=rng.randint(2, 4), nu=rng.choice((1, 2, 2, 3)), omega=round(rng.uniform(0.6, 0.7), 4))
    if path == "adjoint":
        refs = rng.randint(3, 7)
        return dict(path=path, refs=refs, prec=rng.choice(("f32", "f64")),
                    observations=_log_int(rng, 16, min(8192, (2 ** refs - 1) ** 3)))
    if path == "refresh":
        return dict(path=path, refs=rng.randint(3, 7), prec=rng.choice(("f32", "f64")),
                    ordering=rng.choice(("lex", "reference")), nu=rng.choice((1, 2, 2, 3)), omega=omega)
    if path == "product":
        kind = rng.choice((0, 1, 2))
        refs = {0: (3, 7), 1: (5, 11), 2: (1, 5)}[kind]
        return dict(path=path, kind=kind, refs=rng.randint(*refs), ordering=rng.choice(("lex", "reference")),
                    beta=round(rng.uniform(0.5, 2.0), 4))
    if path == "csr":
        rows = _log_int(rng, 1000, 800000) | 1
        return dict(path=path, rows=rows, mean=rng.randint(5, 30), band=_log_int(rng, 100, max(101, rows // 4)))
    if path == "q2_element":
        return dict(path=path, elements=_log_int(rng, 27, 262144))
    kind = rng.choice(("triangle_fv1", "tetrahedron_fv1", "hexahedron_q1"))
    if kind == "triangle_fv1":
        return dict(path=path, kind=kind, nx=_log_int(rng, 16, 400), ny=_log_int(rng, 16, 400), nz=0)
    return dict(path=path, kind=kind, nx=_log_int(rng, 5, 41), ny=_log_int(rng, 5, 41), nz=_log_int(rng, 5, 29))


# ---- inputs --------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _smooth_theta(n, dim, seed):
    """log-diffusion per fine element: i.i.d. N(0,1), three box averages over
    the 3^dim neighbours clipped at the boundary (ugcore_amd.synthetic)"""
    def box(a, ax):
        s = a.clone()
        m = a.shape[ax]
        s.narrow(ax, 1, m - 1).add_(a.narrow(ax, 0, m - 1))
        s.narrow(ax, 0, m - 1).add_(a.narrow(ax, 1, m - 1))
        return s
    t = torch.randn((n,) * dim, generator=_gen(seed), device="cuda", dtype=torch.float64)
    cnt = torch.ones_like(t)
    for ax in range(dim):
        cnt = box(cnt, ax)
    for _ in range(3):
        for ax in range(dim):
            t = box(t, ax)
        t = t / cnt
    return t.reshape(-1).contiguous()


class _Memory:
    """a device buffer of the library, as torch reads it"""

    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _view(ptr, n, owner, typestr="<f8"):
    return torch.as_tensor(_Memory(ptr, n, typestr, owner), device="cuda")


def _vec(n, values=None):
    v = U.Vector(int(n))
    t = _view(v.device_ptr(), n, v)
    if values is None:
        v.set(0.0)
    else:
        torch.cuda.synchronize()
        U.lib().ugx_memcpy_dtod(v.device_ptr(), values.data_ptr(), 8 * int(n))
    return v, t


def _values(A):
    """the values of a device matrix"""
    rp, col, val = (U.C.c_void_p() for _ in range(3))
    if U.lib().ugx_matrix_device_csr_readonly(A.h, U.C.byref(rp), U.C.byref(col), U.C.byref(val)) < 0:
        raise U.UGError("device_csr_readonly")
    return _view(val.value, A.nnz(), A)


def _source_tri(n, seed):
    W = n + 1
    y, x = np.mgrid[0:W, 0:W] / n
    f = 2.0 * np.pi ** 2 * np.sin(np.pi * x) * np.sin(np.pi * y)
    return (f + 0.1 * np.random.default_rng(seed).normal(size=(W, W))).reshape(-1)


def _theta_kind(kind, refs, seed):
    n = (3 if kind == 2 else 1) << refs
    t = _smooth_theta(n, 2 if kind == 1 else 3, seed)
    return 0.5 * t if kind == 1 else t


def _lattice_system(kind, refs, seed, ordering="reference"):
    """the discretisation with its coefficient field, its operator and rhs"""
    d = U.DomainDiscretization(kind, refs, ordering=ordering)
    theta = _theta_kind(kind, refs, seed)
    torch.cuda.synchronize()
    d.set_theta_device(theta.data_ptr())
    U.synchronize()
    if kind == 1:
        f = np.empty(d.num_dofs())
        f[d.dof_of_lattice(refs)] = _source_tri(d.n_fine, seed)
        d.set_source(f)
    else:
        d.set_source(1.0)
    if kind == 2:
        d.set_velocity((20.0, 10.0, 5.0))
        d.set_jitter(11, 0.2 / math.sqrt(3.0))
    A = U.SparseMatrix()
    b, bt = _vec(d.num_dofs())
    d.assemble_linear(A, b)
    return d, theta, A, b, bt


def _mesh(case, seed):
    """a box mesh with displaced inner points: (elements, coordinates, boundary)"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rng = np.random.default_rng(seed)
    if case["kind"] == "triangle_fv1":
        j, i = np.mgrid[0:ny + 1, 0:nx + 1]
        X = np.stack([i.ravel() / nx, j.ravel() / ny], axis=1)
        bnd = ((i == 0) | (i == nx) | (j == 0) | (j == ny)).ravel()
        X += np.where(bnd[:, None], 0.0, rng.uniform(-0.15, 0.15, X.shape) / np.array([nx, ny]))
        j, i = np.mgrid[0:ny, 0:nx]
        a = (j * (nx + 1) + i).ravel()
        b, c, d = a + 1, a + nx + 2, a + nx + 1
        E = np.stack([np.stack([a, b, c], 1), np.stack([a, c, d], 1)], 1).reshape(-1, 3)
        return E.astype(np.int32), X, np.flatnonzero(bnd)
    k, j, i = np.mgrid[0:nz + 1, 0:ny + 1, 0:nx + 1]
    X = np.stack([i.ravel() / nx, j.ravel() / ny, k.ravel() / nz], axis=1)
    bnd = ((i == 0) | (i == nx) | (j == 0) | (j == ny) | (k == 0) | (k == nz)).ravel()
    X += np.where(bnd[:, None], 0.0, rng.uniform(-0.1, 0.1, X.shape) / np.array([nx, ny, nz]))
    k, j, i = np.mgrid[0:nz, 0:ny, 0:nx]
    a = ((k * (ny + 1) + j) * (nx + 1) + i).ravel()
    sx, sy, sz = 1, nx + 1, (nx + 1) * (ny + 1)
    if case["kind"] == "hexahedron_q1":
        o = np.array([0, sx, sx + sy, sy, sz, sx + sz, sx + sy + sz, sy + sz])
        return (a[:, None] + o[None]).astype(np.int32), X, np.flatnonzero(bnd)
    # six tetrahedra around the main diagonal of every cell, positively oriented
    E = []
    for p, q, even in ((sx, sy, 1), (sy, sz, 1), (sz, sx, 1), (sy, sx, 0), (sz, sy, 0), (sx, sz, 0)):
        t = [a, a + p, a + p + q, a + sx + sy + sz]
        E.append(np.stack(t if even else [t[0], t[2], t[1], t[3]], 1))
    return np.stack(E, 1).reshape(-1, 4).astype(np.int32), X, np.flatnonzero(bnd)


def _csr_host(case, seed):
    """ragged rows (1 to 40 entries around `mean`), columns within a band and
    a few far ones, sorted; values of a diagonally dominant matrix"""
    n, mean, band = case["rows"], case["mean"], case["band"]
    g = _gen(seed)
    ln = (mean * torch.exp(0.4 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64))).long().clamp_(1, 40)
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), ln)
    m = row.numel()
    off = (band * torch.randn(m, generator=g, device="cuda", dtype=torch.float64) / 3).long()
    far = torch.rand(m, generator=g, device="cuda") < 0.02
    col = torch.where(far, torch.randint(0, n, (m,), generator=g, device="cuda"), (row + off).remainder(n))
    first = torch.cumsum(ln, 0) - ln
    col[first] = torch.arange(n, device="cuda")
    key = torch.unique(row * n + col)
    row, col = key // n, key % n
    val = torch.randn(key.numel(), generator=g, device="cuda", dtype=torch.float64)
    val = torch.where(row == col, val.abs() + float(mean), 0.5 * val)
    rp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    x = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    v = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
    return rp, col, val, x, v


_HEX = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))


def _q2_inputs(case, seed):
    n = case["elements"]
    g = _gen(seed)
    m = max(1, math.ceil(n ** (1 / 3)))
    e = torch.arange(n, device="cuda")
    base = torch.stack([e % m, (e // m) % m, e // (m * m)], 1).double()
    X = base[:, None, :] + torch.tensor(_HEX, device="cuda", dtype=torch.float64)[None]
    X = (X + 0.2 * torch.rand(X.shape, generator=g, device="cuda", dtype=torch.float64) - 0.1) / m
    k = torch.exp(0.5 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64))
    return X.contiguous(), k


def _observations(case, seed):
    n = 2 ** case["refs"]
    g = _gen(seed + 1000003)
    p = torch.randperm((n - 1) ** 3, generator=g, device="cuda")[:case["observations"]]
    i, j, k = p % (n - 1) + 1, (p // (n - 1)) % (n - 1) + 1, p // (n - 1) ** 2 + 1
    return (k * (n + 1) + j) * (n + 1) + i, 1e-2 * torch.randn(p.numel(), generator=g, device="cuda",
                                                               dtype=torch.float64)


def _base(refs):
    return min(2, refs - 1)


def prepare(case, seed):
    U.init()
    path = case["path"]
    s = dict(path=path)
    if path in ("solve_hex", "solve_tri", "solve_tet"):
        kind = {"solve_hex": 0, "solve_tri": 1, "solve_tet": 2}[path]
        d, theta, A, b, bt = _lattice_system(kind, case["refs"], seed, case.get("ordering", "reference"))
        g = U.GeometricMultiGrid(d, base_level=_base(case["refs"]) if kind == 0 else 0, nu1=case["nu"], nu2=case["nu"],
                                 omega=case["omega"], precision=case["prec"])
        S = (U.BiCGStab if kind == 2 else U.CG)(g, max_steps=500, reduction=1e-10)
        S.init(A)
        x, xt = _vec(d.num_dofs())
        s.update(keep=(d, g, A), S=S, x=x, xt=xt, b=b)
    elif path == "solve_q2":
        q = U.Q2Discretization(case["refs"])
        q.set_theta(_smooth_theta(2 ** case["refs"], 3, seed).cpu().numpy())
        q.set_source(1.0)
        A, P, R, b = q.hierarchy()
        S = U.CG(U.MatrixMultiGrid(A, P, R, nu1=case["nu"], nu2=case["nu"], omega=case["omega"]), max_steps=500,
                 reduction=1e-10)
        S.init(A[-1])
        x, xt = _vec(b.size())
        s.update(keep=(q, A, P, R), S=S, x=x, xt=xt, b=b)
    elif path == "adjoint":
        from ugcore_amd import adjoint
        refs = case["refs"]
        prob = adjoint.DiffusionProblem(refs, base_level=_base(refs), precision=case["prec"], reduction=1e-10)
        theta = _smooth_theta(2 ** refs, 3, seed)
        pts, data = _observations(case, seed)
        dofs = torch.from_numpy(np.asarray(prob.dof_of_lattice()).astype(np.int64)).cuda()[pts]
        s.update(prob=prob, theta=theta, dofs=dofs, data=data, solve=adjoint.solve)
    elif path == "refresh":
        d, _, A, b, bt = _lattice_system(0, case["refs"], seed + 500009, case["ordering"])
        g = U.GeometricMultiGrid(d, base_level=_base(case["refs"]), nu1=case["nu"], nu2=case["nu"], omega=case["omega"],
                                 precision=case["prec"])
        c, ct = _vec(d.num_dofs())
        s.update(d=d, theta=_theta_kind(0, case["refs"], seed), A=A, b=b, g=g, c=c, out=(_values(A), bt, ct))
    elif path == "product":
        d, _, A, _, _ = _lattice_system(case["kind"], case["refs"], seed, case["ordering"])
        n = d.num_dofs()
        x, _ = _vec(n, torch.randn(n, generator=_gen(seed + 7), device="cuda", dtype=torch.float64))
        y, yt = _vec(n)
        s.update(A=A, x=x, y=y, yt=yt, beta=case.get("beta", 1.0))
    elif path == "csr":
        rp, col, val, x, v = _csr_host(case, seed)
        A = U.SparseMatrix()
        A.upload_csr(rp.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy())
        n = case["rows"]
        (y, yt), (z, zt) = _vec(n), _vec(n)
        s.update(A=A, x=_vec(n, x)[0], v=_vec(n, v)[0], y=y, z=z, out=(yt, zt))
        A.apply_transposed(z, s["x"])   # the transpose is kept with the matrix
    elif path == "q2_element":
        X, k = _q2_inputs(case, seed)
        n = case["elements"]
        ke = torch.empty((n, 27, 27), device="cuda", dtype=torch.float64)
        fe = torch.empty((n, 27), device="cuda", dtype=torch.float64)
        s.update(n=n, X=X, k=k, ke=ke, fe=fe)
    else:
        E, X, bnd = _mesh(case, seed)
        rng = np.random.default_rng(seed + 1)
        ed = U.ElementDiscretization(case["kind"], E, X)
        ed.set_diffusion(np.exp(0.5 * rng.normal(size=E.shape[0])))
        ed.set_source(1.0)
        ed.set_dirichlet(bnd)
        n = X.shape[0]
        A = U.SparseMatrix()
        (b, bt), (d, dt) = _vec(n), _vec(n)
        u = U.Vector(values=rng.normal(size=n))
        ed.assemble_linear(A, b)
        s.update(ed=ed, A=A, b=b, d=d, u=u, out=(_values(A), bt, dt))
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------------------------

def run(s):
    path = s["path"]
    if path in ("solve_hex", "solve_tri", "solve_tet", "solve_q2"):
        s["x"].set(0.0)
        if not s["S"].apply(s["x"], s["b"]):
            raise RuntimeError("the solve did not converge")
        return s["xt"]
    if path == "adjoint":
        theta = s["theta"].detach().requires_grad_(True)
        u = s["solve"](theta, s["prob"])
        loss = 0.5 * (u[s["dofs"]] - s["data"]).square().sum()
        loss.backward()
        return {"u": u.detach(), "loss": loss.detach(), "grad": theta.grad}
    if path == "refresh":
        s["d"].set_theta_device(s["theta"].data_ptr())
        s["d"].assemble_linear(s["A"], s["b"])
        s["g"].init(s["A"])
        s["g"].apply(s["c"], s["b"])
        return s["out"]
    if path == "product":
        s["A"].axpy(s["y"], 0.0, s["y"], s["beta"], s["x"])
        return s["yt"]
    if path == "csr":
        s["A"].axpy(s["y"], 1.0, s["v"], -1.0, s["x"])
        s["A"].apply_transposed(s["z"], s["x"])
        return s["out"]
    if path == "q2_element":
        if U.lib().ugx_q2_hex_element_matrices(s["n"], s["X"].data_ptr(), s["k"].data_ptr(), 1.0, s["ke"].data_ptr(),
                                               s["fe"].data_ptr()) < 0:
            raise U.UGError("q2_hex_element_matrices")
        return s["ke"], s["fe"]
    s["ed"].assemble_linear(s["A"], s["b"])
    s["ed"].assemble_defect(s["d"], s["u"])
    return s["out"]


# ---- what a pass cannot do without ---------------------------------------------------------------

def _sizes(kind, refs):
    """(unknowns, entries of the operator, coefficients) of a lattice domain"""
    n = (3 if kind == 2 else 1) << refs
    dim = 2 if kind == 1 else 3
    N = (n + 1) ** dim
    nnz = (3 * n + 1) ** dim if kind == 0 else N + 6 * n * n + 4 * n if kind == 1 else int(14.75 * N)
    return N, nnz, n ** dim


def work(case):
    path = case["path"]
    if path in ("solve_hex", "solve_tri", "solve_tet"):
        kind = {"solve_hex": 0, "solve_tri": 1, "solve_tet": 2}[path]
        N, nnz, ne = _sizes(kind, case["refs"])
        steps = {0: 8, 1: 12, 2: 32}[kind]
        cycles = 2 if kind == 2 else 1
        # theta and b in, x out; per step the cycle's operator passes on all levels and the Krylov step
        return {"bytes": 8 * (ne + 2 * N), "flops": steps * cycles * (2.0 * nnz * (2 * case["nu"] + 2) * 8 / 7 + 20 * N)}
    if path == "solve_q2":
        n = 2 ** case["refs"]
        N, nnz = (2 * n + 1) ** 3, (8 * n + 1) ** 3
        return {"bytes": 12 * nnz + 16 * N, "flops": 15 * 2.0 * nnz * (2 * case["nu"] + 2) * 8 / 7}
    if path == "adjoint":
        N, nnz, ne = _sizes(0, case["refs"])
        # theta in, the operator, u and the gradient out; the two solves
        return {"bytes": 12 * nnz + 8 * (2 * ne + 2 * N), "flops": 2 * 8 * (2.0 * nnz * 6 * 8 / 7 + 20 * N)}
    if path == "refresh":
        N, nnz, ne = _sizes(0, case["refs"])
        # theta in, values, b and the correction out; the cycle's own operator is formed on the way
        return {"bytes": 8 * (ne + nnz + 3 * N), "flops": 128.0 * N * 8 / 7 + 2.0 * nnz * (2 * case["nu"] + 1) * 8 / 7}
    if path == "product":
        N, nnz, _ = _sizes(case["kind"], case["refs"])
        return {"bytes": 12 * nnz + 20 * N, "flops": 2.0 * nnz}
    if path == "csr":
        nnz = 1.05 * case["rows"] * case["mean"]
        return {"bytes": 2 * 12 * nnz + 2 * 4 * case["rows"] + 8 * 5 * case["rows"], "flops": 4.0 * nnz}
    if path == "q2_element":
        return {"bytes": 8 * (24 + 1 + 729 + 27) * case["elements"], "flops": 2.0 * 27 * 27 * 81 * case["elements"]}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["kind"] == "triangle_fv1":
        ne, nv, N, nnz, dim, f = 2 * nx * ny, 3, (nx + 1) * (ny + 1), 7 * nx * ny, 2, 100
    elif case["kind"] == "tetrahedron_fv1":
        ne, nv, N, nnz, dim, f = 6 * nx * ny * nz, 4, (nx + 1) * (ny + 1) * (nz + 1), 15 * nx * ny * nz, 3, 400
    else:
        ne, nv, N, nnz, dim, f = nx * ny * nz, 8, (nx + 1) * (ny + 1) * (nz + 1), 27 * nx * ny * nz, 3, 4000
    # connectivity, coordinates and coefficients in (for the matrix and again for the defect), values, b, d out
    return {"bytes": 2 * (4 * ne * nv + 8 * N * dim + 8 * ne) + 8 * (nnz + 3 * N), "flops": 2.0 * f * ne}


def tolerance(case):
    path = case["path"]
    if path in ("solve_hex", "solve_tri", "solve_tet", "solve_q2"):
        # a residual reduction of 1e-10 leaves up to 2e-10 in the solution; a step more or less is as good an answer
        return {"rel": 4e-10}
    if path == "adjoint":
        return {"rel": 1e-9}       # two such solves, and the gradient's differences of neighbours
    if path == "refresh":
        # one cycle in the levels' precision (FP32 against FP64 levels: 1e-7)
        return {"rel": 4e-7} if case["prec"] == "f32" else {"rel": 1e-12}
    if path in ("product", "csr"):
        return {"rel": 1e-14}      # FP64 sums of up to 40 terms in another order
    return {"rel": 3e-14}          # FP64 element integrals and sums over the elements of a row


# ---- the same in 64 bits by plain torch ----------------------------------------------------------

def _lex_dofs(n, dim):
    """lattice point -> DoF of the lexicographic numbering: inner points first"""
    ax = torch.arange(n + 1, device="cuda")
    e = (ax == 0) | (ax == n)
    bnd = (e[:, None] | e[None, :]) if dim == 2 else (e[:, None, None] | e[None, :, None] | e[None, None, :])
    bnd = bnd.reshape(-1)
    d = torch.empty(bnd.numel(), dtype=torch.int64, device="cuda")
    inner = torch.nonzero(~bnd).reshape(-1)
    outer = torch.nonzero(bnd).reshape(-1)
    d[inner] = torch.arange(inner.numel(), device="cuda")
    d[outer] = inner.numel() + torch.arange(outer.numel(), device="cuda")
    return d, bnd


def _hex_stiffness():
    """the unit cube's Q1 stiffness and load, corners x fastest"""
    m = torch.tensor([[2.0, 1.0], [1.0, 2.0]], dtype=torch.float64) / 6
    s = torch.tensor([[1.0, -1.0], [-1.0, 1.0]], dtype=torch.float64)
    kr = torch.kron
    return (kr(m, kr(m, s)) + kr(m, kr(s, m)) + kr(s, kr(m, m))).cuda()


def _corner_slices(n, dim):
    r = (slice(0, n), slice(1, n + 1))
    if dim == 3:
        return [(r[c >> 2], r[(c >> 1) & 1], r[c & 1]) for c in range(8)]
    return [(r[c >> 1], r[c & 1]) for c in range(4)]


def _lattice_apply(k, K, dim):
    """u -> A u by elements on the lattice, zero on the boundary; its diagonal"""
    n = k.shape[0]
    sl = _corner_slices(n, dim)
    inner = (slice(1, n),) * dim

    def apply(u):
        G = torch.stack([u[s] for s in sl], -1)
        Y = (G @ K) * k[..., None]
        y = torch.zeros_like(u)
        for c, s in enumerate(sl):
            y[s] += Y[..., c]
        out = torch.zeros_like(u)
        out[inner] = y[inner]
        return out
    diag = torch.zeros((n + 1,) * dim, device="cuda", dtype=torch.float64)
    for c, s in enumerate(sl):
        diag[s] += k * K[c, c]
    return apply, diag


def _pcg(apply, diag, b, tol=1e-13, most=20000):
    x = torch.zeros_like(b)
    r = b.clone()
    z = r / diag
    p = z.clone()
    rz = (r * z).sum()
    stop = (tol * b.norm()) ** 2
    for i in range(most):
        q = apply(p)
        a = rz / (p * q).sum()
        x += a * p
        r -= a * q
        if i % 25 == 24 and bool((r * r).sum() <= stop):
            break
        z = r / diag
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def _hex_problem(theta, n):
    h = 1.0 / n
    k = torch.exp(theta).reshape(n, n, n)
    apply, diag = _lattice_apply(k, h * _hex_stiffness(), 3)
    b = torch.zeros((n + 1,) * 3, device="cuda", dtype=torch.float64)
    b[1:n, 1:n, 1:n] = h ** 3
    return k, apply, diag, b


def _tri_problem(theta, n, f):
    """two right triangles per square with one coefficient: half of k on each
    of the square's four sides, a third of the triangle's area per corner"""
    k = torch.exp(theta).reshape(n, n)
    K = torch.tensor([[1.0, -0.5, -0.5, 0.0], [-0.5, 1.0, 0.0, -0.5], [-0.5, 0.0, 1.0, -0.5], [0.0, -0.5, -0.5, 1.0]],
                     dtype=torch.float64, device="cuda")
    apply, diag = _lattice_apply(k, K, 2)
    b = torch.zeros_like(diag)
    for c, s in enumerate(_corner_slices(n, 2)):
        b[s] += (2 if c in (0, 3) else 1) * (0.5 / n ** 2) / 3.0
    b *= torch.from_numpy(f).cuda().reshape(n + 1, n + 1)
    z = torch.zeros_like(b)
    z[1:n, 1:n] = b[1:n, 1:n]
    return apply, diag, z


def _assembled(E, Ke, N, bnd):
    """values in row order, columns ascending, of the sum of element matrices
    with identity rows on the boundary; and the sorted (row, column) keys"""
    nv = E.shape[1]
    key = (E[:, :, None] * N + E[:, None, :]).reshape(-1)
    u, inv = torch.unique(key, return_inverse=True)
    val = torch.zeros(u.numel(), device="cuda", dtype=torch.float64)
    val.index_add_(0, inv, Ke.reshape(-1))
    row, col = u // N, u % N
    flag = torch.zeros(N, dtype=torch.bool, device="cuda")
    flag[bnd] = True
    return torch.where(flag[row], (row == col).double(), val)


def _hex_gauss(X, k, f, shapes, points, weights):
    """element matrices and load vectors of hexahedra with trilinear geometry:
    shapes(x) gives values [m] and gradients [m, 3] on the unit cube"""
    Ke = fe = None
    lin = _shapes(1, _HEX)
    for p, w in zip(points, weights):
        _, G = lin(p)
        J = torch.einsum("ncr,cs->nrs", X, torch.from_numpy(G).cuda())
        phi, D = shapes(p)
        g = torch.from_numpy(D).cuda() @ torch.linalg.inv(J)
        wd = w * torch.linalg.det(J).abs()
        add = (g * (wd * k)[:, None, None]) @ g.transpose(1, 2).contiguous()
        load = (f * wd)[:, None] * torch.from_numpy(phi).cuda()[None]
        Ke, fe = (add, load) if Ke is None else (Ke.add_(add), fe.add_(load))
    return Ke, fe


def _shapes(order, nodes):
    """Lagrange shapes of the unit cube for nodes given in units of 1/order"""
    def one(i, t):
        if order == 1:
            return (1 - t, -1.0) if i == 0 else (t, 1.0)
        return ((2 * t - 1) * (t - 1), 4 * t - 3) if i == 0 else (4 * t * (1 - t), 4 - 8 * t) if i == 1 else \
            (t * (2 * t - 1), 4 * t - 1)

    def at(p):
        phi, D = np.empty(len(nodes)), np.empty((len(nodes), 3))
        for m, nd in enumerate(nodes):
            v = [one(nd[d], p[d]) for d in range(3)]
            phi[m] = v[0][0] * v[1][0] * v[2][0]
            D[m] = (v[0][1] * v[1][0] * v[2][0], v[0][0] * v[1][1] * v[2][0], v[0][0] * v[1][0] * v[2][1])
        return phi, D
    return at


def _gauss(m):
    x, w = np.polynomial.legendre.leggauss(m)
    x, w = (x + 1) / 2, w / 2
    P = [(x[i], x[j], x[k]) for k in range(m) for j in range(m) for i in range(m)]
    return P, [w[i] * w[j] * w[k] for k in range(m) for j in range(m) for i in range(m)]


# the quadratic hexahedron's nodes: corners, edges, faces, the centre
_EDGES = ((0, 1), (1, 2), (2, 3), (3, 0), (0, 4), (1, 5), (2, 6), (3, 7), (4, 5), (5, 6), (6, 7), (7, 4))
_FACES = ((0, 3, 2, 1), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (3, 0, 4, 7), (4, 5, 6, 7))
_Q2 = (tuple(tuple(2 * x for x in c) for c in _HEX) +
       tuple(tuple(_HEX[a][d] + _HEX[b][d] for d in range(3)) for a, b in _EDGES) +
       tuple(tuple(sum(_HEX[a][d] for a in q) // 2 for d in range(3)) for q in _FACES) + ((1, 1, 1),))


def exact(case, seed):
    path = case["path"]
    if path == "solve_hex" and case["ordering"] == "lex":
        n = 2 ** case["refs"]
        _, apply, diag, b = _hex_problem(_theta_kind(0, case["refs"], seed), n)
        x = torch.empty((n + 1) ** 3, device="cuda", dtype=torch.float64)
        x[_lex_dofs(n, 3)[0]] = _pcg(apply, diag, b).reshape(-1)
        return x
    if path == "solve_tri" and case["ordering"] == "lex" and case["refs"] <= 9:
        n = 2 ** case["refs"]
        apply, diag, b = _tri_problem(_theta_kind(1, case["refs"], seed), n, _source_tri(n, seed))
        x = torch.empty((n + 1) ** 2, device="cuda", dtype=torch.float64)
        x[_lex_dofs(n, 2)[0]] = _pcg(apply, diag, b).reshape(-1)
        return x
    if path == "adjoint":
        n = 2 ** case["refs"]
        k, apply, diag, b = _hex_problem(_smooth_theta(n, 3, seed), n)
        u = _pcg(apply, diag, b)
        pts, data = _observations(case, seed)
        res = u.reshape(-1)[pts] - data
        r = torch.zeros_like(b)
        r.view(-1)[pts] = res
        lam = _pcg(apply, diag, r)
        sl = _corner_slices(n, 3)
        ue, le = (torch.stack([v[s] for s in sl], -1) for v in (u, lam))
        grad = -((ue @ (_hex_stiffness() / n)) * le).sum(-1) * k
        # u is numbered by the framework's own refinement
        return {"u": None, "loss": 0.5 * res.square().sum(), "grad": grad.reshape(-1)}
    if path == "refresh" and case["ordering"] == "lex":
        n = 2 ** case["refs"]
        dof, bnd = _lex_dofs(n, 3)
        ax = torch.arange(n, device="cuda")
        cell = ((ax[:, None, None] * (n + 1) + ax[None, :, None]) * (n + 1) + ax[None, None, :]).reshape(-1)
        o = torch.tensor([x + (n + 1) * (y + (n + 1) * z) for z in (0, 1) for y in (0, 1) for x in (0, 1)], device="cuda")
        k, _, _, b = _hex_problem(_theta_kind(0, case["refs"], seed), n)
        K = _hex_stiffness() / n
        N = (n + 1) ** 3
        if case["refs"] <= 6:
            val = _assembled(dof[cell[:, None] + o[None]], k.reshape(-1)[:, None, None] * K, N, dof[bnd])
        else:
            val = None
        bt = torch.empty(N, device="cuda", dtype=torch.float64)
        bt[dof] = b.reshape(-1)
        return val, bt, None
    if path == "csr":
        rp, col, val, x, v = _csr_host(case, seed)
        row = torch.repeat_interleave(torch.arange(case["rows"], device="cuda"), rp[1:] - rp[:-1])
        y = v.clone().index_add_(0, row, -val * x[col])
        z = torch.zeros_like(x).index_add_(0, col, val * x[row])
        return y, z
    if path == "q2_element":
        X, k = _q2_inputs(case, seed)
        P, w = _gauss(3)
        Ke, fe = _hex_gauss(X, k, 1.0, _shapes(2, _Q2), P, w)
        return Ke, fe
    if path == "elements":
        E, X, bnd = _mesh(case, seed)
        rng = np.random.default_rng(seed + 1)
        k = torch.from_numpy(np.exp(0.5 * rng.normal(size=E.shape[0]))).cuda()
        n = X.shape[0]
        u = torch.from_numpy(rng.normal(size=n)).cuda()
        E, Xe = torch.from_numpy(E.astype(np.int64)).cuda(), torch.from_numpy(X[E]).cuda()
        bnd = torch.from_numpy(bnd).cuda()
        if case["kind"] == "hexahedron_q1":
            P, w = _gauss(2)
            Ke, fe = _hex_gauss(Xe, k, 1.0, _shapes(1, _HEX), P, w)
        else:
            # box method on linear simplices: the P1 stiffness, an equal share of the volume per corner
            dim = Xe.shape[2]
            J = (Xe[:, 1:] - Xe[:, :1]).transpose(1, 2).contiguous()
            vol = torch.linalg.det(J).abs() / (2.0 if dim == 2 else 6.0)
            g = torch.linalg.inv(J)
            g = torch.cat([-g.sum(1, keepdim=True), g], 1)
            Ke = (g * (vol * k)[:, None, None]) @ g.transpose(1, 2).contiguous()
            fe = (vol / (dim + 1))[:, None].expand(-1, dim + 1)
        val = _assembled(E, Ke, n, bnd)
        b = torch.zeros(n, device="cuda", dtype=torch.float64).index_add_(0, E.reshape(-1), fe.reshape(-1))
        d = torch.zeros_like(b).index_add_(0, E.reshape(-1), ((Ke * u[E][:, None, :]).sum(-1) - fe).reshape(-1))
        b[bnd] = 0.0
        d[bnd] = 0.0
        return val, b, d
    return None
