// The part of a multigrid V-cycle below the large levels as one kernel: from
// the defect of a level small enough for the LDS of one workgroup down to the
// base-level solve and back to that level's correction
// (mg_solver_impl.hpp:1686-2136: presmoothing and restriction, base solve,
// prolongation and postsmoothing).
//
// On these levels a launch costs more than its work: about seven launches a
// level of 2 - 4 us each for a few hundred rows. Here one workgroup of 1024
// threads keeps the defect, the correction, the inverse diagonal, two staged
// operands (with a zero halo wide enough for every diagonal) and, where they
// fit, the operator's diagonals of every level in LDS; what does not change
// from cycle to cycle lies packed in memory and comes in with one round of
// wide loads. A step is one pass over the rows and one barrier: a row that has
// its new defect also stages its next operand, into the other buffer. The
// limit is that chain of barriers, six a level, so the levels above, whose rows
// keep the whole chip busy, stay with the kernels that use it
// (coarse_levels_fit). 2D FV1 at 128 x 128, FP64, levels 33 x 33 and below: 74 us
// a cycle in 36 launches, 19 us as one; the solve 1852 -> 1277 us on one MI355X.
// Arithmetic and order of every step are those of the separate kernels
// (k_dias_jacobi_step, k_dia_jacobi_step, k_restrict*, k_prolong*,
// k_jacobi_accumulate, k_lu_solve), so the results are identical.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "lu_block.hpp"
#include "ugx_internal.hpp"

namespace ugamd {

namespace {

constexpr int kThreads = 1024;
constexpr size_t kCoarseLds = 160 * 1024;   // all of a CU's

// KIND 0: hexahedra, 1: triangles (both symmetric Dirichlet-eliminated
// storage), 2: tetrahedra (all 27 diagonals)
template <int KIND>
struct Stencil {
    static constexpr int ND = KIND == 1 ? 9 : 27;
    static constexpr bool SYM = KIND != 2;
};

struct Point {
    int x, y, z;
};
template <int KIND>
__device__ __forceinline__ Point point_of(int r, int W) {
    Point p;
    const unsigned q = (unsigned)r / (unsigned)W;
    p.x = r - (int)q * W;
    if (KIND == 1) {
        p.y = (int)q;
        p.z = 0;
    } else {
        p.z = (int)(q / (unsigned)W);
        p.y = (int)q - p.z * W;
    }
    return p;
}
// The rows a workgroup visits on a level. On the symmetric storage every
// vector vanishes on the Dirichlet points, the lattice boundary, so the last
// point of every line (and plane) is left out: (W-1)^dim rows, a power of two
// (33 x 33: one round of the 1024 threads instead of two). Tetrahedra: all rows.
template <int KIND>
__device__ __forceinline__ int row_count(const int W, const int N) {
    return KIND == 2 ? N : KIND == 1 ? (W - 1) * (W - 1) : (W - 1) * (W - 1) * (W - 1);
}
template <int KIND>
__device__ __forceinline__ Point row_point(int t, int W) {
    if (KIND == 2) return point_of<KIND>(t, W);
    const int sh = __ffs(W - 1) - 1, m = W - 2;
    Point p;
    p.x = t & m;
    p.y = KIND == 1 ? t >> sh : (t >> sh) & m;
    p.z = KIND == 1 ? 0 : t >> (2 * sh);
    return p;
}
template <int KIND>
__device__ __forceinline__ int row_index(int t, int W) {
    if (KIND == 2) return t;
    const Point p = row_point<KIND>(t, W);
    return (p.z * W + p.y) * W + p.x;
}
template <int KIND>
__device__ __forceinline__ bool on_boundary(const Point& p, int W) {
    return p.x == 0 || p.y == 0 || p.x == W - 1 || p.y == W - 1 || (KIND != 1 && (p.z == 0 || p.z == W - 1));
}

// sum over the diagonals of row r times the staged operand (row 0 at xs[0]);
// in: the diagonals are in LDS, N apart, else in the level's tiles
template <typename T, int KIND>
__device__ __forceinline__ T row_sum(const CoarseLevel<T>& l, const T* lds, int r, const T* xs) {
    constexpr int ND = Stencil<KIND>::ND, NU = ND / 2 + 1;
    const int W = l.W, N = l.N;
    T a[ND];
    int off[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
        off[d] = d % 3 - 1 + ((d / 3) % 3 - 1) * W + (ND == 27 ? (d / 9 - 1) * W * W : 0);
    if (Stencil<KIND>::SYM) {
        // a coupling that leaves the lattice: any coefficient, times a halo zero
        if (l.a >= 0) {
            const T* A = lds + l.a;
#pragma unroll
            for (int u = 0; u < NU; ++u) a[ND / 2 + u] = A[u * N + r];
#pragma unroll
            for (int d = 0; d < ND / 2; ++d) a[d] = A[(ND - 1 - d - ND / 2) * N + max(r + off[d], 0)];
        } else {
#pragma unroll
            for (int u = 0; u < NU; ++u) a[ND / 2 + u] = l.A[dia_tiled_index(u, r, NU)];
#pragma unroll
            for (int d = 0; d < ND / 2; ++d) a[d] = l.A[dia_tiled_index(ND - 1 - d - ND / 2, max(r + off[d], 0), NU)];
        }
    } else if (l.a >= 0) {
#pragma unroll
        for (int d = 0; d < ND; ++d) a[d] = lds[l.a + d * N + r];
    } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) a[d] = l.A[dia_tiled_index(d, r, ND)];
    }
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xs[r + off[d]], s);
    return s;
}

// what follows a smoothing step's new defect
enum Next { kStage, kAccumulate, kNothing };

// one pass: sd -= A x, with COUNT sc += x; then the next step's operand
// x_next = dinv .* sd, or the last update sc += dinv .* sd
template <typename T, int KIND, bool COUNT>
__device__ __forceinline__ void step(const CoarseLevel<T>& l, T* lds, const T* x, T* x_next, Next next) {
    T *sd = lds + l.sd, *sc = lds + l.sc;
    const T* dinv = lds + l.dinv;
    const int rows = row_count<KIND>(l.W, l.N);
    for (int t = threadIdx.x; t < rows; t += kThreads) {
        const int r = row_index<KIND>(t, l.W);
        const T d = sd[r] - row_sum<T, KIND>(l, lds, r, x);
        sd[r] = d;
        T c = (T)0;
        if (COUNT) c = sc[r] + x[r];
        if (next == kStage) x_next[r] = dinv[r] * d;
        else if (next == kAccumulate) c = (T)((double)(COUNT ? c : sc[r]) + (double)dinv[r] * (double)d);
        if (COUNT || next == kAccumulate) sc[r] = c;
    }
    __syncthreads();
}

// sdc = R sdf and, with dinv, the first operand there xc = dinv .* sdc
template <typename T, int KIND>
__device__ __forceinline__ void restrict_to(const CoarseLevel<T>& f, int Wc, int Nc, const T* sdf, T* sdc,
                                            const T* dinv, T* xc) {
    const int Wf = f.W;
    const int rows = row_count<KIND>(Wc, Nc);
    for (int t = threadIdx.x; t < rows; t += kThreads) {
        const Point p = row_point<KIND>(t, Wc);
        const int c = (p.z * Wc + p.y) * Wc + p.x;
        const int f0 = KIND == 1 ? 2 * p.y * Wf + 2 * p.x : (2 * p.z * Wf + 2 * p.y) * Wf + 2 * p.x;
        // boundary points take the value of their fine copy; the fine
        // neighbours of the others are inside the lattice and off its boundary
        double s = 0.0;
        if (on_boundary<KIND>(p, Wc)) {
            s = (double)sdf[f0];
        } else if (KIND == 1) {
            constexpr int dxs[7] = {0, 1, -1, 0, 0, 1, -1}, dys[7] = {0, 0, 0, 1, -1, 1, -1};
#pragma unroll
            for (int k = 0; k < 7; ++k) s += (k == 0 ? 1.0 : 0.5) * (double)sdf[f0 + dys[k] * Wf + dxs[k]];
        } else if (KIND == 0) {
#pragma unroll
            for (int d = 0; d < 27; ++d) {
                const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
                const int nodd = (dx != 0) + (dy != 0) + (dz != 0);
                const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                s += w * (double)sdf[f0 + (dz * Wf + dy) * Wf + dx];
            }
        } else {
            s = (double)sdf[f0];
            uint8_t code[27];
#pragma unroll
            for (int d = 0; d < 27; ++d)
                code[d] = f.pcode[f0 + ((d / 9 - 1) * Wf + (d / 3) % 3 - 1) * Wf + d % 3 - 1];
#pragma unroll
            for (int d = 0; d < 27; ++d) {
                if (d == 13) continue;
                if (code[d] == (d > 13 ? d - 13 : 13 - d))
                    s += 0.5 * (double)sdf[f0 + ((d / 9 - 1) * Wf + (d / 3) % 3 - 1) * Wf + d % 3 - 1];
            }
        }
        const T v = (T)s;
        sdc[c] = v;
        if (dinv) xc[c] = dinv[c] * v;
    }
}

// x = P scc (staged for the defect update) ; sc += x
template <typename T, int KIND>
__device__ __forceinline__ void prolong_to(const CoarseLevel<T>& f, int Wc, const T* scc, T* x, T* sc) {
    const int W = f.W;
    const int rows = row_count<KIND>(W, f.N);
    for (int t = threadIdx.x; t < rows; t += kThreads) {
        const Point p = row_point<KIND>(t, W);
        const int r = (p.z * W + p.y) * W + p.x;
        const bool bnd = on_boundary<KIND>(p, W);
        const int ox = p.x & 1, oy = p.y & 1, oz = p.z & 1, x0 = p.x >> 1, y0 = p.y >> 1, z0 = p.z >> 1;
        double v = 0.0;
        if (KIND == 2) {
            const int code = f.pcode[r];
            if (code == 0) {
                v = (double)scc[(z0 * Wc + y0) * Wc + x0];
            } else if (!bnd) {
                const int d = code + 13;
                const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
                const int a = (((p.z - dz) >> 1) * Wc + ((p.y - dy) >> 1)) * Wc + ((p.x - dx) >> 1);
                const int b = (((p.z + dz) >> 1) * Wc + ((p.y + dy) >> 1)) * Wc + ((p.x + dx) >> 1);
                v = 0.5 * (double)scc[a] + 0.5 * (double)scc[b];
            }
        } else if (KIND == 1) {
            if (bnd && (ox | oy)) v = 0.0;
            else if (!(ox | oy)) v = (double)scc[y0 * Wc + x0];
            else v = 0.5 * (double)scc[y0 * Wc + x0] + 0.5 * (double)scc[(y0 + oy) * Wc + x0 + ox];
        } else {
            const int nodd = ox + oy + oz;
            if (!(bnd && nodd != 0)) {
                const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                for (int dz = 0; dz <= oz; ++dz)
                    for (int dy = 0; dy <= oy; ++dy)
                        for (int dx = 0; dx <= ox; ++dx)
                            v = fma(w, (double)scc[((z0 + dz) * Wc + y0 + dy) * Wc + x0 + dx], v);
            }
        }
        const T st = (T)v;
        x[r] = st;
        sc[r] = sc[r] + st;
    }
}

template <typename T, int KIND>
__global__ __launch_bounds__(kThreads) void k_coarse_cycle(CoarseCycle<T> c) {
    extern __shared__ __align__(16) unsigned char raw[];
    T* lds = reinterpret_cast<T*>(raw);
    double* lu = reinterpret_cast<double*>(raw + c.lu_bytes);
    typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
    // the packed constants (diagonals that fit, inverse diagonals) and the first
    // level's defect and correction; every other entry starts at zero
    {
        constexpr int U = 4, V = 16 / sizeof(T);
        const vec* src = reinterpret_cast<const vec*>(c.pack);
        vec* dst = reinterpret_cast<vec*>(raw);
        const int nv = c.pack_n / V, nz = c.vec_end / V;
        for (int i = nv + (int)threadIdx.x; i < nz; i += kThreads) dst[i] = (vec)(T)0;
        for (int i0 = threadIdx.x; i0 < nv; i0 += U * kThreads) {
            vec q[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * kThreads < nv) q[u] = src[i0 + u * kThreads];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (i0 + u * kThreads < nv) dst[i0 + u * kThreads] = q[u];
        }
    }
    const CoarseLevel<T>& top = c.L[0];
    const int top_rows = row_count<KIND>(top.W, top.N);
    __syncthreads();
    for (int t = threadIdx.x; t < top_rows; t += kThreads) {
        const int r = row_index<KIND>(t, top.W);
        const T d = c.sd[r];
        lds[top.sd + r] = d;
        lds[top.sc + r] = c.sc[r];
        lds[top.x + r] = lds[top.dinv + r] * d;
    }
    __syncthreads();
    for (int k = 0; k < c.nl; ++k) {
        const CoarseLevel<T>& l = c.L[k];
        T *x = lds + l.x, *xn = lds + l.x1;
        for (int nu = 0; nu < c.nu1; ++nu) {
            step<T, KIND, true>(l, lds, x, xn, nu + 1 < c.nu1 ? kStage : kNothing);
            T* t = x;
            x = xn;
            xn = t;
        }
        if (k + 1 == c.nl)
            restrict_to<T, KIND>(l, c.Wb, c.lu_n, lds + l.sd, lds + c.base_sd, (const T*)nullptr, (T*)nullptr);
        else
            restrict_to<T, KIND>(l, c.L[k + 1].W, c.L[k + 1].N, lds + l.sd, lds + c.L[k + 1].sd,
                                 lds + c.L[k + 1].dinv, lds + c.L[k + 1].x);
        __syncthreads();
    }
    lu_solve_block<T>(c.lu_n, c.Linv, c.Uinv, c.perm, lds + c.base_sd, lds + c.base_sc, lu);
    __syncthreads();
    for (int k = c.nl - 1; k >= 0; --k) {
        const CoarseLevel<T>& l = c.L[k];
        const bool last = k + 1 == c.nl;
        T *x = lds + l.x, *xn = lds + l.x1;
        prolong_to<T, KIND>(l, last ? c.Wb : c.L[k + 1].W, lds + (last ? c.base_sc : c.L[k + 1].sc), x, lds + l.sc);
        __syncthreads();
        for (int nu = 0; nu < c.nu2; ++nu) {
            const Next next = nu + 1 < c.nu2 ? kStage : kAccumulate;
            if (nu == 0) step<T, KIND, false>(l, lds, x, xn, next);
            else step<T, KIND, true>(l, lds, x, xn, next);
            T* t = x;
            x = xn;
            xn = t;
        }
    }
    for (int t = threadIdx.x; t < top_rows; t += kThreads) {
        const int r = row_index<KIND>(t, top.W);
        c.sc[r] = lds[top.sc + r];
    }
}

// the constants of a plan in the order of its LDS: one level per blockIdx.y
template <typename T>
__global__ __launch_bounds__(256) void k_coarse_pack(CoarseCycle<T> c, int ns, T* __restrict__ pack) {
    const CoarseLevel<T>& l = c.L[blockIdx.y];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < l.N) pack[l.dinv + i] = l.g_dinv[i];
    if (l.a >= 0 && i < ns * l.N) {
        const int d = i / l.N, r = i - d * l.N;
        pack[l.a + i] = l.A[dia_tiled_index(d, r, ns)];
    }
}

template <typename T>
const void* coarse_kernel(int kind) {
    return kind == 0   ? reinterpret_cast<const void*>(&k_coarse_cycle<T, 0>)
           : kind == 1 ? reinterpret_cast<const void*>(&k_coarse_cycle<T, 1>)
                       : reinterpret_cast<const void*>(&k_coarse_cycle<T, 2>);
}

}  // namespace

int stored_diagonals(int kind) { return kind == 0 ? 14 : kind == 1 ? 5 : 27; }

// LDS of a plan: the constants (pack_n entries: inverse diagonals, and the
// diagonals from the coarsest level up as long as they fit), the levels'
// vectors and the base level's defect and correction (up to vec_end), the
// scratch of the base solve. Parts start at multiples of 16 bytes
template <typename T>
size_t coarse_plan(int kind, CoarseCycle<T>& c) {
    auto round16 = [](int n) { return (n + 15) / 16 * 16; };
    const int ns = stored_diagonals(kind);
    size_t vec = 2 * (size_t)c.lu_n, lu = 2 * sizeof(double) * (size_t)c.lu_n + 256 * sizeof(T);
    int at = 0;
    for (int k = 0; k < c.nl; ++k) {
        CoarseLevel<T>& l = c.L[k];
        l.halo = (kind == 1 ? 0 : l.W * l.W) + l.W + 1;
        vec += (size_t)4 * l.N + 3 * l.halo;
        l.dinv = at;
        at += l.N;
    }
    for (int k = c.nl - 1; k >= 0; --k) {
        CoarseLevel<T>& l = c.L[k];
        const bool fits = ((size_t)(at + ns * l.N) + vec) * sizeof(T) + lu <= kCoarseLds;
        l.a = fits ? at : -1;
        if (fits) at += ns * l.N;
    }
    c.pack_n = at = round16(at);
    for (int k = 0; k < c.nl; ++k) {
        CoarseLevel<T>& l = c.L[k];
        l.x = at + l.halo;
        l.x1 = l.x + l.N + l.halo;   // the two operands share the zeros between them
        l.sd = l.x1 + l.N + l.halo;
        l.sc = l.sd + l.N;
        at = l.sc + l.N;
    }
    c.base_sd = at;
    c.base_sc = at + c.lu_n;
    c.vec_end = at = round16(at + 2 * c.lu_n);
    c.lu_bytes = (int)((size_t)at * sizeof(T));
    return (size_t)c.lu_bytes + 2 * sizeof(double) * (size_t)c.lu_n;
}
template size_t coarse_plan<float>(int, CoarseCycle<float>&);
template size_t coarse_plan<double>(int, CoarseCycle<double>&);

// Levels of at most kCoarseRows rows whose plan fits the LDS of a workgroup.
template <typename T>
bool coarse_levels_fit(int kind, CoarseCycle<T>& c) {
    if (c.nl < 1 || c.nl > kCoarseMaxLevels || c.lu_n < 1 || c.lu_n > 512) return false;
    if (c.L[0].N > kCoarseRows) return false;
    return coarse_plan<T>(kind, c) <= kCoarseLds;
}
template bool coarse_levels_fit<float>(int, CoarseCycle<float>&);
template bool coarse_levels_fit<double>(int, CoarseCycle<double>&);

template <typename T>
int coarse_pack(int kind, const CoarseCycle<T>& c, T* pack, hipStream_t s) {
    const int ns = stored_diagonals(kind);
    int most = 0;
    for (int k = 0; k < c.nl; ++k) most = c.L[k].N > most ? c.L[k].N : most;
    hipLaunchKernelGGL(k_coarse_pack<T>, dim3((unsigned)((ns * most + 255) / 256), (unsigned)c.nl), dim3(256), 0, s, c, ns,
                       pack);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int coarse_pack<float>(int, const CoarseCycle<float>&, float*, hipStream_t);
template int coarse_pack<double>(int, const CoarseCycle<double>&, double*, hipStream_t);

template <typename T>
int coarse_cycle(int kind, const CoarseCycle<T>& c, hipStream_t s) {
    CoarseCycle<T> a = c;
    const size_t lds = coarse_plan<T>(kind, a);
    void* args[] = {&a};
    return hipLaunchKernel(coarse_kernel<T>(kind), dim3(1), dim3(kThreads), args, lds, s) == hipSuccess ? 0 : -1;
}
template int coarse_cycle<float>(int, const CoarseCycle<float>&, hipStream_t);
template int coarse_cycle<double>(int, const CoarseCycle<double>&, hipStream_t);

}  // namespace ugamd
