// The part of a multigrid V-cycle below the large levels as one kernel: from
// the defect of a level small enough for the LDS of one workgroup down to the
// base-level solve and back to that level's correction
// (mg_solver_impl.hpp:1686-2136: presmoothing and restriction, base solve,
// prolongation and postsmoothing).
//
// On these levels a launch costs more than its work: about seven launches a
// level of 2 - 4 us each for a few hundred rows. Here one workgroup of 1024
// threads keeps the defect, the correction, the inverse diagonal and the
// staged operand of every level in LDS (the operand with a zero halo wide
// enough for every diagonal), and a step is a pass over the rows and a barrier;
// only the operator's diagonals come from memory, 27 (9) independent loads
// per row. The limit is the chain of barriers and first loads, so the levels
// above, whose diagonals alone are more than a CU fetches in a launch's time,
// stay with the kernels that use the whole chip (coarse_levels_fit).
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
template <int KIND>
__device__ __forceinline__ bool on_boundary(const Point& p, int W) {
    return p.x == 0 || p.y == 0 || p.x == W - 1 || p.y == W - 1 || (KIND != 1 && (p.z == 0 || p.z == W - 1));
}

// sum over the diagonals of row r times the staged operand (row 0 at xs[0])
template <typename T, int KIND>
__device__ __forceinline__ T row_sum(const T* __restrict__ A, int r, int N, int W, const T* xs) {
    constexpr int ND = Stencil<KIND>::ND, NU = ND / 2 + 1;
    T a[ND];
    int off[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
        off[d] = d % 3 - 1 + ((d / 3) % 3 - 1) * W + (ND == 27 ? (d / 9 - 1) * W * W : 0);
    if (Stencil<KIND>::SYM) {
#pragma unroll
        for (int u = 0; u < NU; ++u) a[ND / 2 + u] = A[dia_tiled_index(u, r, NU)];
#pragma unroll
        for (int d = 0; d < ND / 2; ++d) {
            int j = r + off[d];
            j = j < 0 ? 0 : j;   // coefficient of a coupling that leaves the lattice: times a halo zero
            a[d] = A[dia_tiled_index(ND - 1 - d - ND / 2, j, NU)];
        }
    } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) a[d] = A[dia_tiled_index(d, r, ND)];
    }
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xs[r + off[d]], s);
    return s;
}

// st = dinv .* sd ; sd -= A st ; sc += st
template <typename T, int KIND>
__device__ __forceinline__ void jacobi(const CoarseLevel<T>& l, T* lds) {
    T *x = lds + l.x, *sd = lds + l.sd, *sc = lds + l.sc;
    const T* dinv = lds + l.dinv;
    for (int r = threadIdx.x; r < l.N; r += kThreads) x[r] = dinv[r] * sd[r];
    __syncthreads();
    for (int r = threadIdx.x; r < l.N; r += kThreads) {
        const T s = row_sum<T, KIND>(l.A, r, l.N, l.W, x);
        sd[r] = sd[r] - s;
        sc[r] = sc[r] + x[r];
    }
    __syncthreads();
}

// sdc = R sdf
template <typename T, int KIND>
__device__ __forceinline__ void restrict_to(const CoarseLevel<T>& f, int Wc, int Nc, const T* sdf, T* sdc) {
    const int Wf = f.W;
    for (int c = threadIdx.x; c < Nc; c += kThreads) {
        const Point p = point_of<KIND>(c, Wc);
        const int f0 = KIND == 1 ? 2 * p.y * Wf + 2 * p.x : (2 * p.z * Wf + 2 * p.y) * Wf + 2 * p.x;
        // boundary points take the value of their fine copy; the fine
        // neighbours of the others are inside the lattice and off its boundary
        if (on_boundary<KIND>(p, Wc)) {
            sdc[c] = sdf[f0];
            continue;
        }
        double s;
        if (KIND == 1) {
            constexpr int dxs[7] = {0, 1, -1, 0, 0, 1, -1}, dys[7] = {0, 0, 0, 1, -1, 1, -1};
            s = 0.0;
#pragma unroll
            for (int k = 0; k < 7; ++k) s += (k == 0 ? 1.0 : 0.5) * (double)sdf[f0 + dys[k] * Wf + dxs[k]];
        } else if (KIND == 0) {
            s = 0.0;
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
        sdc[c] = (T)s;
    }
}

// x = P scc (staged for the defect update) ; sc += x
template <typename T, int KIND>
__device__ __forceinline__ void prolong_to(const CoarseLevel<T>& f, int Wc, const T* scc, T* x, T* sc) {
    const int W = f.W;
    for (int r = threadIdx.x; r < f.N; r += kThreads) {
        const Point p = point_of<KIND>(r, W);
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
        const T t = (T)v;
        x[r] = t;
        sc[r] = sc[r] + t;
    }
}

template <typename T, int KIND>
__global__ __launch_bounds__(kThreads) void k_coarse_cycle(CoarseCycle<T> c) {
    extern __shared__ __align__(16) unsigned char raw[];
    T* lds = reinterpret_cast<T*>(raw);
    double* lu = reinterpret_cast<double*>(raw + c.lu_bytes);
    // operands (with their halos) and the lower levels' corrections start at
    // zero; the inverse diagonals, and the first level's defect and correction
    for (int k = 0; k < c.nl; ++k) {
        const CoarseLevel<T>& l = c.L[k];
        for (int r = (int)threadIdx.x - l.halo; r < l.N + l.halo; r += kThreads) lds[l.x + r] = (T)0;
        for (int r = threadIdx.x; r < l.N; r += kThreads) {
            lds[l.dinv + r] = l.g_dinv[r];
            lds[l.sc + r] = k == 0 ? c.sc[r] : (T)0;
            if (k == 0) lds[l.sd + r] = c.sd[r];
        }
    }
    __syncthreads();
    for (int k = 0; k < c.nl; ++k) {
        const CoarseLevel<T>& l = c.L[k];
        for (int nu = 0; nu < c.nu1; ++nu) jacobi<T, KIND>(l, lds);
        const bool last = k + 1 == c.nl;
        restrict_to<T, KIND>(l, last ? c.Wb : c.L[k + 1].W, last ? c.lu_n : c.L[k + 1].N, lds + l.sd,
                             lds + (last ? c.base_sd : c.L[k + 1].sd));
        __syncthreads();
    }
    lu_solve_block<T>(c.lu_n, c.Linv, c.Uinv, c.perm, lds + c.base_sd, lds + c.base_sc, lu);
    __syncthreads();
    for (int k = c.nl - 1; k >= 0; --k) {
        const CoarseLevel<T>& l = c.L[k];
        const bool last = k + 1 == c.nl;
        T *x = lds + l.x, *sd = lds + l.sd, *sc = lds + l.sc;
        const T* dinv = lds + l.dinv;
        prolong_to<T, KIND>(l, last ? c.Wb : c.L[k + 1].W, lds + (last ? c.base_sc : c.L[k + 1].sc), x, sc);
        __syncthreads();
        if (c.nu2 > 0) {
            for (int r = threadIdx.x; r < l.N; r += kThreads) sd[r] = sd[r] - row_sum<T, KIND>(l.A, r, l.N, l.W, x);
            __syncthreads();
            for (int nu = 0; nu + 1 < c.nu2; ++nu) jacobi<T, KIND>(l, lds);
            for (int r = threadIdx.x; r < l.N; r += kThreads)
                sc[r] = (T)((double)sc[r] + (double)dinv[r] * (double)sd[r]);
            __syncthreads();
        }
    }
    for (int r = threadIdx.x; r < c.L[0].N; r += kThreads) c.sc[r] = lds[c.L[0].sc + r];
}

template <typename T>
const void* coarse_kernel(int kind) {
    return kind == 0   ? reinterpret_cast<const void*>(&k_coarse_cycle<T, 0>)
           : kind == 1 ? reinterpret_cast<const void*>(&k_coarse_cycle<T, 1>)
                       : reinterpret_cast<const void*>(&k_coarse_cycle<T, 2>);
}

}  // namespace

// LDS of a plan: the levels' arrays one after another, then the base level's
// defect and correction, then the scratch of the base solve
template <typename T>
size_t coarse_plan(int kind, CoarseCycle<T>& c) {
    int at = 0;
    for (int k = 0; k < c.nl; ++k) {
        CoarseLevel<T>& l = c.L[k];
        l.halo = (kind == 1 ? 0 : l.W * l.W) + l.W + 1;
        l.x = at + l.halo;
        l.sd = at + l.N + 2 * l.halo;
        l.sc = l.sd + l.N;
        l.dinv = l.sc + l.N;
        at = l.dinv + l.N;
    }
    c.base_sd = at;
    c.base_sc = at + c.lu_n;
    at += 2 * c.lu_n;
    c.lu_bytes = (int)(((size_t)at * sizeof(T) + 7) / 8 * 8);
    return (size_t)c.lu_bytes + 2 * sizeof(double) * (size_t)c.lu_n;
}
template size_t coarse_plan<float>(int, CoarseCycle<float>&);
template size_t coarse_plan<double>(int, CoarseCycle<double>&);

// Levels of at most kCoarseRows rows whose plan fits the LDS of a workgroup.
template <typename T>
bool coarse_levels_fit(int kind, CoarseCycle<T>& c) {
    if (c.nl < 1 || c.nl > kCoarseMaxLevels || c.lu_n < 1 || c.lu_n > 512) return false;
    if (c.L[0].N > kCoarseRows) return false;
    return coarse_plan<T>(kind, c) <= 64 * 1024;
}
template bool coarse_levels_fit<float>(int, CoarseCycle<float>&);
template bool coarse_levels_fit<double>(int, CoarseCycle<double>&);

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
