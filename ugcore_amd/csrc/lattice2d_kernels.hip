// The triangular hierarchy's lattice kernels (2D, diagonals along (1,1)): P1
// transfer between two levels, and the two products of a CG step with the
// stored 9-diagonal top level that end or begin with something else. These
// lattices have 10^3 - 10^6 points: a launch is one chain of dependent loads, so
// every load of a point is issued before the first is looked at, and a vector
// operation is part of the product beside it instead of a launch of its own.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ugx_internal.hpp"

namespace ugamd {

namespace {

// st_f = sum_c P(f,c) c_c ; sc_f += st_f. Odd coordinates lie on axis edges or on
// the (1,1) diagonal: the mean of the two ends. Dirichlet rows of P are zeroed
// except vertex copies. With dinv the coarse correction's last update is folded in
// (coarse_fold). One MI355X, FP64, 65^2 -> 129^2: 4.2 us with the loads behind
// branches, 2.8 us so.
template <typename TV>
__global__ __launch_bounds__(256) void k_prolong2(int Wc, int Wf, int n_f, const TV* __restrict__ c,
                                                  const TV* __restrict__ dinv, const TV* __restrict__ sd,
                                                  const uint8_t* __restrict__ dir_f, TV* __restrict__ st,
                                                  TV* __restrict__ sc) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_f) return;
    const int y = i / Wf, x = i - y * Wf, ox = x & 1, oy = y & 1;
    const int j0 = (y >> 1) * Wc + (x >> 1), j1 = ((y >> 1) + oy) * Wc + (x >> 1) + ox;
    TV a = c[j0], b = c[j1];
    const TV old = sc[i];
    const uint8_t dir = dir_f[i];
    if (dinv) {
        const TV d0 = dinv[j0], d1 = dinv[j1], s0 = sd[j0], s1 = sd[j1];
        a = coarse_fold<TV>(a, d0, s0);
        b = coarse_fold<TV>(b, d1, s1);
    }
    const bool odd = (ox | oy) != 0;
    // Dirichlet DoFs lie on the lattice boundary
    const bool bnd = x == 0 || y == 0 || x == Wf - 1 || y == Wf - 1;
    double v = odd ? 0.5 * (double)a + 0.5 * (double)b : (double)a;
    if (odd && bnd && dir) v = 0.0;
    // c += t in the vector precision (mg_solver_impl.hpp:1905)
    const TV t = (TV)v;
    st[i] = t;
    sc[i] = old + t;
}

// d_c = sum_f P(f,c) d_f, the transpose; zc: the coarse correction, set to zero.
// One MI355X, FP64, 129^2 -> 65^2: 5.0 us with the loads behind branches, 2.7 us so.
template <typename TV>
__global__ __launch_bounds__(256) void k_restrict2(int Wc, int Wf, int n_c, const TV* __restrict__ sdf,
                                                   const uint8_t* __restrict__ dir_c,
                                                   const uint8_t* __restrict__ dir_f, TV* __restrict__ sdc,
                                                   TV* __restrict__ zc) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= n_c) return;
    const int y = c / Wc, x = c - y * Wc;
    constexpr int dx[7] = {0, 1, -1, 0, 0, 1, -1}, dy[7] = {0, 0, 0, 1, -1, 1, -1};
    TV v[7];
    uint8_t dir[7];
    bool in[7];
    const uint8_t own = dir_c[c];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        const int fx = 2 * x + dx[k], fy = 2 * y + dy[k];
        in[k] = fx >= 0 && fy >= 0 && fx < Wf && fy < Wf;
        const int f = in[k] ? fy * Wf + fx : 0;
        v[k] = sdf[f];
        dir[k] = dir_f[f];
    }
    double s = (double)v[0];
#pragma unroll
    for (int k = 1; k < 7; ++k)
        if (in[k] && !dir[k]) s += 0.5 * (double)v[k];   // Dirichlet rows of P are zero
    sdc[c] = own ? v[0] : (TV)s;
    if (zc) zc[c] = (TV)0;
}

__device__ __forceinline__ void block_partial2(double acc, double* partial) {
    __shared__ double sh[4];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// the nine coefficients of row i in symmetric storage (the lower ones are the
// upper ones of the rows that they point to)
template <typename TM>
__device__ __forceinline__ void row9(const TM* __restrict__ U, int W, int n, int i, TM (&a)[9], int (&j)[9]) {
#pragma unroll
    for (int d = 0; d < 9; ++d) j[d] = i + (d / 3 - 1) * W + d % 3 - 1;
#pragma unroll
    for (int u = 0; u < 5; ++u) a[4 + u] = U[dia_tiled_index(u, i, 5)];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int r = j[d] < 0 ? 0 : j[d];
        a[d] = U[dia_tiled_index(4 - d, r, 5)];
    }
}

// y = A x and the partial sums of (y, x): x carries the halo
__global__ __launch_bounds__(256) void k_dias9_product_dot(int W, int n, const double* __restrict__ U,
                                                           const double* __restrict__ x, double* __restrict__ y,
                                                           double* __restrict__ partial) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    double dot = 0.0;
    if (i < n) {
        double a[9], v[9];
        int j[9];
        row9(U, W, n, i, a, j);
#pragma unroll
        for (int d = 0; d < 9; ++d) v[d] = x[j[d]];
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < 9; ++d) s = fma(a[d], v[d], s);
        y[i] = s;
        dot = s * v[4];
    }
    block_partial2(dot, partial);
}

// the first Jacobi step of a cycle from the FP64 defect and a zero correction:
// sd = (T)d64 - A st, sc = st, st = dinv .* (T)d64 (d64 without a halo)
template <typename T>
__global__ __launch_bounds__(256) void k_dias9_first(int W, int n, const T* __restrict__ U,
                                                     const T* __restrict__ dinv, const double* __restrict__ d64,
                                                     T* __restrict__ sd, T* __restrict__ sc) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    T a[9], dv[9], v[9];
    int j[9];
    row9(U, W, n, i, a, j);
#pragma unroll
    for (int d = 0; d < 9; ++d) {
        dv[d] = dinv[j[d]];
        const bool in = j[d] >= 0 && j[d] < n;
        const T t = (T)d64[in ? j[d] : i];
        v[d] = in ? t : (T)0;
    }
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < 9; ++d) s = fma(a[d], dv[d] * v[d], s);
    sd[i] = v[4] - s;
    sc[i] = dv[4] * v[4];
}

}  // namespace

template <typename TV>
int prolong2(int Wc, int Wf, const TV* c, const TV* dinv, const TV* sd, const uint8_t* dir_f, TV* st, TV* sc,
             hipStream_t s) {
    const int64_t n = (int64_t)Wf * Wf;
    if (n > INT32_MAX || Wf != 2 * Wc - 1) return -1;
    hipLaunchKernelGGL(k_prolong2<TV>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Wc, Wf, (int)n, c, dinv, sd,
                       dir_f, st, sc);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int prolong2<float>(int, int, const float*, const float*, const float*, const uint8_t*, float*, float*,
                             hipStream_t);
template int prolong2<double>(int, int, const double*, const double*, const double*, const uint8_t*, double*, double*,
                              hipStream_t);

template <typename TV>
int restrict2(int Wc, int Wf, const TV* sdf, const uint8_t* dir_c, const uint8_t* dir_f, TV* sdc, TV* zero_c,
              hipStream_t s) {
    const int64_t n = (int64_t)Wc * Wc;
    if ((int64_t)Wf * Wf > INT32_MAX || Wf != 2 * Wc - 1) return -1;
    hipLaunchKernelGGL(k_restrict2<TV>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, Wc, Wf, (int)n, sdf, dir_c,
                       dir_f, sdc, zero_c);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int restrict2<float>(int, int, const float*, const uint8_t*, const uint8_t*, float*, float*, hipStream_t);
template int restrict2<double>(int, int, const double*, const uint8_t*, const uint8_t*, double*, double*, hipStream_t);

int dias9_product_dot(int W, const double* U, const double* x, double* y, double* partial, int* n_partial,
                      hipStream_t s) {
    const int64_t n = (int64_t)W * W, g = (n + 255) / 256;
    if (n > INT32_MAX || g > *n_partial) return -1;
    hipLaunchKernelGGL(k_dias9_product_dot, dim3((unsigned)g), dim3(256), 0, s, W, (int)n, U, x, y, partial);
    *n_partial = (int)g;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename T>
int dias9_first(int W, const T* U, const T* dinv, const double* d64, T* sd, T* sc, hipStream_t s) {
    const int64_t n = (int64_t)W * W;
    if (n > INT32_MAX) return -1;
    hipLaunchKernelGGL(k_dias9_first<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, W, (int)n, U, dinv, d64, sd,
                       sc);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int dias9_first<float>(int, const float*, const float*, const double*, float*, float*, hipStream_t);
template int dias9_first<double>(int, const double*, const double*, const double*, double*, double*, hipStream_t);

}  // namespace ugamd
