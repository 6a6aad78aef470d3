// BiCGStab (bicgstab.h:112-385) on lattice-ordered vectors with the FP64
// scalars of a step formed on the device: the two vector updates of a half
// step, each fused with the partial sums that the next one needs and with the
// defect that the preconditioning cycle reads, in the cycle's precision.
// Bound by HBM: every vector of an update is read and written once.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ugx_internal.hpp"

namespace ugamd {

namespace {

constexpr int kE = 2;   // elements per thread and pass
inline unsigned grid_of(int64_t n) {
    const int64_t g = (n + 256 * kE - 1) / (256 * kE);
    return (unsigned)(g < 1 ? 1 : (g > kBicgMaxBlocks ? kBicgMaxBlocks : g));
}

#define BICG_LOOP(n)                                                             \
    for (int64_t b0 = blockIdx.x * (int64_t)(256 * kE); b0 < (n);               \
         b0 += (int64_t)gridDim.x * (256 * kE))

template <int M>
__device__ __forceinline__ void partials(double (&acc)[M], double* part) {
    __shared__ double sh[M][4];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        for (int o = 32; o > 0; o >>= 1) acc[m] += __shfl_down(acc[m], o, 64);
        if ((threadIdx.x & 63) == 0) sh[m][threadIdx.x >> 6] = acc[m];
    }
    __syncthreads();
    if (threadIdx.x < M) {
        const double* s = sh[threadIdx.x];
        part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
    }
}

// p = r (first), else p = r + beta p - beta omega v; the cycle's defect
// sd = (T)p and its zero correction
template <typename T>
__global__ __launch_bounds__(256) void k_bicg_p(int64_t n, int first, double beta, double omega,
                                                const double* __restrict__ r, double* __restrict__ p,
                                                const double* __restrict__ v, double* __restrict__ r0,
                                                T* __restrict__ sd, T* __restrict__ sc) {
    const double bo = -beta * omega;
    BICG_LOOP(n) {
        double rv[kE], pv[kE], vv[kE];
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const int64_t i = b0 + e * 256 + threadIdx.x, j = i < n ? i : 0;
            rv[e] = r[j];
            pv[e] = first ? 0.0 : p[j];
            vv[e] = first ? 0.0 : v[j];
        }
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const int64_t i = b0 + e * 256 + threadIdx.x;
            if (i >= n) continue;
            double q = rv[e];
            if (!first) {
                q = 1.0 * rv[e] + beta * pv[e];
                q += bo * vv[e];
            } else {
                r0[i] = rv[e];   // a restart takes the defect as the shadow vector
            }
            p[i] = q;
            sd[i] = (T)q;
            sc[i] = (T)0;
        }
    }
}

// alpha = rho / (v, r0); s = r - alpha v, x += alpha q, (s, s); sd = (T)s and
// a zero correction. (v, r0) == 0: nothing is changed (the host stops)
template <typename T>
__global__ __launch_bounds__(256) void k_bicg_s(int64_t n, double rho, const double* __restrict__ sc_dev,
                                                const double* __restrict__ r, const double* __restrict__ v,
                                                const T* __restrict__ q, double* __restrict__ s,
                                                double* __restrict__ x, double* __restrict__ part, T* __restrict__ sd,
                                                T* __restrict__ sc) {
    const double vr0 = sc_dev[0];
    double acc[1] = {0.0};
    if (vr0 != 0.0) {
        const double alpha = rho / vr0;
        BICG_LOOP(n) {
            double rv[kE], vv[kE], qv[kE], xv[kE];
#pragma unroll
            for (int e = 0; e < kE; ++e) {
                const int64_t i = b0 + e * 256 + threadIdx.x, j = i < n ? i : 0;
                rv[e] = r[j];
                vv[e] = v[j];
                qv[e] = (double)q[j];
                xv[e] = x[j];
            }
#pragma unroll
            for (int e = 0; e < kE; ++e) {
                const int64_t i = b0 + e * 256 + threadIdx.x;
                if (i >= n) continue;
                x[i] = 1.0 * xv[e] + alpha * qv[e];
                const double sv = 1.0 * rv[e] + (-alpha) * vv[e];
                s[i] = sv;
                sd[i] = (T)sv;
                sc[i] = (T)0;
                acc[0] += sv * sv;
            }
        }
    }
    partials<1>(acc, part);
}

// omega = (s, t) / (t, t); x += omega q, r = s - omega t, (r, r) and (r0, r).
// (t, t) == 0: nothing is changed
template <typename T>
__global__ __launch_bounds__(256) void k_bicg_r(int64_t n, const double* __restrict__ sc_dev,
                                                const double* __restrict__ s, const double* __restrict__ t,
                                                const T* __restrict__ q, const double* __restrict__ r0,
                                                double* __restrict__ r, double* __restrict__ x,
                                                double* __restrict__ part) {
    const double st = sc_dev[0], tt = sc_dev[1];
    double acc[2] = {0.0, 0.0};
    if (tt != 0.0) {
        const double omega = st / tt;
        BICG_LOOP(n) {
            double sv[kE], tv[kE], qv[kE], xv[kE], ov[kE];
#pragma unroll
            for (int e = 0; e < kE; ++e) {
                const int64_t i = b0 + e * 256 + threadIdx.x, j = i < n ? i : 0;
                sv[e] = s[j];
                tv[e] = t[j];
                qv[e] = (double)q[j];
                xv[e] = x[j];
                ov[e] = r0[j];
            }
#pragma unroll
            for (int e = 0; e < kE; ++e) {
                const int64_t i = b0 + e * 256 + threadIdx.x;
                if (i >= n) continue;
                x[i] = 1.0 * xv[e] + omega * qv[e];
                const double rv = 1.0 * sv[e] + (-omega) * tv[e];
                r[i] = rv;
                acc[0] += rv * rv;
                acc[1] += ov[e] * rv;
            }
        }
    }
    partials<2>(acc, part);
}

// out[m] = sum of part[m * np .. m * np + np - 1], one workgroup per m, in a
// fixed order
__global__ __launch_bounds__(1024) void k_sum_arrays(int np, const double* __restrict__ part, double* __restrict__ out) {
    part += (int64_t)blockIdx.x * np;
    double s = 0.0;
    int i = threadIdx.x;
    for (; i + 3 * 1024 < np; i += 4 * 1024) {
        const double a = part[i], b = part[i + 1024], c = part[i + 2048], d = part[i + 3072];
        s = (((s + a) + b) + c) + d;
    }
    for (; i < np; i += 1024) s += part[i];
    __shared__ double sh[16];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0;
        for (int w = 0; w < 16; ++w) r += sh[w];
        out[blockIdx.x] = r;
    }
}

// through a row numbering: out[i] = map[in[i]], -1 stays
__global__ __launch_bounds__(256) void k_renumber(int64_t n, const int32_t* __restrict__ in,
                                                  const int32_t* __restrict__ map, int32_t* __restrict__ out) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= n) return;
    const int32_t k = in[i];
    out[i] = k < 0 ? -1 : map[k];
}

}  // namespace

template <typename T>
int bicg_p(int64_t n, bool first, double beta, double omega, const double* r, double* p, const double* v, double* r0,
           T* sd, T* sc, hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_bicg_p<T>, dim3(grid_of(n)), dim3(256), 0, st, n, first ? 1 : 0, beta, omega, r, p, v, r0, sd,
                       sc);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <typename T>
int bicg_s(int64_t n, double rho, const double* vr0, const double* r, const double* v, const T* q, double* s,
           double* x, double* part, double* ss_out, T* sd, T* sc, hipStream_t st) {
    const unsigned g = grid_of(n);
    hipLaunchKernelGGL(k_bicg_s<T>, dim3(g), dim3(256), 0, st, n, rho, vr0, r, v, q, s, x, part, sd, sc);
    hipLaunchKernelGGL(k_sum_arrays, dim3(1), dim3(1024), 0, st, (int)g, part, ss_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <typename T>
int bicg_r(int64_t n, const double* st_tt, const double* s, const double* t, const T* q, const double* r0, double* r,
           double* x, double* part, double* rr_r0r_out, hipStream_t st) {
    const unsigned g = grid_of(n);
    hipLaunchKernelGGL(k_bicg_r<T>, dim3(g), dim3(256), 0, st, n, st_tt, s, t, q, r0, r, x, part);
    hipLaunchKernelGGL(k_sum_arrays, dim3(2), dim3(1024), 0, st, (int)g, part, rr_r0r_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
#define BICG_INST(T)                                                                                                   \
    template int bicg_p<T>(int64_t, bool, double, double, const double*, double*, const double*, double*, T*, T*,     \
                           hipStream_t);                                                                              \
    template int bicg_s<T>(int64_t, double, const double*, const double*, const double*, const T*, double*, double*,  \
                           double*, double*, T*, T*, hipStream_t);                                                    \
    template int bicg_r<T>(int64_t, const double*, const double*, const double*, const T*, const double*, double*,    \
                           double*, double*, double*, hipStream_t);
BICG_INST(float)
BICG_INST(double)

int sum_arrays(int count, int np, const double* part, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_sum_arrays, dim3(count), dim3(1024), 0, st, np, part, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int renumber(int64_t n, const int32_t* in, const int32_t* map, int32_t* out, hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_renumber, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, in, map, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugamd
