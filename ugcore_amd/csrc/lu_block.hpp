// The base-level solve with the LU factors of the dense base matrix (FP64),
// shared by the kernels that end a multigrid cycle's descent.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace ugamd {
namespace {

// x = U^{-1} L^{-1} P b by one workgroup; Linv, Uinv: the triangular inverses,
// row-major; sh: 2n doubles. Barriers inside, so the whole workgroup calls it;
// x is written behind the last one.
template <typename TV>
__device__ __forceinline__ void lu_solve_block(int n, const double* __restrict__ Linv, const double* __restrict__ Uinv,
                                               const int32_t* __restrict__ perm, const TV* __restrict__ b,
                                               TV* __restrict__ x, double* sh) {
    // Linv, Uinv row-major; 8 lanes per row, partial sums combined by shuffles
    // (the sum of a row does not depend on the workgroup size)
    double* pb = sh;        // permuted rhs
    double* t = sh + n;     // L^{-1} P b
    for (int i = threadIdx.x; i < n; i += blockDim.x) pb[i] = (double)b[perm[i]];
    __syncthreads();
    const int g = threadIdx.x & 7, rows = blockDim.x >> 3;
    for (int i = threadIdx.x >> 3; i < n; i += rows) {
        double s = 0.0;
#pragma unroll 8
        for (int k = g; k <= i; k += 8) s += Linv[(int64_t)i * n + k] * pb[k];
        s += __shfl_xor(s, 1, 8);
        s += __shfl_xor(s, 2, 8);
        s += __shfl_xor(s, 4, 8);
        if (g == 0) t[i] = s;
    }
    __syncthreads();
    for (int i = threadIdx.x >> 3; i < n; i += rows) {
        double s = 0.0;
#pragma unroll 8
        for (int k = i + g; k < n; k += 8) s += Uinv[(int64_t)i * n + k] * t[k];
        s += __shfl_xor(s, 1, 8);
        s += __shfl_xor(s, 2, 8);
        s += __shfl_xor(s, 4, 8);
        if (g == 0) x[i] = (TV)s;
    }
}

}  // namespace
}  // namespace ugamd
