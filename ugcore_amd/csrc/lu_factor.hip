// The LU factors of the multigrid's base matrix (no_lapack/lu_decomp.h:47-200,
// FP64, partial pivoting) as the triangular inverses and the row permutation
// that the base solve applies, on the device.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "ugx_internal.hpp"

namespace ugamd {

namespace {

struct BaseOffsets {
    int32_t o[27];
};

// a thread's 8 x 8 entries, the 16 x 16 threads' stride
constexpr int kR = 8, kT = 16;

// the largest of 64 lanes' values in every lane (row shifts, then the rows'
// last lanes broadcast onwards: lane 63 holds it)
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#define UGX_MAX_STEP(ctrl, rows)                                                                          \
    {                                                                                                     \
        const uint32_t t = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, true);       \
        v = t > v ? t : v;                                                                                \
    }
    UGX_MAX_STEP(0x111, 0xf)   // row_shr:1
    UGX_MAX_STEP(0x112, 0xf)   // row_shr:2
    UGX_MAX_STEP(0x114, 0xf)   // row_shr:4
    UGX_MAX_STEP(0x118, 0xf)   // row_shr:8
    UGX_MAX_STEP(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
    UGX_MAX_STEP(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef UGX_MAX_STEP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The base operator in tiled DIA form, up to kLuDeviceMax rows, one workgroup:
// thread (ti, tj) of 16 x 16 keeps the entries (ti + 16 a, tj + 16 b) in registers
// from the first step to the last. Rows stay where they are; the position of a
// row is what the row swaps of the sequential algorithm would have made it, so
// pivots (largest magnitude, lowest position of equal ones; a NaN only where it
// already stands) and permutation are the same.
// Forward step k: the rows not yet taken lose l_i times the pivot row, in all
// columns: right of k that eliminates, left of k, where the eliminated entries
// were, it builds L^-1 in place (its column k starts as -l_i). Backward step k:
// row k of U^-1 is what is left of that row divided by its diagonal entry, and the
// rows above lose it times their column k, in place in the upper triangle.
// A chain of 2 m steps, each bound by its barriers, the pivot search and the
// issue of its instructions, so few waves (four, one a SIMD; with sixteen, which
// repeat the search, 490 us) and blocks of 16 columns unrolled, which makes a
// thread's register for a column a constant. 125 rows: 270 us on one MI355X; the
// host took 650 us, with the device idle and a copy in each direction.
__global__ __launch_bounds__(256) void k_lu_factors(int m, int nd, BaseOffsets off, const double* __restrict__ A,
                                                    double* __restrict__ linv, double* __restrict__ uinv,
                                                    int32_t* __restrict__ perm, int* __restrict__ singular) {
    extern __shared__ double dense[];   // m x m
    __shared__ double col[2][128], row[2][128], mul[128], diag[128], inv[128];
    __shared__ int32_t at[128], ord[128];   // row at a position, position of a row
    const int tid = threadIdx.x, ti = tid >> 4, tj = tid & 15, lane = tid & 63;
    for (int e = tid; e < m * m; e += 256) dense[e] = 0.0;
    __syncthreads();
    if (tid < m) {
        double v[27];
#pragma unroll
        for (int d = 0; d < 27; ++d) v[d] = d < nd ? A[dia_tiled_index(d, tid, nd)] : 0.0;
#pragma unroll
        for (int d = 0; d < 27; ++d) {
            const int c = tid + (d < nd ? off.o[d] : 0);
            if (d < nd && c >= 0 && c < m) dense[tid * m + c] += v[d];
        }
    }
    __syncthreads();
    double r[kR][kR];
#pragma unroll
    for (int a = 0; a < kR; ++a)
#pragma unroll
        for (int b = 0; b < kR; ++b) {
            const int i = ti + kT * a, c = tj + kT * b;
            r[a][b] = i < m && c < m ? dense[i * m + c] : 0.0;
        }
    // every wave keeps the positions of rows lane and lane + 64
    int p0 = lane < m ? lane : -1, p1 = lane + 64 < m ? lane + 64 : -1;
    bool bad = false;
    auto forward = [&](auto block) __attribute__((always_inline)) {
        constexpr int bk = decltype(block)::value;
#pragma unroll 1
        for (int jk = 0; jk < kT; ++jk) {
            const int k = kT * bk + jk;
            if (k >= m) break;
            if (tj == jk)
#pragma unroll
                for (int a = 0; a < kR; ++a) col[0][ti + kT * a] = r[a][bk];
            __syncthreads();
            const double c0 = col[0][lane], c1 = col[0][lane + 64];
            auto key = [&](double c, int p) -> unsigned long long {
                const unsigned long long v = (unsigned long long)__double_as_longlong(fabs(c)) + 1ull;
                const unsigned long long n = c != c ? (p == k ? 0x7ff0000000000002ull : 1ull) : v;
                return p < k ? 0ull : n;   // taken, or no row
            };
            const unsigned long long k0 = key(c0, p0), k1 = key(c1, p1);
            const bool second = k1 > k0 || (k1 == k0 && p1 >= k && p1 < p0);
            const unsigned long long best = second ? k1 : k0;
            const int bpos = second ? p1 : p0;
            const uint32_t hi = (uint32_t)(best >> 32), lw = (uint32_t)best;
            const uint32_t mhi = wave_max(hi);
            bool cand = hi == mhi;
            unsigned long long who = __ballot(cand);
            if (who & (who - 1)) {
                const uint32_t mlo = wave_max(cand ? lw : 0u);
                cand = cand && lw == mlo;
                who = __ballot(cand);
                if (who & (who - 1)) {   // equal magnitudes: the lowest position
                    const uint32_t mp = wave_max(cand ? 255u - (uint32_t)bpos : 0u);
                    who = __ballot(cand && 255u - (uint32_t)bpos == mp);
                }
            }
            const int src = __ffsll(who) - 1;
            const int q = __builtin_amdgcn_readlane(bpos, src);
            const int p = __builtin_amdgcn_readlane(second ? lane + 64 : lane, src);
            // the row at position k and the pivot change places
            p0 = lane == p ? k : p0 == k ? q : p0;
            p1 = lane + 64 == p ? k : p1 == k ? q : p1;
            const long long pb = __double_as_longlong(second ? c1 : c0);
            const double piv = __longlong_as_double(
                (long long)(uint32_t)__builtin_amdgcn_readlane((int)pb, src) |
                (long long)__builtin_amdgcn_readlane((int)(pb >> 32), src) << 32);
            bad = bad || fabs(piv) < 1e-10;
            if (tid < 64) {
                mul[lane] = p0 > k ? c0 / piv : 0.0;
                ord[lane] = p0;
            } else if (tid < 128) {
                mul[lane + 64] = p1 > k ? c1 / piv : 0.0;
                ord[lane + 64] = p1;
            }
            if (tid == 0) at[k] = p;
#pragma unroll
            for (int a = 0; a < kR; ++a)
                if ((p >> 4) == a && ti == (p & 15))
#pragma unroll
                    for (int b = 0; b < kR; ++b) row[0][tj + kT * b] = r[a][b];
            __syncthreads();
            double u[kR];
#pragma unroll
            for (int b = 0; b < kR; ++b) u[b] = row[0][tj + kT * b];
            // rows already taken have l = 0 and stay; so does column k of a row
            // with l = 0, which is zero there or taken
#pragma unroll
            for (int a = 0; a < kR; ++a) {
                const double l = mul[ti + kT * a];
                const double keep = r[a][bk];
#pragma unroll
                for (int b = 0; b < kR; ++b) r[a][b] = fma(-l, u[b], r[a][b]);
                if (tj == jk) r[a][bk] = l != 0.0 ? -l : keep;
            }
        }
    };
    forward(std::integral_constant<int, 0>());
    forward(std::integral_constant<int, 1>());
    forward(std::integral_constant<int, 2>());
    forward(std::integral_constant<int, 3>());
    forward(std::integral_constant<int, 4>());
    forward(std::integral_constant<int, 5>());
    forward(std::integral_constant<int, 6>());
    forward(std::integral_constant<int, 7>());
    if (bad) {   // the same in every wave
        if (tid == 0) *singular = 1;
        return;
    }
    // the diagonal entries and their inverses; a row's position (beyond all for
    // none)
    int pos[kR];
#pragma unroll
    for (int a = 0; a < kR; ++a) {
        const int i = ti + kT * a;
        pos[a] = i < m ? ord[i] : 255;
#pragma unroll
        for (int b = 0; b < kR; ++b)
            if (i < m && tj + kT * b == pos[a]) {
                diag[pos[a]] = r[a][b];
                inv[pos[a]] = 1.0 / r[a][b];
            }
    }
    __syncthreads();
    auto backward = [&](auto block) __attribute__((always_inline)) {
        constexpr int bk = decltype(block)::value;
#pragma unroll 1
        for (int jk = kT - 1; jk >= 0; --jk) {
            const int k = kT * bk + jk, s = jk & 1;
            if (k >= m) continue;
            const int p = __builtin_amdgcn_readfirstlane(at[k]);
            // the rows above, zero for the others
            if (tj == jk)
#pragma unroll
                for (int a = 0; a < kR; ++a) col[s][ti + kT * a] = pos[a] < k ? r[a][bk] : 0.0;
#pragma unroll
            for (int a = 0; a < kR; ++a)
                if ((p >> 4) == a && ti == (p & 15)) {
                    // divided by the diagonal entry: its inverse and one correction
                    const double u = diag[k], v = inv[k];
#pragma unroll
                    for (int b = bk; b < kR; ++b) {
                        const int c = tj + kT * b;
                        const double t = r[a][b] * v;
                        const double x = c == k ? v : fma(fma(-t, u, r[a][b]), v, t);
                        r[a][b] = c >= k ? x : r[a][b];
                        row[s][c] = c >= k ? x : 0.0;
                    }
                }
            __syncthreads();
            double x[kR];
#pragma unroll
            for (int b = bk; b < kR; ++b) x[b] = row[s][tj + kT * b];
#pragma unroll
            for (int a = 0; a < kR; ++a) {
                const double u = col[s][ti + kT * a], keep = r[a][bk];
#pragma unroll
                for (int b = bk; b < kR; ++b) r[a][b] = fma(-u, x[b], r[a][b]);
                if (tj == jk) r[a][bk] = u != 0.0 ? -(u * x[bk]) : keep;
            }
        }
    };
    backward(std::integral_constant<int, 7>());
    backward(std::integral_constant<int, 6>());
    backward(std::integral_constant<int, 5>());
    backward(std::integral_constant<int, 4>());
    backward(std::integral_constant<int, 3>());
    backward(std::integral_constant<int, 2>());
    backward(std::integral_constant<int, 1>());
    backward(std::integral_constant<int, 0>());
#pragma unroll
    for (int a = 0; a < kR; ++a)
#pragma unroll
        for (int b = 0; b < kR; ++b) {
            const int i = ti + kT * a, c = tj + kT * b;
            if (i >= m || c >= m) continue;
            const int o = pos[a];
            linv[o * m + c] = c < o ? r[a][b] : c == o ? 1.0 : 0.0;
            uinv[o * m + c] = c >= o ? r[a][b] : 0.0;
        }
    if (tid < m) perm[tid] = at[tid];
}

}  // namespace

bool lu_factors_fit(int m, int nd) { return m <= kLuDeviceMax && nd <= 27; }

int lu_factors(int m, int nd, const int32_t* off, const double* A, double* linv, double* uinv, int32_t* perm,
               int* singular, hipStream_t s) {
    if (m <= 0 || !lu_factors_fit(m, nd)) return -1;
    BaseOffsets o{};
    for (int d = 0; d < nd; ++d) o.o[d] = off[d];
    hipLaunchKernelGGL(k_lu_factors, dim3(1), dim3(256), sizeof(double) * (size_t)m * m, s, m, nd, o, A, linv, uinv,
                       perm, singular);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugamd
