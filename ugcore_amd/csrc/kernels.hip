// HIP kernels for gfx950 (MI355X) behind the ugx_* C ABI.
//
// Roles (reference files they replace or restate):
//  * CSR SpMV          SparseMatrix::axpy / apply_ignore_zero_rows
//                      (lib_algebra/cpu_algebra/sparsematrix_impl.h:271-339)
//  * vector ops        VecScaleAdd 2/3-term, set, scale (lib_algebra/common/operations_vec.h:55-63,162-202)
//  * reductions        Vector::dotprod / norm (cpu_algebra/vector_impl.h:70-79, 323-329)
//  * Jacobi            jacobi.h:155-249 (diagInv = 1/(a_ii/omega), c = diagInv*d)
//  * level operators   AssembledMultiGridCycle smoothing/transfer stages
//                      (lib_disc/operator/linear_operator/multi_grid_solver/mg_solver_impl.hpp:1686-1964)
//                      on diagonal-offset (DIA) level matrices in lattice order
//  * transfer          StdTransfer P1 prolongation/restriction with Dirichlet
//                      adjustment (std_transfer_impl.h:45-168, lagrange_dirichlet_boundary_impl.h:485-740)
//  * assembly          Q1 FE hexahedra / FV1 triangles, colour-ordered scatter
//
// All kernels are stream ordered; none allocates. Wavefront size is 64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <utility>
#include <vector>

#include <cstdint>

#include "elem_local.hpp"
#include "lu_block.hpp"
#include "ugx_internal.hpp"

namespace ugamd {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

// Blocks are dispatched round-robin over the 8 XCDs; remap so that each XCD
// walks one contiguous range of logical blocks (its L2 then sees neighbouring
// rows, which share x-vector lines).
__device__ __forceinline__ int64_t xcd_block(int64_t nblocks) {
    const int64_t b = blockIdx.x;
    if (nblocks < 64) return b;
    const int64_t per = (nblocks + 7) / 8;
    const int64_t xcd = b % 8, slot = b / 8;
    const int64_t lb = xcd * per + slot;
    return lb;   // may exceed nblocks-1 for the last XCD: callers bound-check rows
}

// Division by a run-time constant d >= 1 of 32-bit unsigned n (round-up
// multiplier method, Granlund & Montgomery 1994): q = (umulhi(n, m) + n) >> s
// with s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1.
struct FastDiv {
    uint32_t d, m, s;
};
static inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f{d, 0u, 0u};
    if (d <= 1) return f;
    uint32_t s = 0;
    while ((1ull << s) < d) ++s;
    f.s = s;
    f.m = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1);
    return f;
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) {
    return (uint32_t)(((uint64_t)__umulhi(n, f.m) + n) >> f.s);
}

// Row schedule of the lattice (DIA) kernels. Flat mode: 256 consecutive rows
// per block, blocks remapped by xcd_block. Banded mode (3D lattices): the W
// lines of every plane are split into 8 bands, XCD c (blockIdx % 8) owns band
// c of every plane and walks its blocks plane by plane, so the rows one plane
// below (offsets -W^2 +- W +- 1, whose coefficients and vector entries a row
// reads again) were streamed through the same L2 one band-plane earlier.
struct RowMap {
    int64_t nblocks;   // flat mode: logical blocks
    int64_t plane;     // banded mode: rows per plane (0 = flat mode)
    int64_t nplanes;
    int32_t lo[8];     // first row of band c within a plane
    int32_t len[8];    // rows of band c within a plane
    int32_t cps[8];    // 256-row chunks of band c per plane
};

// first row of this thread and the end of its block's row range; false when
// the block has no rows
__device__ __forceinline__ bool map_row(const RowMap& m, int64_t n, int64_t& i) {
    if (m.plane == 0) {
        const int64_t lb = xcd_block(m.nblocks);
        i = lb * 256 + threadIdx.x;
        return lb < m.nblocks && i < n;
    }
    const int c = blockIdx.x & 7;
    const int64_t q = blockIdx.x >> 3;
    const int64_t cps = m.cps[c];
    const int64_t k = q / cps;
    if (k >= m.nplanes) return false;
    const int64_t ch = q - k * cps;
    const int64_t r = ch * 256 + threadIdx.x;
    i = k * m.plane + m.lo[c] + r;
    return r < m.len[c];
}

// Level operators are stored as ND diagonals in wavefront tiles: the 64
// values of diagonal d for rows 64t..64t+63 are contiguous, and the ND
// diagonals of one tile follow each other, so a wavefront streams one
// contiguous ND*64*sizeof(T) block.

template <typename T>
__device__ __forceinline__ T wave_sum_group(T v, int G) {
    for (int off = G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// ---------------------------------------------------------------------------
// CSR SpMV: dest = alpha*v1 + beta*A*w   (mode 0)
//           dest = beta*A*w on non-empty rows only (mode 1, apply_ignore_zero_rows)
// G lanes cooperate on one row; rowptr/col are int32.
// ---------------------------------------------------------------------------
template <typename TM, typename TV, int G>
__global__ __launch_bounds__(256) void k_spmv_csr(int64_t nrows, const int32_t* __restrict__ rowptr,
                                                  const int32_t* __restrict__ col, const TM* __restrict__ val,
                                                  double alpha, const TV* v1, double beta,
                                                  const TV* __restrict__ w, TV* dest, int mode,
                                                  int64_t nblocks) {
    const int64_t lb = xcd_block(nblocks);
    const int lane = threadIdx.x % G;
    const int64_t row = (lb * 256 + threadIdx.x) / G;
    const bool active = (lb < nblocks) && (row < nrows);
    double s = 0.0;
    int32_t rb = 0, re = 0;
    if (active) {
        rb = rowptr[row];
        re = rowptr[row + 1];
        // two independent (column, value) pairs in flight per lane; the matrix
        // streams are read once, so they bypass the cache (non-temporal)
        for (int32_t k = rb + lane; k < re; k += 2 * G) {
            const int32_t k1 = k + G;
            const int32_t c0 = __builtin_nontemporal_load(col + k);
            const double a0 = (double)__builtin_nontemporal_load(val + k);
            int32_t c1 = c0;
            double a1 = 0.0;
            if (k1 < re) {
                c1 = __builtin_nontemporal_load(col + k1);
                a1 = (double)__builtin_nontemporal_load(val + k1);
            }
            s += a0 * (double)w[c0] + a1 * (double)w[c1];
        }
    }
    s = wave_sum_group(s, G);
    if (active && lane == 0) {
        if (mode == 1) {
            if (re > rb) dest[row] = (TV)(beta * s);
        } else {
            const double base = (alpha == 0.0) ? 0.0 : alpha * (double)v1[row];
            dest[row] = (TV)(base + beta * s);
        }
    }
}

template <typename TM, typename TV>
static int launch_spmv_csr(int64_t nrows, const int32_t* rowptr, const int32_t* col, const TM* val,
                           double alpha, const TV* v1, double beta, const TV* w, TV* dest, int mode,
                           int lanes, hipStream_t s) {
    if (nrows <= 0) return 0;
    int G = lanes;
    if (G != 4 && G != 8 && G != 16 && G != 32 && G != 64) G = 8;
    const int64_t rows_per_block = 256 / G;
    const int64_t nblocks = (nrows + rows_per_block - 1) / rows_per_block;
    const int64_t grid = nblocks < 64 ? nblocks : ((nblocks + 7) / 8) * 8;
    switch (G) {
        case 4: hipLaunchKernelGGL((k_spmv_csr<TM, TV, 4>), dim3(grid), dim3(256), 0, s, nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, nblocks); break;
        case 8: hipLaunchKernelGGL((k_spmv_csr<TM, TV, 8>), dim3(grid), dim3(256), 0, s, nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, nblocks); break;
        case 16: hipLaunchKernelGGL((k_spmv_csr<TM, TV, 16>), dim3(grid), dim3(256), 0, s, nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, nblocks); break;
        case 32: hipLaunchKernelGGL((k_spmv_csr<TM, TV, 32>), dim3(grid), dim3(256), 0, s, nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, nblocks); break;
        default: hipLaunchKernelGGL((k_spmv_csr<TM, TV, 64>), dim3(grid), dim3(256), 0, s, nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, nblocks); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------
// Sliced ELL (64-row slices): the SpMV layout of GPUSparseMatrix. Slice
// position p = 64t + lane holds row order[p] (row p without an order); entry k
// of that row is stored at slice_ptr[t] + 64*k + lane (columns int32, values
// TM). Rows shorter than the slice width are padded with value 0 and a valid
// column, so every lane runs the same trip count and every load is one
// coalesced 64-lane access. The order (a permutation of the rows, e.g. the
// lattice walk of the assembling discretization) only decides which rows share
// a slice: it keeps the column gathers of neighbouring lanes close in memory;
// each row's entries and summation order are unchanged.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int64_t sell_row(const int32_t* order, int64_t p) { return order ? order[p] : p; }

__global__ void k_sell_widths(int64_t nrows, const int32_t* __restrict__ rowptr, const int32_t* __restrict__ order,
                              int32_t* __restrict__ width) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t nslices = (nrows + 63) / 64;
    if (t >= nslices) return;
    int32_t w = 0;
    const int64_t p1 = (t + 1) * 64 < nrows ? (t + 1) * 64 : nrows;
    for (int64_t p = t * 64; p < p1; ++p) {
        const int64_t r = sell_row(order, p);
        const int32_t len = rowptr[r + 1] - rowptr[r];
        w = len > w ? len : w;
    }
    width[t] = w;
}

// one wavefront per slice: the slice's entries move through LDS in chunks of
// 8 per row, read row by row (contiguous CSR runs) and written column by
// column (contiguous 64-entry runs of the slice block); padding: the row's own
// index as column (0 beyond the columns), value 0. vals_only: the columns are
// already in place (same pattern), only the values are rewritten
template <typename TM>
__global__ __launch_bounds__(64) void k_sell_fill(int64_t nrows, int64_t ncols, const int32_t* __restrict__ rowptr,
                                                  const int32_t* __restrict__ col, const TM* __restrict__ val,
                                                  const int32_t* __restrict__ order, const int64_t* __restrict__ slice_ptr,
                                                  const int32_t* __restrict__ width, int32_t* __restrict__ scol,
                                                  TM* __restrict__ sval, int vals_only) {
    constexpr int C = 8;
    __shared__ int32_t rbs[64], lens[64];
    __shared__ int32_t ct[C * 64];
    __shared__ TM vt[C * 64];
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const int64_t p = t * 64 + lane;
    const int64_t r = p < nrows ? sell_row(order, p) : p;
    rbs[lane] = r < nrows ? rowptr[r] : 0;
    lens[lane] = r < nrows ? rowptr[r + 1] - rowptr[r] : 0;
    const int32_t pad_col = (int32_t)(r < ncols ? r : 0);
    const int32_t w = width[t];
    const int64_t base = slice_ptr[t] + lane;
    __syncthreads();
    for (int k0 = 0; k0 < w; k0 += C) {
#pragma unroll
        for (int it = 0; it < C; ++it) {
            const int e = it * 64 + lane;
            const int j = e / C, kk = e % C, k = k0 + kk;
            int32_t c = -1;
            TM v = (TM)0;
            if (k < lens[j]) {
                const int64_t a = (int64_t)rbs[j] + k;
                v = val[a];
                if (!vals_only) c = col[a];
            }
            const int slot = kk * 64 + ((j + 8 * kk) & 63);   // rotated: fewer bank conflicts
            ct[slot] = c;
            vt[slot] = v;
        }
        __syncthreads();
        const int kc = w - k0 < C ? w - k0 : C;
        for (int kk = 0; kk < kc; ++kk) {
            const int slot = kk * 64 + ((lane + 8 * kk) & 63);
            const int64_t o = base + (int64_t)64 * (k0 + kk);
            if (!vals_only) {
                const int32_t c = ct[slot];
                scol[o] = c >= 0 ? c : pad_col;
            }
            sval[o] = vt[slot];
        }
        __syncthreads();
    }
}

// The row sums of a sliced-ELL matrix and what a product does with them.
// Each of a slice's 64 rows belongs to one lane; WAVES wavefronts share a
// slice, each summing every WAVES-th entry, combined through LDS in a fixed
// order. WAVES 1 (four slices a workgroup) streams the matrices of many short
// rows: 400,003 rows of about 16 entries, 57 us, bound by the gathers. Where rows
// are wide and few (Q2 operators and transfers: up to 125 entries, 1 - 560
// slices), one lane's chain of loads and gathers is the time: 20 - 30 us
// whatever the size with one wave, 6.3 - 14.9 us with four or sixteen (one
// MI355X, 729 - 35,937 rows). sell_waves() draws the line.
constexpr int sell_block(int waves) { return waves == 1 ? 256 : 64 * waves; }

template <typename TM, typename TV, int WAVES>
__device__ __forceinline__ bool sell_row_sum(int64_t nrows, const int64_t* __restrict__ slice_ptr,
                                             const int32_t* __restrict__ width, const int32_t* __restrict__ scol,
                                             const TM* __restrict__ sval, const TV* __restrict__ w,
                                             const int32_t* __restrict__ order, int64_t nblocks, int64_t& r,
                                             double& sum) {
    const int64_t lb = xcd_block(nblocks);
    if (lb >= nblocks) return false;   // the whole workgroup
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t = WAVES == 1 ? lb * 4 + wave : lb;
    const int64_t nslices = (nrows + 63) / 64;
    if (WAVES == 1 && t >= nslices) return false;
    const int64_t p = t * 64 + lane;
    const int32_t wd = width[t];
    const int32_t* cp = scol + slice_ptr[t] + lane;
    const TM* vp = sval + slice_ptr[t] + lane;
    double s0 = 0.0, s1 = 0.0;
    if (WAVES == 1) {
        int32_t k = 0;
        for (; k + 4 <= wd; k += 4) {
            int32_t c[4];
            double a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) c[u] = __builtin_nontemporal_load(cp + 64 * (k + u));
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = (double)__builtin_nontemporal_load(vp + 64 * (k + u));
#pragma unroll
            for (int u = 0; u < 4; u += 2) {
                s0 = fma(a[u], (double)w[c[u]], s0);
                s1 = fma(a[u + 1], (double)w[c[u + 1]], s1);
            }
        }
        for (; k < wd; ++k) {
            const int32_t c0 = __builtin_nontemporal_load(cp + 64 * k);
            const double a0 = (double)__builtin_nontemporal_load(vp + 64 * k);
            s0 = fma(a0, (double)w[c0], s0);
        }
    } else {
        // entries wave, wave + WAVES, ...: which sum an entry goes to depends on
        // its place in the row alone, not on the width of the slice. The last
        // round loads the slice's last entry for the ones it lacks.
        for (int32_t k0 = wave; k0 < wd; k0 += 8 * WAVES) {
            int32_t c[8];
            double a[8], x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int32_t k = k0 + u * WAVES < wd ? k0 + u * WAVES : wd - 1;
                c[u] = __builtin_nontemporal_load(cp + 64 * k);
                a[u] = (double)__builtin_nontemporal_load(vp + 64 * k);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = (double)w[c[u]];
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                const double t0 = fma(a[u], x[u], s0), t1 = fma(a[u + 1], x[u + 1], s1);
                s0 = k0 + u * WAVES < wd ? t0 : s0;
                s1 = k0 + (u + 1) * WAVES < wd ? t1 : s1;
            }
        }
    }
    sum = s0 + s1;
    if (WAVES > 1) {
        __shared__ double sh[WAVES][64];
        sh[wave][lane] = sum;
        __syncthreads();
        if (wave != 0) return false;
        sum = sh[0][lane];
#pragma unroll
        for (int u = 1; u < WAVES; ++u) sum += sh[u][lane];
    }
    if (p >= nrows) return false;
    r = sell_row(order, p);
    return true;
}

// dest = alpha*v1 + beta*A*w (mode 0) or dest = beta*A*w on rows with entries
// (mode 1, needs rowptr)
template <typename TM, typename TV, int WAVES>
__global__ __launch_bounds__(sell_block(WAVES)) void k_sell_spmv(int64_t nrows, const int64_t* __restrict__ slice_ptr,
                                                   const int32_t* __restrict__ width, const int32_t* __restrict__ scol,
                                                   const TM* __restrict__ sval, double alpha, const TV* v1, double beta,
                                                   const TV* __restrict__ w, TV* dest, int mode,
                                                   const int32_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ order, int64_t nblocks) {
    int64_t r;
    double sum;
    if (!sell_row_sum<TM, TV, WAVES>(nrows, slice_ptr, width, scol, sval, w, order, nblocks, r, sum)) return;
    if (mode == 1) {
        if (rowptr[r + 1] > rowptr[r]) dest[r] = (TV)(beta * sum);
    } else {
        const double base = (alpha == 0.0) ? 0.0 : alpha * (double)v1[r];
        dest[r] = (TV)(base + beta * sum);
    }
}

// a product of the multigrid cycle over matrices with the row operations that
// follow it (SellEpilogue)
template <int WAVES>
__global__ __launch_bounds__(sell_block(WAVES)) void k_sell_cycle(int64_t nrows, const int64_t* __restrict__ slice_ptr,
                                                    const int32_t* __restrict__ width, const int32_t* __restrict__ scol,
                                                    const double* __restrict__ sval, const double* __restrict__ w,
                                                    const int32_t* __restrict__ rowptr,
                                                    const int32_t* __restrict__ order, int64_t nblocks,
                                                    SellEpilogue e) {
    int64_t r;
    double v;
    if (!sell_row_sum<double, double, WAVES>(nrows, slice_ptr, width, scol, sval, w, order, nblocks, r, v)) return;
    const double d = e.dinv ? e.dinv[r] : 0.0, c = e.sc && !e.sc_set ? e.sc[r] : 0.0;   // in flight together
    if (e.sub) v = 1.0 * e.sub[r] + -1.0 * v;
    else if (e.keep_empty && rowptr[r + 1] == rowptr[r]) v = e.out[r];
    if (e.out) e.out[r] = v;
    if (e.dinv) {
        v = d * v;
        e.st[r] = v;
    }
    if (e.sc) e.sc[r] = e.sc_set ? v : 1.0 * c + 1.0 * v;
}

// ---------------------------------------------------------------------------
// vector kernels (grid-stride)
// ---------------------------------------------------------------------------
static inline int64_t vec_grid(int64_t n) {
    int64_t g = (n + 255) / 256;
    if (g > 16384) g = 16384;
    if (g < 1) g = 1;
    return g;
}

// Streaming vector kernels: a block covers kStreamE * 256 consecutive
// elements per pass (thread t takes b0 + t and b0 + 256 + t), the grid covers
// the whole vector (grid-stride only beyond 2^20 blocks), all loads of a pass
// are issued before its stores, and every access is nontemporal (each element
// is touched once). On one MI355X, for 257^3 vectors with cold caches, this
// runs 25-30 % faster than a 16K-block grid-stride loop with plain accesses.
// Lanes past the end load element 0 and store nothing.
constexpr int kStreamE = 2;
static inline int64_t stream_grid(int64_t n) {
    int64_t g = (n + 256 * kStreamE - 1) / (256 * kStreamE);
    if (g > ((int64_t)1 << 20)) g = (int64_t)1 << 20;
    if (g < 1) g = 1;
    return g;
}
template <typename T>
__device__ __forceinline__ T ldnt(const T* p) { return __builtin_nontemporal_load(p); }
template <typename T>
__device__ __forceinline__ void stnt(T v, T* p) { __builtin_nontemporal_store(v, p); }
#define UGX_STREAM_LOOP(n)                                                                  \
    for (int64_t b0_ = blockIdx.x * (int64_t)(256 * kStreamE); b0_ < (n);                  \
         b0_ += (int64_t)gridDim.x * (256 * kStreamE))
#define UGX_STREAM_IDX(e) (b0_ + (e) * 256 + (int64_t)threadIdx.x)
#define UGX_STREAM_SAFE(e, n) (UGX_STREAM_IDX(e) < (n) ? UGX_STREAM_IDX(e) : (int64_t)0)

template <typename T>
__global__ __launch_bounds__(256) void k_set(int64_t n, T* x, T v) {
    UGX_STREAM_LOOP(n) {
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt(v, x + UGX_STREAM_IDX(e));
    }
}

// dest = a1*v1 + a2*v2 (+ a3*v3 when v3 != nullptr); any of them may alias
// dest (each element is read and then written by the same thread)
template <typename T>
__global__ __launch_bounds__(256) void k_scale_add(int64_t n, T* dest, double a1, const T* v1, double a2,
                                                   const T* v2, double a3, const T* v3) {
    UGX_STREAM_LOOP(n) {
        T x1[kStreamE], x2[kStreamE], x3[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            x1[e] = ldnt(v1 + i);
            x2[e] = ldnt(v2 + i);
            x3[e] = v3 ? ldnt(v3 + i) : (T)0;
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            if (UGX_STREAM_IDX(e) >= n) continue;
            double r = a1 * (double)x1[e] + a2 * (double)x2[e];
            if (v3) r += a3 * (double)x3[e];
            stnt((T)r, dest + UGX_STREAM_IDX(e));
        }
    }
}

// dest[i] = d[i] * x[i]  (Jacobi step with the damped inverse diagonal)
template <typename TD, typename TV>
__global__ __launch_bounds__(256) void k_diag_mult(int64_t n, TV* dest, const TD* d, const TV* x) {
    UGX_STREAM_LOOP(n) {
        TD dv[kStreamE];
        TV xv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            dv[e] = ldnt(d + i);
            xv[e] = ldnt(x + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt((TV)((double)dv[e] * (double)xv[e]), dest + UGX_STREAM_IDX(e));
    }
}

// dinv_i = 1 / (a_ii * (1/omega)) from a CSR matrix (Jacobi::preprocess)
template <typename TM, typename TD>
__global__ void k_jacobi_diag_csr(int64_t n, const int32_t* rowptr, const int32_t* col, const TM* val, double omega,
                                  TD* dinv, int* bad) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double d = 0.0;
        for (int32_t k = rowptr[i]; k < rowptr[i + 1]; ++k)
            if (col[k] == i) d = (double)val[k];
        double m = d;
        m *= 1.0 / omega;
        if (m == 0.0) { bad[0] = 1; dinv[i] = (TD)0; }
        else dinv[i] = (TD)(1.0 / m);
    }
}

// surface (DoF order) <-> level (lattice order) copies with precision
// conversion, written as gathers so the stores are coalesced:
//   dst_lat[l] = src_dof[dof_of_lat[l]]   and   dst_dof[i] += src_lat[lat_of_dof[i]]
// In the streaming layout above: a pass loads its kStreamE indices, then
// issues its gathers (plain loads: neighbouring points share cache lines
// that other waves read), then stores.
template <typename TS, typename TL>
__global__ __launch_bounds__(256) void k_permute_to(int64_t n, const int32_t* __restrict__ dof_of_lat,
                                                    const TS* __restrict__ src, TL* __restrict__ dst) {
    UGX_STREAM_LOOP(n) {
        int32_t k[kStreamE];
        TS v[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) k[e] = ldnt(dof_of_lat + UGX_STREAM_SAFE(e, n));
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) v[e] = src[k[e]];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt((TL)v[e], dst + UGX_STREAM_IDX(e));
    }
}
// the same into an FP64 and an FP32 lattice vector
__global__ __launch_bounds__(256) void k_permute_to_dual(int64_t n, const int32_t* __restrict__ dof_of_lat,
                                                         const double* __restrict__ src, double* __restrict__ dst,
                                                         float* __restrict__ dst32) {
    UGX_STREAM_LOOP(n) {
        int32_t k[kStreamE];
        double v[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) k[e] = ldnt(dof_of_lat + UGX_STREAM_SAFE(e, n));
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) v[e] = src[k[e]];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) {
                stnt(v[e], dst + UGX_STREAM_IDX(e));
                stnt((float)v[e], dst32 + UGX_STREAM_IDX(e));
            }
    }
}
template <typename TL, typename TS>
__global__ __launch_bounds__(256) void k_permute_from(int64_t n, const int32_t* __restrict__ lat_of_dof,
                                                      const TL* __restrict__ src, TS* __restrict__ dst) {
    UGX_STREAM_LOOP(n) {
        int32_t k[kStreamE];
        TL v[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) k[e] = ldnt(lat_of_dof + UGX_STREAM_SAFE(e, n));
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) v[e] = src[k[e]];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt((TS)v[e], dst + UGX_STREAM_IDX(e));
    }
}
// dst_dof[dof_of_lat[l]] = src_lat[l], the scatter form of k_permute_from for
// a bijective numbering: the reads are coalesced, and the writes of a wave
// fall into a few runs of consecutive DoFs (the lattice points of one line
// alternate between a handful of DoF ranges, each numbered along the line)
template <typename TL, typename TS>
__global__ __launch_bounds__(256) void k_permute_scatter(int64_t n, const int32_t* __restrict__ dof_of_lat,
                                                         const TL* __restrict__ src, TS* __restrict__ dst) {
    UGX_STREAM_LOOP(n) {
        int32_t k[kStreamE];
        TL v[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            k[e] = ldnt(dof_of_lat + UGX_STREAM_SAFE(e, n));
            v[e] = ldnt(src + UGX_STREAM_SAFE(e, n));
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) dst[k[e]] = (TS)v[e];
    }
}
template <typename TL, typename TS>
__global__ __launch_bounds__(256) void k_permute_add_from(int64_t n, const int32_t* __restrict__ lat_of_dof,
                                                          const TL* __restrict__ src, TS* __restrict__ dst) {
    UGX_STREAM_LOOP(n) {
        int32_t k[kStreamE];
        TL v[kStreamE];
        TS d[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            k[e] = ldnt(lat_of_dof + UGX_STREAM_SAFE(e, n));
            d[e] = ldnt(dst + UGX_STREAM_SAFE(e, n));
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) v[e] = src[k[e]];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt((TS)((double)d[e] + (double)v[e]), dst + UGX_STREAM_IDX(e));
    }
}

// ---------------------------------------------------------------------------
// deterministic reductions: pass 1 writes one partial per block, pass 2 sums
// the partials in a fixed order
// ---------------------------------------------------------------------------
// one partial per block of the streaming grid, at most kRedMaxBlocks
constexpr int kRedMaxBlocks = 65536;
static inline int red_grid(int64_t n) {
    int64_t g = (n + 256 * kStreamE - 1) / (256 * kStreamE);
    if (g > kRedMaxBlocks) g = kRedMaxBlocks;
    if (g < 1) g = 1;
    return (int)g;
}

__device__ __forceinline__ void block_partial(double acc, double* partial) {
    __shared__ double sh[4];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <typename T>
__global__ __launch_bounds__(256) void k_dot_partial(int64_t n, const T* __restrict__ a, const T* __restrict__ b,
                                                     double* partial) {
    double acc = 0.0;
    UGX_STREAM_LOOP(n) {
        T av[kStreamE], bv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            av[e] = ldnt(a + i);
            bv[e] = ldnt(b + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) acc += (double)av[e] * (double)bv[e];
    }
    block_partial(acc, partial);
}

// partial counts of the nonzero entries (exact in double below 2^53; unlike
// a.a, entries whose square underflows still count)
__global__ __launch_bounds__(256) void k_nonzero_partial(int64_t n, const double* __restrict__ a,
                                                         double* partial) {
    double acc = 0.0;
    UGX_STREAM_LOOP(n) {
        double av[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) av[e] = ldnt(a + UGX_STREAM_SAFE(e, n));
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n && av[e] != 0.0) acc += 1.0;
    }
    block_partial(acc, partial);
}

// one workgroup of 1024: thread t sums partial[t], partial[t + 1024], ... in
// that order (eight loads in flight), then the waves and the 16 wave sums are
// combined in a fixed order, so the result does not depend on timing
// the sum of np partials by a workgroup of 1024, in its thread 0
__device__ __forceinline__ double sum_1024(int np, const double* __restrict__ partial) {
    double s = 0.0;
    int i = threadIdx.x;
    for (; i + 7 * 1024 < np; i += 8 * 1024) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = partial[i + u * 1024];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; i < np; i += 1024) s += partial[i];
    __shared__ double sh[16];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < 16; ++w) r += sh[w];
    return r;
}
__global__ __launch_bounds__(1024) void k_sum_partials(int np, const double* partial, double* out, int sqrt_flag) {
    const double r = sum_1024(np, partial);
    if (threadIdx.x == 0) out[0] = sqrt_flag ? sqrt(r) : r;
}

// ---------------------------------------------------------------------------
// CG building blocks with the scalars kept in device memory
// (sc[0] rho of the step before, sc[1] lambda, sc[2] alpha, sc[4] rho, sc[5]
//  |r|^2, sc[6] = 1 after a breakdown lambda == 0)
// On the small lattices a step is bound by its launches, so the scalars are
// formed where they are used: lambda by every workgroup of the update from the
// operator's partial sums, beta = rho / rho_old by the direction update, and the
// kernel that sums |r|^2 keeps rho and hands the host its two values. The 33^3
// solve: 97 us a step with a kernel for each of them and a copy, 90 so.
// ---------------------------------------------------------------------------
// the sum of np partials, the same in every thread of a workgroup of 256
__device__ __forceinline__ double block_sum_partials(int np, const double* __restrict__ partial) {
    __shared__ double sh[4];
    double s = 0.0;
    for (int i = threadIdx.x; i < np; i += 256) s += partial[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// |r|^2 = sum of the partials, the breakdown flag beside it in pinned host
// memory, and rho kept for the next step
__global__ __launch_bounds__(1024) void k_cg_norm(int np, const double* __restrict__ partial, double* __restrict__ sc,
                                                  double* __restrict__ host) {
    const double s = sum_1024(np, partial);
    if (threadIdx.x == 0) {
        sc[5] = s;
        sc[0] = sc[4];
        host[0] = s;
        host[1] = sc[6];
    }
}

// alpha = rho / lambda (0, with the breakdown flag, when lambda == 0), formed
// by every thread and recorded by the first (lambda: the sum of nl partials,
// or sc[1] where nl is 0); x += alpha p ; r -= alpha q ;
// partial sums of r.r
__global__ __launch_bounds__(256) void k_cg_update(int64_t n, double* __restrict__ sc,
                                                   const double* __restrict__ p, const double* __restrict__ q,
                                                   double* __restrict__ x, double* __restrict__ r,
                                                   double* __restrict__ partial, float* __restrict__ rf, int nl,
                                                   const double* __restrict__ lpart) {
    const double lambda = nl > 0 ? block_sum_partials(nl, lpart) : sc[1];
    const double alpha = lambda == 0.0 ? 0.0 : sc[4] / lambda;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (nl > 0) sc[1] = lambda;
        sc[2] = alpha;
        if (lambda == 0.0) sc[6] = 1.0;
    }
    double acc = 0.0;
    UGX_STREAM_LOOP(n) {
        double xv[kStreamE], pv[kStreamE], rv[kStreamE], qv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            xv[e] = ldnt(x + i);
            pv[e] = ldnt(p + i);
            rv[e] = ldnt(r + i);
            qv[e] = ldnt(q + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_IDX(e);
            if (i >= n) continue;
            stnt(1.0 * xv[e] + alpha * pv[e], x + i);
            const double ri = 1.0 * rv[e] + (-alpha) * qv[e];
            stnt(ri, r + i);
            if (rf) stnt((float)ri, rf + i);   // the FP32 cycle's copy of the defect
            acc += ri * ri;
        }
    }
    block_partial(acc, partial);
}


// p = beta p + z
__global__ __launch_bounds__(256) void k_cg_direction(int64_t n, const double* __restrict__ sc, double* __restrict__ p,
                                                      const double* __restrict__ z) {
    const double beta = sc[4] / sc[0];
    UGX_STREAM_LOOP(n) {
        double pv[kStreamE], zv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            pv[e] = ldnt(p + i);
            zv[e] = ldnt(z + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt(fma(beta, pv[e], zv[e]), p + UGX_STREAM_IDX(e));
    }
}

// z = (double) c ; partial sums of z.r
template <typename T>
__global__ __launch_bounds__(256) void k_convert_dot(int64_t n, const T* __restrict__ c, double* __restrict__ z,
                                                     const double* __restrict__ r, double* __restrict__ partial) {
    double acc = 0.0;
    UGX_STREAM_LOOP(n) {
        T cv[kStreamE];
        double rv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            cv[e] = ldnt(c + i);
            rv[e] = ldnt(r + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_IDX(e);
            if (i >= n) continue;
            const double zi = (double)cv[e];
            stnt(zi, z + i);
            acc += zi * rv[e];
        }
    }
    block_partial(acc, partial);
}

// ---------------------------------------------------------------------------
// DIA level operators. Vectors carry a zero halo so x[i + off] is always in
// bounds; values of couplings that leave the lattice are stored as 0.
// ---------------------------------------------------------------------------
struct DiaOffsets {
    int32_t off[27];
};

// Accumulation type: FP32 level operators compute in FP32, FP64 in FP64.
template <typename T>
struct Acc {
    typedef T type;
};

// d_out = d_in - A*x  (x may be any vector; d_out may equal d_in). ND is the
// number of stored diagonals (27 in 3D, 9 in 2D); all loads of a row are issued
// before the multiply-adds.
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dia_apply_sub(int64_t n, DiaOffsets o, const TM* __restrict__ A,
                                                       const TV* __restrict__ x, const TV* d_in, TV* d_out,
                                                       RowMap rm) {
    typedef typename Acc<TV>::type T;
    int64_t i;
    if (!map_row(rm, n, i)) return;
    T a[ND], xv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) a[d] = (T)A[dia_tiled_index(d, i, ND)];
#pragma unroll
    for (int d = 0; d < ND; ++d) xv[d] = (T)x[i + o.off[d]];
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xv[d], s);
    d_out[i] = (TV)((T)d_in[i] - s);
}

// y = alpha*v + beta*A*x
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dia_axpy(int64_t n, DiaOffsets o, const TM* __restrict__ A,
                                                  double alpha, const TV* v, double beta, const TV* __restrict__ x,
                                                  TV* y, RowMap rm) {
    typedef typename Acc<TV>::type T;
    int64_t i;
    if (!map_row(rm, n, i)) return;
    T a[ND], xv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) a[d] = (T)A[dia_tiled_index(d, i, ND)];
#pragma unroll
    for (int d = 0; d < ND; ++d) xv[d] = (T)x[i + o.off[d]];
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xv[d], s);
    y[i] = (TV)((alpha == 0.0 ? 0.0 : alpha * (double)v[i]) + beta * (double)s);
}

// One damped-Jacobi smoothing step fused with the defect update and the
// correction update (mg_solver_impl.hpp:1702-1730 / 1917-1947):
//   st = dinv .* sd_in ;  sd_out = sd_in - A*st ;  sc += st
// sd_out must not alias sd_in (neighbours read the old defect).
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dia_jacobi_step(int64_t n, DiaOffsets o, const TM* __restrict__ A,
                                                         const TV* __restrict__ dinv, const TV* __restrict__ sd_in,
                                                         TV* __restrict__ sd_out, TV* __restrict__ sc,
                                                         RowMap rm) {
    typedef typename Acc<TV>::type T;
    int64_t i;
    if (!map_row(rm, n, i)) return;
    T a[ND], dv[ND], sv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) a[d] = (T)A[dia_tiled_index(d, i, ND)];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int64_t j = i + o.off[d];
        dv[d] = (T)dinv[j];
        sv[d] = (T)sd_in[j];
    }
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], dv[d] * sv[d], s);
    const T sdi = sv[ND / 2];
    const T st = dv[ND / 2] * sdi;
    sd_out[i] = (TV)(sdi - s);
    sc[i] = (TV)((T)sc[i] + st);
}

// ---------------------------------------------------------------------------
// Symmetric storage of the level operators. Every level vector of the cycle
// vanishes on Dirichlet DoFs (the defect enters with zero Dirichlet entries,
// Dirichlet rows of A, P and R keep them zero), so A may be replaced by its
// Dirichlet-eliminated form (Dirichlet columns of interior rows zeroed),
// which gives identical products on those vectors and is symmetric. Only the
// centre and the ND/2 "upper" diagonals (offset >= 0) are stored (NU =
// ND/2+1, tiled like the full storage); the coupling of row i to the lower
// neighbour j = i + off_d (d < ND/2) is the upper entry of row j at the mirrored
// offset, U[ND-1-d-ND/2][j].
// ---------------------------------------------------------------------------
template <typename TM>
__global__ void k_dia_symmetrize(int64_t n, int nd, DiaOffsets o, const uint8_t* __restrict__ dir,
                                 const TM* __restrict__ full, TM* __restrict__ up) {
    const int nu = nd / 2 + 1;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        for (int u = 0; u < nu; ++u) {
            const int d = nd / 2 + u;
            const int64_t j = i + o.off[d];
            TM v = full[dia_tiled_index(d, i, nd)];
            if (u != 0 && j >= 0 && j < n && dir[j]) v = (TM)0;   // eliminate Dirichlet columns
            up[dia_tiled_index(u, i, nu)] = v;
        }
    }
}

template <int ND>
__device__ __forceinline__ int64_t clamp_row(int64_t j, int64_t n) {
    return j < 0 ? 0 : (j >= n ? n - 1 : j);
}

// d_out = d_in - A*x with symmetric storage (x must vanish on Dirichlet DoFs)
template <typename TM, typename TV, int ND>
__device__ __forceinline__ void dias_apply_sub_row(int64_t i, int64_t n, const DiaOffsets& o, const TM* __restrict__ U,
                                                   const TV* __restrict__ x, const TV* d_in, TV* d_out) {
    typedef typename Acc<TV>::type T;
    constexpr int NU = ND / 2 + 1;
    T a[ND], xv[ND];
#pragma unroll
    for (int u = 0; u < NU; ++u) a[ND / 2 + u] = (T)U[dia_tiled_index(u, i, NU)];
#pragma unroll
    for (int d = 0; d < ND / 2; ++d)
        a[d] = (T)U[dia_tiled_index(ND - 1 - d - ND / 2, clamp_row<ND>(i + o.off[d], n), NU)];
#pragma unroll
    for (int d = 0; d < ND; ++d) xv[d] = (T)x[i + o.off[d]];
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xv[d], s);
    d_out[i] = (TV)((T)d_in[i] - s);
}
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dias_apply_sub(int64_t n, DiaOffsets o, const TM* __restrict__ U,
                                                        const TV* __restrict__ x, const TV* d_in, TV* d_out,
                                                        RowMap rm) {
    int64_t i;
    if (!map_row(rm, n, i)) return;
    dias_apply_sub_row<TM, TV, ND>(i, n, o, U, x, d_in, d_out);
}

// y = alpha*v + beta*A*x with symmetric storage (x vanishing on Dirichlet DoFs)
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dias_axpy(int64_t n, DiaOffsets o, const TM* __restrict__ U, double alpha,
                                                   const TV* v, double beta, const TV* __restrict__ x, TV* y,
                                                   RowMap rm) {
    typedef typename Acc<TV>::type T;
    constexpr int NU = ND / 2 + 1;
    int64_t i;
    if (!map_row(rm, n, i)) return;
    T a[ND], xv[ND];
#pragma unroll
    for (int u = 0; u < NU; ++u) a[ND / 2 + u] = (T)U[dia_tiled_index(u, i, NU)];
#pragma unroll
    for (int d = 0; d < ND / 2; ++d)
        a[d] = (T)U[dia_tiled_index(ND - 1 - d - ND / 2, clamp_row<ND>(i + o.off[d], n), NU)];
#pragma unroll
    for (int d = 0; d < ND; ++d) xv[d] = (T)x[i + o.off[d]];
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], xv[d], s);
    y[i] = (TV)((alpha == 0.0 ? 0.0 : alpha * (double)v[i]) + beta * (double)s);
}

// fused damped-Jacobi step with symmetric storage:
//   st = dinv .* sd_in ;  sd_out = sd_in - A*st ;  sc += st
template <typename TM, typename TV, int ND>
__device__ __forceinline__ void dias_jacobi_row(int64_t i, int64_t n, const DiaOffsets& o, const TM* __restrict__ U,
                                                const TV* __restrict__ dinv, const TV* __restrict__ sd_in,
                                                TV* __restrict__ sd_out, TV* __restrict__ sc) {
    typedef typename Acc<TV>::type T;
    constexpr int NU = ND / 2 + 1;
    T a[ND], dv[ND], sv[ND];
#pragma unroll
    for (int u = 0; u < NU; ++u) a[ND / 2 + u] = (T)U[dia_tiled_index(u, i, NU)];
#pragma unroll
    for (int d = 0; d < ND / 2; ++d)
        a[d] = (T)U[dia_tiled_index(ND - 1 - d - ND / 2, clamp_row<ND>(i + o.off[d], n), NU)];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int64_t j = i + o.off[d];
        dv[d] = (T)dinv[j];
        sv[d] = (T)sd_in[j];
    }
    T s = (T)0;
#pragma unroll
    for (int d = 0; d < ND; ++d) s = fma(a[d], dv[d] * sv[d], s);
    const T sdi = sv[ND / 2];
    const T st = dv[ND / 2] * sdi;
    sd_out[i] = (TV)(sdi - s);
    sc[i] = (TV)((T)sc[i] + st);
}
template <typename TM, typename TV, int ND>
__global__ __launch_bounds__(256) void k_dias_jacobi_step(int64_t n, DiaOffsets o, const TM* __restrict__ U,
                                                          const TV* __restrict__ dinv, const TV* __restrict__ sd_in,
                                                          TV* __restrict__ sd_out, TV* __restrict__ sc,
                                                          RowMap rm) {
    int64_t i;
    if (!map_row(rm, n, i)) return;
    dias_jacobi_row<TM, TV, ND>(i, n, o, U, dinv, sd_in, sd_out, sc);
}

// ---------------------------------------------------------------------------
// LDS-staged symmetric 27-point kernels for full 3D lattices (n = W^3).
// A workgroup owns TY consecutive lines [j0, j0+TY) of one plane k (rows
// k*W^2 + j0*W ... contiguous) and first stages, for dz = -1, 0, 1, the
// contiguous vector range covering lines j0-1 .. j0+TY of plane k+dz plus one
// entry on each side. The 27 neighbour values of a row are then LDS reads;
// global loads per row drop from 14 + 13 + 27*(vectors) to
// 14 + 13 + 3*(TY+2)/TY*(vectors). Operand values and the order of the
// multiply-adds are those of the unstaged kernels, so results are identical.
// Workgroups are grouped per XCD as in the banded row schedule: XCD c owns a
// contiguous group of bands in every plane and walks them plane by plane.
// ---------------------------------------------------------------------------
struct StagedMap {
    int32_t W, TY, maxg;
    int32_t glo[8];   // first band of XCD c's group
    int32_t gsz[8];   // bands in XCD c's group
};

template <typename T>
__device__ __forceinline__ T* lds_base() {
    extern __shared__ __align__(16) unsigned char ugx_lds[];
    return reinterpret_cast<T*>(ugx_lds);
}

// (plane k, first line j0, rows R of this workgroup); false if the block is idle
__device__ __forceinline__ bool staged_block(const StagedMap& m, int64_t& k, int64_t& j0, int64_t& R) {
    const int c = blockIdx.x & 7;
    const int64_t q = blockIdx.x >> 3;
    const int64_t g = m.gsz[c];
    if (g == 0) return false;
    k = q / g;
    if (k >= m.W) return false;
    j0 = (int64_t)(m.glo[c] + (q - k * g)) * m.TY;
    const int64_t j1 = j0 + m.TY < m.W ? j0 + m.TY : m.W;
    R = (j1 - j0) * m.W;
    return true;
}

// stage f(j) for j in [base_dz - 1, base_dz - 1 + S) of the three planes;
// S = R + 2W + 2
template <typename T, typename F>
__device__ __forceinline__ void stage3(T* lds, int64_t S, int64_t W2, int64_t first, F f) {
    // the three planes are one flat index space of 3S entries; each thread
    // issues its loads in batches of 8 independent ones before the stores
    const int n3 = 3 * (int)S, Si = (int)S, step = blockDim.x;
    constexpr int B = 8;
    for (int t0 = threadIdx.x; t0 < n3; t0 += B * step) {
        T v[B];
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int t = t0 + q * step;
            if (t < n3) {
                const int dz = t >= 2 * Si ? 2 : (t >= Si ? 1 : 0);
                v[q] = f(first + (int64_t)(dz - 1) * W2 + (t - dz * Si));
            }
        }
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int t = t0 + q * step;
            if (t < n3) lds[t] = v[q];
        }
    }
}

// LDS index of neighbour d (dx,dy,dz = d%3-1, d/3%3-1, d/9-1) of local row r
__device__ __forceinline__ int64_t staged_idx(int d, int64_t r, int64_t W, int64_t S) {
    const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9;
    return dz * S + r + W + 1 + dy * W + dx;
}

template <typename TM, typename T>
__device__ __forceinline__ void load_sym27(const TM* __restrict__ U, const DiaOffsets& o, int64_t i, int64_t n,
                                           T (&a)[27]) {
#pragma unroll
    for (int u = 0; u < 14; ++u) a[13 + u] = (T)U[dia_tiled_index(u, i, 14)];
#pragma unroll
    for (int d = 0; d < 13; ++d) a[d] = (T)U[dia_tiled_index(26 - d - 13, clamp_row<27>(i + o.off[d], n), 14)];
}

// d_out = d_in - A*x
template <typename TM, typename TV>
__global__ __launch_bounds__(256) void k_dias27_staged_apply_sub(int64_t n, DiaOffsets o, StagedMap m,
                                                                 const TM* __restrict__ U, const TV* __restrict__ x,
                                                                 const TV* d_in, TV* d_out) {
    typedef typename Acc<TV>::type T;
    int64_t k, j0, R;
    if (!staged_block(m, k, j0, R)) return;
    const int64_t W = m.W, W2 = W * W, S = R + 2 * W + 2;
    const int64_t base = k * W2 + j0 * W;
    T* lds = lds_base<T>();
    stage3(lds, S, W2, base - W - 1, [&](int64_t j) { return (T)x[j]; });
    __syncthreads();
    // lanes start on a 64-row storage tile boundary so that the coefficient
    // loads of a wavefront are aligned
    const int64_t a0 = base & 63;
    for (int64_t rr = threadIdx.x; rr < R + a0; rr += blockDim.x) {
        const int64_t r = rr - a0;
        if (r < 0) continue;
        const int64_t i = base + r;
        T a[27];
        load_sym27(U, o, i, n, a);
        T s = (T)0;
#pragma unroll
        for (int d = 0; d < 27; ++d) s = fma(a[d], lds[staged_idx(d, r, W, S)], s);
        d_out[i] = (TV)((T)d_in[i] - s);
    }
}

// y = alpha*v + beta*A*x
template <typename TM, typename TV>
__global__ __launch_bounds__(256) void k_dias27_staged_axpy(int64_t n, DiaOffsets o, StagedMap m,
                                                            const TM* __restrict__ U, double alpha, const TV* v,
                                                            double beta, const TV* __restrict__ x, TV* y) {
    typedef typename Acc<TV>::type T;
    int64_t k, j0, R;
    if (!staged_block(m, k, j0, R)) return;
    const int64_t W = m.W, W2 = W * W, S = R + 2 * W + 2;
    const int64_t base = k * W2 + j0 * W;
    T* lds = lds_base<T>();
    stage3(lds, S, W2, base - W - 1, [&](int64_t j) { return (T)x[j]; });
    __syncthreads();
    // lanes start on a 64-row storage tile boundary so that the coefficient
    // loads of a wavefront are aligned
    const int64_t a0 = base & 63;
    for (int64_t rr = threadIdx.x; rr < R + a0; rr += blockDim.x) {
        const int64_t r = rr - a0;
        if (r < 0) continue;
        const int64_t i = base + r;
        T a[27];
        load_sym27(U, o, i, n, a);
        T s = (T)0;
#pragma unroll
        for (int d = 0; d < 27; ++d) s = fma(a[d], lds[staged_idx(d, r, W, S)], s);
        y[i] = (TV)((alpha == 0.0 ? 0.0 : alpha * (double)v[i]) + beta * (double)s);
    }
}

// st = dinv .* sd_in (staged) ;  sd_out = sd_in - A*st ;  sc += st
template <typename TM, typename TV>
__global__ __launch_bounds__(256) void k_dias27_staged_jacobi_step(int64_t n, DiaOffsets o, StagedMap m,
                                                                   const TM* __restrict__ U,
                                                                   const TV* __restrict__ dinv,
                                                                   const TV* __restrict__ sd_in,
                                                                   TV* __restrict__ sd_out, TV* __restrict__ sc) {
    typedef typename Acc<TV>::type T;
    int64_t k, j0, R;
    if (!staged_block(m, k, j0, R)) return;
    const int64_t W = m.W, W2 = W * W, S = R + 2 * W + 2;
    const int64_t base = k * W2 + j0 * W;
    T* lds = lds_base<T>();
    stage3(lds, S, W2, base - W - 1, [&](int64_t j) { return (T)dinv[j] * (T)sd_in[j]; });
    __syncthreads();
    // lanes start on a 64-row storage tile boundary so that the coefficient
    // loads of a wavefront are aligned
    const int64_t a0 = base & 63;
    for (int64_t rr = threadIdx.x; rr < R + a0; rr += blockDim.x) {
        const int64_t r = rr - a0;
        if (r < 0) continue;
        const int64_t i = base + r;
        T a[27];
        load_sym27(U, o, i, n, a);
        T s = (T)0;
#pragma unroll
        for (int d = 0; d < 27; ++d) s = fma(a[d], lds[staged_idx(d, r, W, S)], s);
        const T sdi = (T)sd_in[i];
        const T st = lds[staged_idx(13, r, W, S)];
        sd_out[i] = (TV)(sdi - s);
        sc[i] = (TV)((T)sc[i] + st);
    }
}

// ---------------------------------------------------------------------------
// The matrix-free Q1 operator (q1mf_kernels.hip) plane by plane, for the
// widths that file has no schedule for (513): the operator of a uniformly
// refined cube with a coefficient that is constant per element,
// A = sum_e c_e K_ref with c_e = h k_e and the unit-cube Q1 stiffness K_ref
// (diagonal 1/3, face diagonals -1/12, body diagonal -1/12, couplings along
// element edges 0), so for an interior row
//   (A x)_i = sum_{8 cells e at i} c_e (x_i/3 - (x_f1 + x_f2 + x_f3 + x_b)/12)
// with f1..f3 the face-diagonal and b the body-diagonal corner of e seen from
// i. Boundary (Dirichlet) rows are identity rows. The products equal those of
// the Dirichlet-eliminated stored operator on vectors vanishing on Dirichlet
// DoFs, up to rounding (the assembled entries carry quadrature round-off).
// Staging as in the symmetric kernels; the block's cells (planes k-1, k,
// lines j0-1 .. j0+TY-1) are staged too.
// ---------------------------------------------------------------------------
struct MfMap {
    int32_t W, TY;
    int32_t glo[8], gsz[8];
};

template <typename T, typename F, typename O>
__device__ __forceinline__ void q1mf_block(const MfMap& m, const T* __restrict__ cell, F stage_value, O out) {
    StagedMap sm;
    sm.W = m.W;
    sm.TY = m.TY;
    for (int c = 0; c < 8; ++c) {
        sm.glo[c] = m.glo[c];
        sm.gsz[c] = m.gsz[c];
    }
    int64_t k, j0, R64;
    if (!staged_block(sm, k, j0, R64)) return;
    const int W = m.W, n = W - 1, TY = m.TY, R = (int)R64;
    const int64_t W2 = (int64_t)W * W;
    const int S = R + 2 * W + 2;
    const int64_t base = k * W2 + j0 * W;
    T* lds = lds_base<T>();
    T* cl = lds + 3 * S;                       // cells: [2][TY+1][n+2], x shifted by one
    const int CX = n + 2;
    stage3(lds, (int64_t)S, W2, base - W - 1, stage_value);
    {
        // cells: 2 (TY+1) lines of CX entries, loads batched as in stage3
        const int nc = 2 * (TY + 1) * CX, step = blockDim.x;
        constexpr int B = 8;
        for (int t0 = threadIdx.x; t0 < nc; t0 += B * step) {
            T v[B];
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int t = t0 + q * step;
                v[q] = (T)0;
                if (t < nc) {
                    const int line = t / CX, cx = t - line * CX;
                    const int64_t cz = k - 1 + line / (TY + 1), cy = j0 - 1 + line % (TY + 1);
                    if (cz >= 0 && cz < n && cy >= 0 && cy < n && cx >= 1 && cx <= n)
                        v[q] = cell[(cz * n + cy) * n + cx - 1];
                }
            }
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int t = t0 + q * step;
                if (t < nc) cl[t] = v[q];
            }
        }
    }
    __syncthreads();
    const int a0 = (int)(base & 63);
    const bool plane_bnd = (k == 0 || k == W - 1);
    for (int rr = threadIdx.x; rr < R + a0; rr += blockDim.x) {
        const int r = rr - a0;
        if (r < 0) continue;
        const int jl = (int)((unsigned)r / (unsigned)W), x = r - jl * W;
        const int y = (int)j0 + jl;
        // neighbour (dx,dy,dz) of local row r in the staged planes
        const int c0 = r + W + 1;
        auto X = [&](int dx, int dy, int dz) { return lds[(dz + 1) * S + c0 + dy * W + dx]; };
        const T xi = X(0, 0, 0);
        T s;
        if (plane_bnd || x == 0 || x == W - 1 || y == 0 || y == W - 1) {
            s = xi;
        } else {
            // cell (a,b,c) = element (x-1+a, y-1+b, k-1+c)
            auto Cc = [&](int a, int b, int c) { return cl[(c * (TY + 1) + jl + b) * CX + x + a]; };
            T ce[2][2][2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int a = 0; a < 2; ++a) ce[c][b][a] = Cc(a, b, c);
            T csum = (T)0, off = (T)0;
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        csum += ce[c][b][a];
                        off = fma(ce[c][b][a], X(2 * a - 1, 2 * b - 1, 2 * c - 1), off);   // body diagonal
                    }
            // face diagonals: each shared by the two cells of the element face
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int a = 0; a < 2; ++a)
                    off = fma(ce[0][b][a] + ce[1][b][a], X(2 * a - 1, 2 * b - 1, 0), off);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int a = 0; a < 2; ++a)
                    off = fma(ce[c][0][a] + ce[c][1][a], X(2 * a - 1, 0, 2 * c - 1), off);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    off = fma(ce[c][b][0] + ce[c][b][1], X(0, 2 * b - 1, 2 * c - 1), off);
            s = csum * xi * (T)(1.0 / 3.0) - off * (T)(1.0 / 12.0);
        }
        out(base + r, xi, s);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_q1mf_jacobi_step(MfMap m, const T* __restrict__ cell,
                                                          const T* __restrict__ dinv, const T* __restrict__ sd_in,
                                                          T* __restrict__ sd_out, T* __restrict__ sc) {
    q1mf_block<T>(
        m, cell, [&](int64_t j) { return dinv[j] * sd_in[j]; },
        [&](int64_t i, T st, T s) {
            sd_out[i] = sd_in[i] - s;
            sc[i] = sc[i] + st;
        });
}

template <typename T>
__global__ __launch_bounds__(256) void k_q1mf_apply_sub(MfMap m, const T* __restrict__ cell, const T* __restrict__ x,
                                                        const T* d_in, T* d_out) {
    q1mf_block<T>(
        m, cell, [&](int64_t j) { return x[j]; }, [&](int64_t i, T, T s) { d_out[i] = d_in[i] - s; });
}

template <typename T>
__global__ __launch_bounds__(256) void k_q1mf_axpy(MfMap m, const T* __restrict__ cell, double alpha, const T* v,
                                                   double beta, const T* __restrict__ x, T* y) {
    q1mf_block<T>(
        m, cell, [&](int64_t j) { return x[j]; },
        [&](int64_t i, T, T s) { y[i] = (T)((alpha == 0.0 ? 0.0 : alpha * (double)v[i]) + beta * (double)s); });
}

// c_e = h exp(theta_e) per element (lattice order of elements); theta null: k = 1
template <typename T>
__global__ void k_q1mf_coeff(int64_t ne, double h, const double* __restrict__ theta, T* __restrict__ c) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < ne; e += (int64_t)gridDim.x * blockDim.x)
        c[e] = (T)(h * (theta ? exp(theta[e]) : 1.0));
}

// sc += dinv .* sd  (last post-smoothing step on levels below the top, where
// the final defect update is skipped: mg_solver_impl.hpp:1954)
template <typename TV>
__global__ __launch_bounds__(256) void k_jacobi_accumulate(int64_t n, const TV* dinv, const TV* sd, TV* sc) {
    UGX_STREAM_LOOP(n) {
        TV dv[kStreamE], sv[kStreamE], cv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            dv[e] = ldnt(dinv + i);
            sv[e] = ldnt(sd + i);
            cv[e] = ldnt(sc + i);
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n)
                stnt((TV)((double)cv[e] + (double)dv[e] * (double)sv[e]), sc + UGX_STREAM_IDX(e));
    }
}

// the last top-level post-smoothing step fused with the conversion of the
// correction: z = (double)(sc + dinv .* sd), with the arithmetic of
// k_jacobi_accumulate, and (partial != nullptr) partial sums of z.r as
// k_convert_dot forms them
template <typename TV>
__global__ __launch_bounds__(256) void k_jacobi_convert_dot(int64_t n, const TV* __restrict__ dinv,
                                                            const TV* __restrict__ sd, const TV* __restrict__ sc,
                                                            double* __restrict__ z, const double* __restrict__ r,
                                                            double* __restrict__ partial) {
    double acc = 0.0;
    UGX_STREAM_LOOP(n) {
        TV dv[kStreamE], sv[kStreamE], cv[kStreamE];
        double rv[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_SAFE(e, n);
            dv[e] = ldnt(dinv + i);
            sv[e] = ldnt(sd + i);
            cv[e] = ldnt(sc + i);
            rv[e] = partial ? ldnt(r + i) : 0.0;
        }
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) {
            const int64_t i = UGX_STREAM_IDX(e);
            if (i >= n) continue;
            const double zi = (double)(TV)((double)cv[e] + (double)dv[e] * (double)sv[e]);
            stnt(zi, z + i);
            acc += zi * rv[e];
        }
    }
    if (partial) block_partial(acc, partial);
}

// dinv from the DIA centre diagonal
template <typename TM, typename TV>
__global__ void k_dia_jacobi_diag(int64_t n, int nd, const TM* dia, double omega, TV* dinv, int* bad) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double m = (double)dia[dia_tiled_index(nd / 2, i, nd)];
        m *= 1.0 / omega;
        if (m == 0.0) { bad[0] = 1; dinv[i] = (TV)0; }
        else dinv[i] = (TV)(1.0 / m);
    }
}

// ---------------------------------------------------------------------------
// Matrix-free P1 transfer between the lattice levels of hexahedra. Weights are
// the exact dyadic P entries; the Dirichlet adjustment is applied exactly as on
// the assembled matrices.
// ---------------------------------------------------------------------------

// prolongation with accumulation: st_f = sum_c P(f,c) sc_c ; sc_f += st_f
// The coarse correction a prolongation reads: sc, or (with dinv) the value the
// coarse level's last post-smoothing update sc + dinv .* sd would store, with
// the arithmetic of k_jacobi_accumulate. Folding that update into the
// prolongation saves its launch; the level's own sc is not read again.
template <typename TV>
struct CoarseCorr {
    const TV* sc;
    const TV* dinv;
    const TV* sd;
    __device__ __forceinline__ TV operator()(int64_t j) const {
        if (!dinv) return sc[j];
        return coarse_fold<TV>(sc[j], dinv[j], sd[j]);
    }
};

template <typename TV>
__global__ __launch_bounds__(256) void k_prolong_add(int Wc, int Wf, int64_t n_f, CoarseCorr<TV> scc,
                                                     const uint8_t* __restrict__ dir_f, TV* __restrict__ st,
                                                     TV* __restrict__ sc, FastDiv fw) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= n_f) return;
    const uint32_t q1 = fdiv((uint32_t)i, fw);
    const int x = (int)((uint32_t)i - q1 * (uint32_t)Wf);
    const uint32_t q2 = fdiv(q1, fw);
    const int y = (int)(q1 - q2 * (uint32_t)Wf);
    const int z = (int)q2;
    const int x0 = x >> 1, y0 = y >> 1, z0 = z >> 1;
    const int ox = x & 1, oy = y & 1, oz = z & 1;
    double v = 0.0;
    // Dirichlet DoFs lie on the lattice boundary: only there is the flag read
    const bool bnd = x == 0 || y == 0 || x == Wf - 1 || y == Wf - 1 || z == 0 || z == Wf - 1;
    const int nodd = ox + oy + oz;
    if (bnd && dir_f[i] && nodd != 0) {
        v = 0.0;   // Dirichlet rows of P are zeroed except vertex copies
    } else {
        const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
        for (int dz = 0; dz <= oz; ++dz)
            for (int dy = 0; dy <= oy; ++dy)
                for (int dx = 0; dx <= ox; ++dx)
                    v = fma(w, (double)scc(((int64_t)(z0 + dz) * Wc + (y0 + dy)) * Wc + (x0 + dx)), v);
    }
    // c += t in the vector precision (mg_solver_impl.hpp:1905)
    const TV t = (TV)v;
    st[i] = t;
    sc[i] = sc[i] + t;
}

// restriction: sdc_c = sum_f R(c,f) sd_f with R = P^T (Dirichlet coarse rows:
// injection from the vertex copy)
// 3D prolongation driven by the coarse points: thread c loads its (up to 8)
// coarse corners once and writes its 2x2x2 fine children (fine x pairs of
// neighbouring threads are contiguous). Weights and summation order as in
// k_prolong_add, so the values are identical.
template <typename TV>
__device__ __forceinline__ void prolong3_point(int x, int y, int z, int Wc, int Wf, const CoarseCorr<TV>& scc,
                                               const uint8_t* __restrict__ dir_f, TV* __restrict__ st,
                                               TV* __restrict__ sc) {
    double v[2][2][2];
#pragma unroll
    for (int dz = 0; dz < 2; ++dz)
#pragma unroll
        for (int dy = 0; dy < 2; ++dy)
#pragma unroll
            for (int dx = 0; dx < 2; ++dx) {
                const bool in = x + dx < Wc && y + dy < Wc && z + dz < Wc;
                v[dz][dy][dx] = in ? (double)scc(((int64_t)(z + dz) * Wc + (y + dy)) * Wc + (x + dx)) : 0.0;
            }
#pragma unroll
    for (int oz = 0; oz < 2; ++oz)
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
#pragma unroll
            for (int ox = 0; ox < 2; ++ox) {
                const int fx = 2 * x + ox, fy = 2 * y + oy, fz = 2 * z + oz;
                if (fx >= Wf || fy >= Wf || fz >= Wf) continue;
                const int64_t f = ((int64_t)fz * Wf + fy) * Wf + fx;
                const int nodd = ox + oy + oz;
                const bool bnd = fx == 0 || fy == 0 || fz == 0 || fx == Wf - 1 || fy == Wf - 1 || fz == Wf - 1;
                double val = 0.0;
                if (!(bnd && nodd != 0 && dir_f[f])) {
                    const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                    for (int dz = 0; dz <= oz; ++dz)
                        for (int dy = 0; dy <= oy; ++dy)
                            for (int dx = 0; dx <= ox; ++dx) val = fma(w, v[dz][dy][dx], val);
                }
                const TV t = (TV)val;
                st[f] = t;
                sc[f] = sc[f] + t;
            }
}
template <typename TV>
__global__ __launch_bounds__(256) void k_prolong_add3(int Wc, int Wf, int64_t n_c, CoarseCorr<TV> scc,
                                                      const uint8_t* __restrict__ dir_f, TV* __restrict__ st,
                                                      TV* __restrict__ sc, FastDiv fc) {
    // consecutive coarse points (and so fine planes) on one XCD
    const int64_t c = xcd_block((n_c + 255) / 256) * 256 + threadIdx.x;
    if (c >= n_c) return;
    const uint32_t q1 = fdiv((uint32_t)c, fc);
    const int x = (int)((uint32_t)c - q1 * (uint32_t)Wc);
    const uint32_t q2 = fdiv(q1, fc);
    const int y = (int)(q1 - q2 * (uint32_t)Wc), z = (int)q2;
    prolong3_point<TV>(x, y, z, Wc, Wf, scc, dir_f, st, sc);
}

template <typename TV>
__global__ __launch_bounds__(256) void k_restrict(int Wc, int Wf, int64_t n_c, const TV* __restrict__ sdf,
                                                  const uint8_t* __restrict__ dir_c, const uint8_t* __restrict__ dir_f,
                                                  TV* __restrict__ sdc, FastDiv fw, TV* __restrict__ zc) {
    const int64_t c = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (c >= n_c) return;
    if (zc) zc[c] = (TV)0;   // the coarse correction starts from zero
    const uint32_t q1 = fdiv((uint32_t)c, fw);
    const int x = (int)((uint32_t)c - q1 * (uint32_t)Wc);
    const uint32_t q2 = fdiv(q1, fw);
    const int y = (int)(q1 - q2 * (uint32_t)Wc);
    const int z = (int)q2;
    const int fx = 2 * x, fy = 2 * y, fz = 2 * z;
    const int nf = Wf - 1;
    // Dirichlet DoFs lie on the lattice boundary: away from it no flag is read
    const bool inner = x >= 2 && y >= 2 && x <= Wc - 3 && y <= Wc - 3 && z >= 2 && z <= Wc - 3;
    if (inner) {
        double s = 0.0;
#pragma unroll
        for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
                for (int dx = -1; dx <= 1; ++dx) {
                    const int nodd = (dx != 0) + (dy != 0) + (dz != 0);
                    const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                    s += w * (double)sdf[((int64_t)(fz + dz) * Wf + (fy + dy)) * Wf + (fx + dx)];
                }
        sdc[c] = (TV)s;
        return;
    }
    if (dir_c[c]) {
        sdc[c] = sdf[((int64_t)fz * Wf + fy) * Wf + fx];
        return;
    }
    double s = 0.0;
    for (int dz = -1; dz <= 1; ++dz) {
        const int zz = fz + dz;
        if (zz < 0 || zz > nf) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            const int yy = fy + dy;
            if (yy < 0 || yy > nf) continue;
            for (int dx = -1; dx <= 1; ++dx) {
                const int xx = fx + dx;
                if (xx < 0 || xx > nf) continue;
                const int nodd = (dx != 0) + (dy != 0) + (dz != 0);
                const int64_t f = ((int64_t)zz * Wf + yy) * Wf + xx;
                if (dir_f[f] && nodd != 0) continue;   // zeroed P rows
                const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                s += w * (double)sdf[f];
            }
        }
    }
    sdc[c] = (TV)s;
}

// ---------------------------------------------------------------------------
// Tiled 3D transfers between lattices with Wf = 2 Wc - 1 whose Dirichlet DoFs
// are exactly the lattice boundary (the level flags the multigrid levels
// carry). Then an interior coarse point has no fine neighbour outside the
// lattice or on its boundary (2x - 1 >= 1 and 2x + 1 <= Wf - 2 for
// 1 <= x <= Wc - 2), so its restriction is the full 27-term sum and a
// boundary coarse point takes the value of its fine copy; a fine boundary
// point receives only the injection from its copy. Each workgroup stages the
// lines it needs in LDS with contiguous loads, so every global access is
// coalesced; the per-point arithmetic and its order are those of k_restrict
// and k_prolong_add3, so the results are identical.
// ---------------------------------------------------------------------------
template <typename TV>
struct TransferTile {
    static constexpr int TY = sizeof(TV) == 4 ? 4 : 2;   // coarse lines per workgroup
};

// restriction: one workgroup per TY coarse lines of a coarse plane z; LDS
// holds fine planes 2z-1 .. 2z+1, lines 2y0-1 .. 2y0+2TY-1 of each, every
// line padded with one zero on either side
template <typename TV>
__global__ __launch_bounds__(256) void k_restrict3_tiled(int Wc, int Wf, int nbands, const TV* __restrict__ sdf,
                                                         TV* __restrict__ sdc, TV* __restrict__ zc) {
    constexpr int TY = TransferTile<TV>::TY;
    constexpr int NL = 2 * TY + 1;
    // consecutive coarse planes on one XCD (its L2 then fetches each fine
    // plane about once)
    const int64_t lb = xcd_block((int64_t)Wc * nbands);
    if (lb >= (int64_t)Wc * nbands) return;
    const int z = (int)(lb / nbands), band = (int)(lb - (int64_t)z * nbands);
    const int y0 = band * TY;
    const int LW = Wf + 2;
    TV* lds = lds_base<TV>();
    const int total = 3 * NL * LW;
    // the loads of 4 entries per thread are issued before any is stored
    for (int t0 = threadIdx.x; t0 < total; t0 += 4 * 256) {
        int64_t j[4];
        TV v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = t0 + u * 256;
            const int row = t / LW, xi = t - row * LW;
            const int pl = row >= 2 * NL ? 2 : row >= NL ? 1 : 0, ln = row - pl * NL;
            const int fz = 2 * z - 1 + pl, fy = 2 * y0 - 1 + ln, fx = xi - 1;
            j[u] = (t < total && fz >= 0 && fz < Wf && fy >= 0 && fy < Wf && fx >= 0 && fx < Wf)
                       ? ((int64_t)fz * Wf + fy) * Wf + fx
                       : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = j[u] >= 0 ? sdf[j[u]] : (TV)0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (t0 + u * 256 < total) lds[t0 + u * 256] = v[u];
    }
    __syncthreads();
    const int ny = min(TY, Wc - y0);
    int ly = 0, x = threadIdx.x;
    while (x >= Wc) {
        x -= Wc;
        ++ly;
    }
    for (int t = threadIdx.x; t < ny * Wc; t += 256, x += 256) {
        while (x >= Wc) {
            x -= Wc;
            ++ly;
        }
        const int y = y0 + ly;
        const int64_t c = ((int64_t)z * Wc + y) * Wc + x;
        if (zc) zc[c] = (TV)0;   // the coarse correction starts from zero
        // fine point (2x + dx, 2y + dy, 2z + dz): plane 1 + dz, line 2 ly + 1 + dy, column 2x + 1 + dx
        auto at = [&](int dz, int dy, int dx) { return lds[((1 + dz) * NL + 2 * ly + 1 + dy) * LW + 2 * x + 1 + dx]; };
        if (x == 0 || y == 0 || z == 0 || x == Wc - 1 || y == Wc - 1 || z == Wc - 1) {
            sdc[c] = at(0, 0, 0);
            continue;
        }
        double s = 0.0;
#pragma unroll
        for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
                for (int dx = -1; dx <= 1; ++dx) {
                    const int nodd = (dx != 0) + (dy != 0) + (dz != 0);
                    const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                    s += w * (double)at(dz, dy, dx);
                }
        sdc[c] = (TV)s;
    }
}

// prolongation st = P scc, sc += st: one workgroup per fine plane fz and the
// fine lines 2y0 .. 2y0+2TY-1 of a coarse band; LDS holds coarse planes
// fz/2 and fz/2 + 1, lines y0 .. y0+TY, each line padded with one zero. The
// Dirichlet rows of P are those of the lattice boundary (every boundary point
// of the hexahedral hierarchy is Dirichlet), so no flags are read.
template <typename TV>
__global__ __launch_bounds__(256) void k_prolong3_tiled(int Wc, int Wf, int nbands, CoarseCorr<TV> scc,
                                                        TV* __restrict__ st, TV* __restrict__ sc, FastDiv fwf) {
    constexpr int TY = TransferTile<TV>::TY;
    constexpr int NL = TY + 1;
    // consecutive fine planes on one XCD: its L2 then fetches each coarse
    // plane about once instead of every XCD fetching all of them
    const int64_t lb = xcd_block((int64_t)Wf * nbands);
    if (lb >= (int64_t)Wf * nbands) return;
    const int fz = (int)(lb / nbands), band = (int)(lb - (int64_t)fz * nbands);
    const int y0 = band * TY, cz0 = fz >> 1, oz = fz & 1;
    const int LW = Wc + 1;
    TV* lds = lds_base<TV>();
    // coarse plane cz0 + 1 only for an odd fine plane; the loads of 4
    // entries per thread are issued before any is stored
    const int total = (1 + oz) * NL * LW;
    for (int t0 = threadIdx.x; t0 < total; t0 += 4 * 256) {
        int64_t j[4];
        TV v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = t0 + u * 256;
            const int row = t / LW, xs = t - row * LW;
            const int pl = row >= NL ? 1 : 0, ln = row - pl * NL;
            const int cz = cz0 + pl, cy = y0 + ln;
            j[u] = (t < total && cz < Wc && cy < Wc && xs < Wc) ? ((int64_t)cz * Wc + cy) * Wc + xs : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = j[u] >= 0 ? scc(j[u]) : (TV)0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (t0 + u * 256 < total) lds[t0 + u * 256] = v[u];
    }
    __syncthreads();
    const int fy0 = 2 * y0, ny = min(2 * TY, Wf - fy0);
    // every fine point: the (up to 8) coarse values around it times w =
    // 2^-nodd, accumulated in the order (dz, dy, dx) as prolong3_point does
    // with fma; a power-of-two w commutes with rounding, so that chain equals
    // w times the plain sum in the same order. Terms a point does not have add
    // 0 and read a value that is there, so the 8 reads of a point are issued
    // together and no read waits for the previous sum.
    const TV* zl = lds;
    const TV* zh = lds + oz * NL * LW;
    // the fine points in rounds of 4 per thread: the 4 loads of sc of a round
    // are issued before any of them is used (8 per round, or loading the
    // first round before the staging, measured slower: more registers, fewer
    // resident waves)
    constexpr int U = 4;
    const int nf = ny * Wf;
    for (int t0 = threadIdx.x; t0 < nf; t0 += U * 256) {
        int64_t f[U];
        int fx[U], fy[U];
        TV cold[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = t0 + u * 256;
            const int lyf = (int)fdiv((uint32_t)t, fwf);
            fx[u] = t - lyf * Wf;
            fy[u] = fy0 + lyf;
            f[u] = ((int64_t)fz * Wf + fy[u]) * Wf + fx[u];
            cold[u] = t < nf ? sc[f[u]] : (TV)0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t0 + u * 256 >= nf) continue;
            const int ox = fx[u] & 1, oy = fy[u] & 1, x = fx[u] >> 1, ly = (fy[u] - fy0) >> 1;
            const int nodd = ox + oy + oz;
            const bool bnd = fx[u] == 0 || fy[u] == 0 || fz == 0 || fx[u] == Wf - 1 || fy[u] == Wf - 1 || fz == Wf - 1;
            const int o = ly * LW + x, sy = oy * LW;
            const TV a0 = zl[o], a1 = zl[o + ox], a2 = zl[o + sy], a3 = zl[o + sy + ox];
            const TV b0 = zh[o], b1 = zh[o + ox], b2 = zh[o + sy], b3 = zh[o + sy + ox];
            double sum = (double)a0;
            sum += ox ? (double)a1 : 0.0;
            sum += oy ? (double)a2 : 0.0;
            sum += (ox & oy) ? (double)a3 : 0.0;
            sum += oz ? (double)b0 : 0.0;
            sum += (oz & ox) ? (double)b1 : 0.0;
            sum += (oz & oy) ? (double)b2 : 0.0;
            sum += (oz & ox & oy) ? (double)b3 : 0.0;
            const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
            const double val = (bnd && nodd != 0) ? 0.0 : w * sum;
            const TV tv = (TV)val;
            st[f[u]] = tv;
            sc[f[u]] = cold[u] + tv;
        }
    }
}

// z-marching restriction: a workgroup owns TY coarse lines of a chunk of
// coarse planes and keeps the fine planes 2z-1, 2z, 2z+1 of its band (lines
// 2y0-1 .. 2y0+2TY-1, padded by one zero per side) in an LDS ring of three;
// coarse plane z+1 needs two new fine planes, which are loaded into registers
// while plane z is computed and then replace 2z-1 and 2z. Each fine value is
// loaded once per chunk (plus one plane per chunk), by long-lived workgroups.
// Arithmetic and order as k_restrict3_tiled.
struct RzMap {
    int32_t Wc, Wf, TY, nchunks;
    int32_t glo[8], gsz[8];
};
constexpr int kRzSlots = 6;   // staged entries per thread and fine plane (5 lines x (Wf + 2) <= 6 * 256)

template <typename TV>
__global__ __launch_bounds__(256) void k_restrict3_z(RzMap m, const TV* __restrict__ sdf, TV* __restrict__ sdc,
                                                     TV* __restrict__ zc) {
    const int xc = blockIdx.x & 7, q = blockIdx.x >> 3, g = m.gsz[xc];
    const int chunk = g == 0 ? 0 : q / g;
    if (g == 0 || chunk >= m.nchunks) return;
    const int band = m.glo[xc] + (q - chunk * g);
    const int Wc = m.Wc, Wf = m.Wf, TY = m.TY;
    const int y0 = band * TY, ny = min(TY, Wc - y0);
    const int z0 = (int)((int64_t)chunk * Wc / m.nchunks), z1 = (int)((int64_t)(chunk + 1) * Wc / m.nchunks);
    const int NL = 2 * TY + 1, LW = Wf + 2, PL = NL * LW;
    const int tid = threadIdx.x;
    const int64_t Wf2 = (int64_t)Wf * Wf;
    TV* lds = lds_base<TV>();
    // offset inside a fine plane of each staging slot (-1: outside the lattice
    // or the tile); the same in every plane
    int off[kRzSlots];
#pragma unroll
    for (int u = 0; u < kRzSlots; ++u) {
        const int t = tid + u * 256;
        off[u] = -1;
        if (t < PL) {
            const int ln = t / LW, xi = t - ln * LW;
            const int fy = 2 * y0 - 1 + ln, fx = xi - 1;
            if (fy >= 0 && fy < Wf && fx >= 0 && fx < Wf) off[u] = fy * Wf + fx;
        }
    }
    auto slot = [&](int f) { return lds + ((f + 3) % 3) * PL; };
    auto fetch = [&](int f, int u) -> TV {
        return (f >= 0 && f < Wf && off[u] >= 0) ? sdf[(int64_t)f * Wf2 + off[u]] : (TV)0;
    };
    for (int f = 2 * z0 - 1; f <= 2 * z0 + 1; ++f) {
        TV* dst = slot(f);
#pragma unroll
        for (int u = 0; u < kRzSlots; ++u) {
            const int t = tid + u * 256;
            if (t < PL) dst[t] = fetch(f, u);
        }
    }
    __syncthreads();
    // (line, column) of this thread's first output, advanced without divisions
    int ly0 = 0, x0 = tid;
    while (x0 >= Wc) {
        x0 -= Wc;
        ++ly0;
    }
    for (int z = z0; z < z1; ++z) {
        const bool more = z + 1 < z1;
        TV pa[kRzSlots], pb[kRzSlots];
#pragma unroll
        for (int u = 0; u < kRzSlots; ++u) {
            pa[u] = more ? fetch(2 * z + 2, u) : (TV)0;
            pb[u] = more ? fetch(2 * z + 3, u) : (TV)0;
        }
        const TV* sm = slot(2 * z - 1);
        const TV* s0 = slot(2 * z);
        const TV* sp = slot(2 * z + 1);
        int ly = ly0, x = x0;
        for (int t = tid; t < ny * Wc; t += 256, x += 256) {
            while (x >= Wc) {
                x -= Wc;
                ++ly;
            }
            const int y = y0 + ly;
            const int64_t c = ((int64_t)z * Wc + y) * Wc + x;
            if (zc) zc[c] = (TV)0;   // the coarse correction starts from zero
            auto at = [&](int dz, int dy, int dx) {
                const TV* pl = dz < 0 ? sm : (dz > 0 ? sp : s0);
                return pl[(2 * ly + 1 + dy) * LW + 2 * x + 1 + dx];
            };
            if (x == 0 || y == 0 || z == 0 || x == Wc - 1 || y == Wc - 1 || z == Wc - 1) {
                sdc[c] = at(0, 0, 0);
                continue;
            }
            double sum = 0.0;
#pragma unroll
            for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
                for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
                    for (int dx = -1; dx <= 1; ++dx) {
                        const int nodd = (dx != 0) + (dy != 0) + (dz != 0);
                        const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                        sum += w * (double)at(dz, dy, dx);
                    }
            sdc[c] = (TV)sum;
        }
        __syncthreads();   // every thread is done with planes 2z-1 and 2z
        if (more) {
            TV* da = slot(2 * z + 2);
            TV* db = slot(2 * z + 3);
#pragma unroll
            for (int u = 0; u < kRzSlots; ++u) {
                const int t = tid + u * 256;
                if (t < PL) {
                    da[t] = pa[u];
                    db[t] = pb[u];
                }
            }
        }
        __syncthreads();
    }
}

static size_t restrict3_tiled_lds(int Wf, size_t elem, int TY) { return (size_t)3 * (2 * TY + 1) * (Wf + 2) * elem; }
static size_t prolong3_tiled_lds(int Wc, size_t elem, int TY) { return (size_t)2 * (TY + 1) * (Wc + 1) * elem; }

// ---------------------------------------------------------------------------
// base-level solve (lu_block.hpp), one workgroup
// ---------------------------------------------------------------------------
template <typename TV>
__global__ __launch_bounds__(1024) void k_lu_solve(int n, const double* __restrict__ Linv, const double* __restrict__ Uinv,
                                                   const int32_t* __restrict__ perm, const TV* __restrict__ b,
                                                   TV* __restrict__ x) {
    extern __shared__ double sh[];
    lu_solve_block<TV>(n, Linv, Uinv, perm, b, x, sh);
}


// ---------------------------------------------------------------------------
// Assembly
// ---------------------------------------------------------------------------

// lattice -> DoF inverse map
__global__ void k_invert_map(int64_t n, const int32_t* dof_of_lat, int32_t* lat_of_dof) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        lat_of_dof[dof_of_lat[i]] = (int32_t)i;
}

// number of lattice neighbours (including self) of every DoF row: 27-point box
// (hexahedra) or 7-point (triangles with (1,1) diagonals)
__global__ void k_pattern_count(int dim, int W, int64_t n, const int32_t* lat_of_dof, int32_t* cnt) {
    for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = lat_of_dof[r];
        const int x = (int)(l % W), y = (int)((l / W) % W);
        const int nx = 1 + (x > 0) + (x < W - 1), ny = 1 + (y > 0) + (y < W - 1);
        if (dim == 3) {
            const int z = (int)(l / ((int64_t)W * W));
            const int nz = 1 + (z > 0) + (z < W - 1);
            cnt[r] = nx * ny * nz;
        } else {
            cnt[r] = nx * ny - ((x > 0 && y < W - 1) ? 1 : 0) - ((x < W - 1 && y > 0) ? 1 : 0);
        }
    }
}

__device__ __forceinline__ int32_t csr_slot(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                            int32_t r, int32_t c) {
    int32_t lo = rowptr[r], hi = rowptr[r + 1] - 1;
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (col[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    return lo;   // the pattern contains (r,c) by construction
}

// Q1 FE element matrix of a hexahedron with trilinear geometry, 2x2x2 Gauss,
// k(x) = exp(theta[fine element containing x]) (1 without theta); rhs
// f_const * int phi_i. Local vertex order is the reference hexahedron's.
__device__ void q1_hex_element(const double X[8][3], const double* __restrict__ theta, int nfine, double f_const,
                               double Ke[8][8], double fe[8]) {
    q1_hex_element_k(
        X,
        [=](const double* xq) {
            if (!theta) return 1.0;
            int cx = (int)floor(xq[0] * nfine), cy = (int)floor(xq[1] * nfine), cz = (int)floor(xq[2] * nfine);
            cx = cx < 0 ? 0 : (cx >= nfine ? nfine - 1 : cx);
            cy = cy < 0 ? 0 : (cy >= nfine ? nfine - 1 : cy);
            cz = cz < 0 ? 0 : (cz >= nfine ? nfine - 1 : cz);
            return exp(theta[((int64_t)cz * nfine + cy) * nfine + cx]);
        },
        f_const, Ke, fe);
}

// corner c of lattice element (ex,ey,ez): reference hexahedron order
__device__ __forceinline__ void hex_corner(int c, int& dx, int& dy, int& dz) {
    dx = (c == 1 || c == 2 || c == 5 || c == 6);
    dy = (c == 2 || c == 3 || c == 6 || c == 7);
    dz = (c >= 4);
}

// Adjoint element gradient on the finest level (one element per thread, no
// scatter): g_e = -sum_{a interior} lambda_a (A_e u_e)_a. On the finest level
// k = exp(theta_e) at every quadrature point of e, so dA_e/dtheta_e = A_e; A_e
// is recomputed here rather than stored. Dirichlet rows (DoF >= n_inner) do not
// depend on theta.
__global__ __launch_bounds__(128) void k_adjoint_grad_q1_hex(int n, double h, const double* __restrict__ theta,
                                                             const int32_t* __restrict__ dof_of_lat, int64_t n_inner,
                                                             const double* __restrict__ u,
                                                             const double* __restrict__ lambda,
                                                             double* __restrict__ grad) {
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * n * n) return;
    const int ex = (int)(e % n), ey = (int)((e / n) % n), ez = (int)(e / ((int64_t)n * n));
    const int W = n + 1;
    double X[8][3];
    int32_t dof[8];
    for (int a = 0; a < 8; ++a) {
        int dx, dy, dz;
        hex_corner(a, dx, dy, dz);
        X[a][0] = (ex + dx) * h;
        X[a][1] = (ey + dy) * h;
        X[a][2] = (ez + dz) * h;
        dof[a] = dof_of_lat[((int64_t)(ez + dz) * W + (ey + dy)) * W + (ex + dx)];
    }
    double Ke[8][8], fe[8];
    q1_hex_element(X, theta, n, 0.0, Ke, fe);
    double ue[8];
    for (int b = 0; b < 8; ++b) ue[b] = u[dof[b]];
    double acc = 0.0;
    for (int a = 0; a < 8; ++a) {
        if (dof[a] >= n_inner) continue;
        double row = 0.0;
        for (int b = 0; b < 8; ++b) row += Ke[a][b] * ue[b];
        acc += lambda[dof[a]] * row;
    }
    grad[e] = -acc;
}

// zero the Dirichlet entries (DoF >= n_inner) of a top-level vector
__global__ void k_zero_range(int64_t lo, int64_t hi, double* x) {
    for (int64_t i = lo + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < hi; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = 0.0;
}

// FV1 on P1 triangles (box method), lattice squares split along (1,1), k =
// exp(theta[fine square containing the scvf's integration point]).
// Colour = (sx%2, sy%2, which triangle).
__device__ void fv1_tri_element(const double X[3][2], const double* __restrict__ theta, int nfine, double Ke[3][3],
                                double& area) {
    fv1_tri_element_k(
        X,
        [=](const double* ip) {
            if (!theta) return 1.0;
            int cx = (int)floor(ip[0] * nfine), cy = (int)floor(ip[1] * nfine);
            cx = cx < 0 ? 0 : (cx >= nfine ? nfine - 1 : cx);
            cy = cy < 0 ? 0 : (cy >= nfine ? nfine - 1 : cy);
            return exp(theta[(int64_t)cy * nfine + cx]);
        },
        Ke, area);
}

template <typename TM>
__global__ __launch_bounds__(128) void k_assemble_fv1_tri(int n, int color, double h, const double* __restrict__ theta,
                                                          int nfine, const double* __restrict__ f_at_dof,
                                                          const int32_t* __restrict__ dof_of_lat,
                                                          const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                          TM* __restrict__ csr_val, TM* __restrict__ dia, int64_t dia_n,
                                                          double* __restrict__ rhs) {
    const int hn = (n + 1) / 2;
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= (int64_t)hn * hn) return;
    const int sx = 2 * (int)(e % hn) + (color & 1), sy = 2 * (int)(e / hn) + ((color >> 1) & 1);
    const int upper = (color >> 2) & 1;
    if (sx >= n || sy >= n) return;
    const int W = n + 1;
    // lower: (0,0),(1,0),(1,1); upper: (0,0),(1,1),(0,1)
    const int cxs[2][3] = {{0, 1, 1}, {0, 1, 0}};
    const int cys[2][3] = {{0, 0, 1}, {0, 1, 1}};
    double X[3][2];
    int64_t lat[3];
    for (int a = 0; a < 3; ++a) {
        const int xx = sx + cxs[upper][a], yy = sy + cys[upper][a];
        X[a][0] = xx * h;
        X[a][1] = yy * h;
        lat[a] = (int64_t)yy * W + xx;
    }
    double Ke[3][3], area;
    fv1_tri_element(X, theta, nfine, Ke, area);
    if (rowptr) {
        int32_t dof[3];
        for (int a = 0; a < 3; ++a) dof[a] = dof_of_lat[lat[a]];
        for (int a = 0; a < 3; ++a) {
            for (int b = 0; b < 3; ++b) {
                const int32_t k = csr_slot(rowptr, col, dof[a], dof[b]);
                csr_val[k] = (TM)((double)csr_val[k] + Ke[a][b]);
            }
            if (rhs && f_at_dof) rhs[dof[a]] += f_at_dof[dof[a]] * (area / 3.0);
        }
    } else {
        for (int a = 0; a < 3; ++a) {
            for (int b = 0; b < 3; ++b) {
                const int dx = (int)((lat[b] % W) - (lat[a] % W)), dy = (int)((lat[b] / W) - (lat[a] / W));
                const int d = (dy + 1) * 3 + (dx + 1);
                TM* p = dia + dia_tiled_index(d, lat[a], 9);
                *p = (TM)((double)*p + Ke[a][b]);
            }
            if (rhs && f_at_dof) rhs[lat[a]] += f_at_dof[dof_of_lat[lat[a]]] * (area / 3.0);
        }
    }
}

// Dirichlet rows in the CSR (DoF numbering): all values 0, diagonal 1, rhs 0
template <typename TM>
__global__ void k_dirichlet_csr(int64_t n, int64_t n_inner, const int32_t* rowptr, const int32_t* col, TM* val,
                                double* rhs) {
    for (int64_t r = n_inner + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n;
         r += (int64_t)gridDim.x * blockDim.x) {
        for (int32_t k = rowptr[r]; k < rowptr[r + 1]; ++k) val[k] = (TM)(col[k] == r ? 1.0 : 0.0);
        if (rhs) rhs[r] = 0.0;
    }
}

// Dirichlet rows in the DIA (lattice numbering)
template <typename TM>
__global__ void k_dirichlet_dia(int64_t n, int nd, int centre, const uint8_t* dir, TM* dia) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if (!dir[i]) continue;
        for (int d = 0; d < nd; ++d) dia[dia_tiled_index(d, i, nd)] = (TM)(d == centre ? 1.0 : 0.0);
    }
}

// the zero halos of up to five level vectors (n entries between h and h zeros)
template <typename T>
__global__ __launch_bounds__(256) void k_zero_halos(int64_t n, int64_t h, T* a, T* b, T* c, T* d, T* e) {
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (i >= 2 * h) return;
    const int64_t j = i < h ? i : n + i;
    a[j] = b[j] = c[j] = d[j] = e[j] = (T)0;
}

// convert DIA values between precisions
template <typename TA, typename TB>
__global__ __launch_bounds__(256) void k_convert(int64_t n, const TA* a, TB* b) {
    UGX_STREAM_LOOP(n) {
        TA av[kStreamE];
#pragma unroll
        for (int e = 0; e < kStreamE; ++e) av[e] = ldnt(a + UGX_STREAM_SAFE(e, n));
#pragma unroll
        for (int e = 0; e < kStreamE; ++e)
            if (UGX_STREAM_IDX(e) < n) stnt((TB)av[e], b + UGX_STREAM_IDX(e));
    }
}

// Dirichlet flag per lattice point of a level: boundary of the unit box/square
__global__ void k_boundary_flags(int dim, int W, int64_t n, uint8_t* dir) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % W), y = (int)((i / W) % W);
        bool b = x == 0 || y == 0 || x == W - 1 || y == W - 1;
        if (dim == 3) {
            const int z = (int)(i / ((int64_t)W * W));
            b = b || z == 0 || z == W - 1;
        }
        dir[i] = b ? 1 : 0;
    }
}

// ---------------------------------------------------------------------------
// exported launchers
// ---------------------------------------------------------------------------

#define UGX_CHECK_LAUNCH() return hipGetLastError() == hipSuccess ? 0 : -1

template <typename TM, typename TV>
int spmv_csr(int64_t nrows, const int32_t* rowptr, const int32_t* col, const TM* val, double alpha, const TV* v1,
             double beta, const TV* w, TV* dest, int mode, int lanes, hipStream_t s) {
    return launch_spmv_csr<TM, TV>(nrows, rowptr, col, val, alpha, v1, beta, w, dest, mode, lanes, s);
}
template int spmv_csr<double, double>(int64_t, const int32_t*, const int32_t*, const double*, double, const double*, double, const double*, double*, int, int, hipStream_t);
template int spmv_csr<float, float>(int64_t, const int32_t*, const int32_t*, const float*, double, const float*, double, const float*, float*, int, int, hipStream_t);
template int spmv_csr<float, double>(int64_t, const int32_t*, const int32_t*, const float*, double, const double*, double, const double*, double*, int, int, hipStream_t);

template <typename T>
int vec_set(int64_t n, T* x, double v, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_set<T>, dim3(stream_grid(n)), dim3(256), 0, s, n, x, (T)v);
    UGX_CHECK_LAUNCH();
}
template int vec_set<double>(int64_t, double*, double, hipStream_t);
template int vec_set<float>(int64_t, float*, double, hipStream_t);
template int vec_set<uint8_t>(int64_t, uint8_t*, double, hipStream_t);
template int vec_set<int32_t>(int64_t, int32_t*, double, hipStream_t);

template <typename T>
int vec_scale_add(int64_t n, T* dest, double a1, const T* v1, double a2, const T* v2, double a3, const T* v3,
                  hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_scale_add<T>, dim3(stream_grid(n)), dim3(256), 0, s, n, dest, a1, v1, a2, v2, a3, v3);
    UGX_CHECK_LAUNCH();
}
template int vec_scale_add<double>(int64_t, double*, double, const double*, double, const double*, double, const double*, hipStream_t);
template int vec_scale_add<float>(int64_t, float*, double, const float*, double, const float*, double, const float*, hipStream_t);

template <typename TD, typename TV>
int diag_mult(int64_t n, TV* dest, const TD* d, const TV* x, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_diag_mult<TD, TV>), dim3(stream_grid(n)), dim3(256), 0, s, n, dest, d, x);
    UGX_CHECK_LAUNCH();
}
template int diag_mult<double, double>(int64_t, double*, const double*, const double*, hipStream_t);
template int diag_mult<float, float>(int64_t, float*, const float*, const float*, hipStream_t);

template <typename TM, typename TD>
int jacobi_diag_csr(int64_t n, const int32_t* rowptr, const int32_t* col, const TM* val, double omega, TD* dinv,
                    int* bad, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_jacobi_diag_csr<TM, TD>), dim3(vec_grid(n)), dim3(256), 0, s, n, rowptr, col, val, omega, dinv, bad);
    UGX_CHECK_LAUNCH();
}
template int jacobi_diag_csr<double, double>(int64_t, const int32_t*, const int32_t*, const double*, double, double*, int*, hipStream_t);

template <typename T>
int dot(int64_t n, const T* a, const T* b, double* partial, double* out, bool take_sqrt, hipStream_t s) {
    const int g = red_grid(n);
    hipLaunchKernelGGL(k_dot_partial<T>, dim3(g), dim3(256), 0, s, n, a, b, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, g, partial, out, take_sqrt ? 1 : 0);
    UGX_CHECK_LAUNCH();
}
template int dot<double>(int64_t, const double*, const double*, double*, double*, bool, hipStream_t);

int count_nonzero(int64_t n, const double* a, double* partial, double* out, hipStream_t s) {
    const int g = red_grid(n);
    hipLaunchKernelGGL(k_nonzero_partial, dim3(g), dim3(256), 0, s, n, a, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, g, partial, out, 0);
    UGX_CHECK_LAUNCH();
}

int dot_partials(int64_t n) { return red_grid(n); }

int sum_partials(int np, const double* partial, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, np, partial, out, 0);
    UGX_CHECK_LAUNCH();
}
int cg_update(int64_t n, double* sc, const double* p, const double* q, double* x, double* r, double* partial,
              double* host, hipStream_t s, float* rf, int nl, const double* lpart) {
    const int g = red_grid(n);
    hipLaunchKernelGGL(k_cg_update, dim3(g), dim3(256), 0, s, n, sc, p, q, x, r, partial, rf, nl, lpart);
    hipLaunchKernelGGL(k_cg_norm, dim3(1), dim3(1024), 0, s, g, partial, sc, host);
    UGX_CHECK_LAUNCH();
}
// every workgroup of the update reads the partials again. One MI355X: 65^3
// (580,000 reads) 6.9 us against 5.6 with a sum of 3.0 before it; 129^3 (4.3
// million) 21.1 against 18.1 and 4.1, no gain
bool cg_update_sums(int64_t n, int nl) { return (int64_t)red_grid(n) * nl <= (1 << 20); }
int cg_direction(int64_t n, const double* sc, double* p, const double* z, hipStream_t s) {
    hipLaunchKernelGGL(k_cg_direction, dim3(stream_grid(n)), dim3(256), 0, s, n, sc, p, z);
    UGX_CHECK_LAUNCH();
}
template <typename T>
int convert_dot(int64_t n, const T* c, double* z, const double* r, double* partial, double* out, hipStream_t s) {
    const int g = red_grid(n);
    hipLaunchKernelGGL(k_convert_dot<T>, dim3(g), dim3(256), 0, s, n, c, z, r, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, g, partial, out, 0);
    UGX_CHECK_LAUNCH();
}
template int convert_dot<float>(int64_t, const float*, double*, const double*, double*, double*, hipStream_t);
template int convert_dot<double>(int64_t, const double*, double*, const double*, double*, double*, hipStream_t);
template int dot<float>(int64_t, const float*, const float*, double*, double*, bool, hipStream_t);

template <typename TS, typename TL>
int permute_to(int64_t n, const int32_t* dof_of_lat, const TS* src, TL* dst, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_permute_to<TS, TL>), dim3(stream_grid(n)), dim3(256), 0, s, n, dof_of_lat, src, dst);
    UGX_CHECK_LAUNCH();
}
template int permute_to<double, double>(int64_t, const int32_t*, const double*, double*, hipStream_t);
template int permute_to<double, float>(int64_t, const int32_t*, const double*, float*, hipStream_t);
int permute_to_dual(int64_t n, const int32_t* dof_of_lat, const double* src, double* dst, float* dst32, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_permute_to_dual, dim3(stream_grid(n)), dim3(256), 0, s, n, dof_of_lat, src, dst, dst32);
    UGX_CHECK_LAUNCH();
}

template <typename TL, typename TS>
int permute_add_from(int64_t n, const int32_t* lat_of_dof, const TL* src, TS* dst, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_permute_add_from<TL, TS>), dim3(stream_grid(n)), dim3(256), 0, s, n, lat_of_dof, src, dst);
    UGX_CHECK_LAUNCH();
}
template int permute_add_from<double, double>(int64_t, const int32_t*, const double*, double*, hipStream_t);
template int permute_add_from<float, double>(int64_t, const int32_t*, const float*, double*, hipStream_t);

static DiaOffsets make_offsets(const int32_t* off, int nd) {
    DiaOffsets o;
    for (int d = 0; d < 27; ++d) o.off[d] = d < nd ? off[d] : 0;
    return o;
}

static inline int64_t remapped_grid(int64_t nblocks) { return nblocks < 64 ? nblocks : ((nblocks + 7) / 8) * 8; }

// Row schedule for a DIA launch over n rows with offsets `off`: banded when
// the operator is a full 3D lattice (27 diagonals, n = W^3) wide enough for
// the bands to matter, flat otherwise. Returns the grid size.
static int64_t make_row_map(int64_t n, int nd, const int32_t* off, RowMap& m) {
    m = RowMap{};
    m.nblocks = (n + 255) / 256;
    if (nd == 27) {
        const int64_t W = (int64_t)off[25] - off[22];
        const int64_t plane = off[22];
        if (W >= 128 && plane == W * W && n == W * W * W) {
            int64_t maxcps = 0;
            for (int c = 0; c < 8; ++c) {
                const int64_t j0 = c * W / 8, j1 = (c + 1) * W / 8;
                m.lo[c] = (int32_t)(j0 * W);
                m.len[c] = (int32_t)((j1 - j0) * W);
                m.cps[c] = (int32_t)((m.len[c] + 255) / 256);
                maxcps = m.cps[c] > maxcps ? m.cps[c] : maxcps;
            }
            m.plane = plane;
            m.nplanes = W;
            return 8 * maxcps * W;
        }
    }
    return remapped_grid(m.nblocks);
}

// LDS-staged launch plan for symmetric 27-point operators on full 3D lattices:
// bands of TY lines, grouped per XCD. Returns the grid size, 0 if not eligible.
// Lattices below min_w keep the unstaged kernels: at 65^3 the rows' 81 loads come
// from the caches, and only the FP64 Jacobi step, with two vectors of 8 bytes
// around every row, gains by staging (14.7 -> 12.2 us; FP32 7.2 -> 9.5, FP64
// d -= A x 10.6 -> 11.3, one MI355X). Three lines of 65 rows fill a workgroup
// once.
static int64_t make_staged_map(int64_t n, int nd, const int32_t* off, size_t elem, StagedMap& m, size_t& lds,
                               int min_w = 128) {
    if (nd != 27) return 0;
    const int64_t W = (int64_t)off[25] - off[22];
    if (W < min_w || off[22] != W * W || n != W * W * W) return 0;
    m = StagedMap{};
    m.W = (int32_t)W;
    m.TY = W < 128 ? 3 : 4;
    const int64_t nb = (W + m.TY - 1) / m.TY;
    int32_t maxg = 0;
    for (int c = 0; c < 8; ++c) {
        const int64_t b0 = c * nb / 8, b1 = (c + 1) * nb / 8;
        m.glo[c] = (int32_t)b0;
        m.gsz[c] = (int32_t)(b1 - b0);
        maxg = m.gsz[c] > maxg ? m.gsz[c] : maxg;
    }
    m.maxg = maxg;
    lds = (size_t)3 * (size_t)(m.TY * W + 2 * W + 2) * elem;
    if (lds > 64 * 1024) return 0;
    return 8 * (int64_t)maxg * W;
}

// workgroups of `kernel` (256 threads, `lds` bytes of LDS) resident on one CU,
// and the device's CU count; both asked once and kept
int resident_blocks(const void* kernel, size_t lds) {
    static std::mutex mu;
    static std::vector<std::pair<std::pair<const void*, size_t>, int>> cache;
    std::lock_guard<std::mutex> lock(mu);
    for (const auto& e : cache)
        if (e.first.first == kernel && e.first.second == lds) return e.second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, 256, lds) != hipSuccess || nb < 1) nb = 1;
    cache.push_back({{kernel, lds}, nb});
    return nb;
}
int device_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8)
            n = 8;
        cus = n;
    }
    return cus;
}

// matrix-free launch plan: bands of 4 lines grouped per XCD (any W >= 3)
static int64_t make_mf_map(int W, size_t elem, MfMap& m, size_t& lds) {
    m = MfMap{};
    m.W = W;
    m.TY = 4;
    const int64_t nb = (W + m.TY - 1) / m.TY;
    int32_t maxg = 0;
    for (int c = 0; c < 8; ++c) {
        const int64_t b0 = c * nb / 8, b1 = (c + 1) * nb / 8;
        m.glo[c] = (int32_t)b0;
        m.gsz[c] = (int32_t)(b1 - b0);
        maxg = m.gsz[c] > maxg ? m.gsz[c] : maxg;
    }
    const int64_t S = (int64_t)m.TY * W + 2 * W + 2;
    lds = (size_t)(3 * S + 2 * (int64_t)(m.TY + 1) * (W + 1)) * elem;
    return 8 * (int64_t)maxg * W;
}

#define UGX_DIA_DISPATCH(KERNEL, ...)                                                                      \
    do {                                                                                                  \
        RowMap rm;                                                                                        \
        const int64_t grid = make_row_map(n, nd, off, rm);                                                \
        if (nd == 27)                                                                                     \
            hipLaunchKernelGGL((KERNEL<TM, TV, 27>), dim3(grid), dim3(256), 0, s, __VA_ARGS__, rm);       \
        else if (nd == 9)                                                                                 \
            hipLaunchKernelGGL((KERNEL<TM, TV, 9>), dim3(grid), dim3(256), 0, s, __VA_ARGS__, rm);        \
        else                                                                                              \
            return -1;                                                                                    \
    } while (0)

template <typename TM>
int dia_symmetrize(int64_t n, int nd, const int32_t* off, const uint8_t* dir, const TM* full, TM* up, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_dia_symmetrize<TM>, dim3(vec_grid(n)), dim3(256), 0, s, n, nd, make_offsets(off, nd), dir, full, up);
    UGX_CHECK_LAUNCH();
}
template int dia_symmetrize<double>(int64_t, int, const int32_t*, const uint8_t*, const double*, double*, hipStream_t);

template <typename TM, typename TV>
int dias_apply_sub(int64_t n, int nd, const int32_t* off, const TM* U, const TV* x, const TV* d_in, TV* d_out,
                   hipStream_t s) {
    if (n <= 0) return 0;
    StagedMap sm;
    size_t lds = 0;
    typedef typename Acc<TV>::type T;
    if (const int64_t grid = make_staged_map(n, nd, off, sizeof(T), sm, lds)) {
        hipLaunchKernelGGL((k_dias27_staged_apply_sub<TM, TV>), dim3(grid), dim3(256), lds, s, n, make_offsets(off, nd), sm, U, x, d_in, d_out);
        UGX_CHECK_LAUNCH();
    }
    UGX_DIA_DISPATCH(k_dias_apply_sub, n, make_offsets(off, nd), U, x, d_in, d_out);
    UGX_CHECK_LAUNCH();
}
template int dias_apply_sub<double, double>(int64_t, int, const int32_t*, const double*, const double*, const double*, double*, hipStream_t);
template int dias_apply_sub<float, float>(int64_t, int, const int32_t*, const float*, const float*, const float*, float*, hipStream_t);

template <typename TM, typename TV>
int dias_axpy(int64_t n, int nd, const int32_t* off, const TM* U, double alpha, const TV* v, double beta, const TV* x,
              TV* y, hipStream_t s) {
    if (n <= 0) return 0;
    StagedMap sm;
    size_t lds = 0;
    typedef typename Acc<TV>::type T;
    if (const int64_t grid = make_staged_map(n, nd, off, sizeof(T), sm, lds)) {
        hipLaunchKernelGGL((k_dias27_staged_axpy<TM, TV>), dim3(grid), dim3(256), lds, s, n, make_offsets(off, nd), sm, U, alpha, v, beta, x, y);
        UGX_CHECK_LAUNCH();
    }
    UGX_DIA_DISPATCH(k_dias_axpy, n, make_offsets(off, nd), U, alpha, v, beta, x, y);
    UGX_CHECK_LAUNCH();
}
template int dias_axpy<double, double>(int64_t, int, const int32_t*, const double*, double, const double*, double, const double*, double*, hipStream_t);

template <typename TL, typename TS>
int permute_from(int64_t n, const int32_t* lat_of_dof, const TL* src, TS* dst, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_permute_from<TL, TS>), dim3(stream_grid(n)), dim3(256), 0, s, n, lat_of_dof, src, dst);
    UGX_CHECK_LAUNCH();
}
template int permute_from<double, double>(int64_t, const int32_t*, const double*, double*, hipStream_t);
template <typename TL, typename TS>
int permute_scatter(int64_t n, const int32_t* dof_of_lat, const TL* src, TS* dst, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_permute_scatter<TL, TS>), dim3(stream_grid(n)), dim3(256), 0, s, n, dof_of_lat, src, dst);
    UGX_CHECK_LAUNCH();
}
template int permute_scatter<double, double>(int64_t, const int32_t*, const double*, double*, hipStream_t);

template <typename TM, typename TV>
int dias_jacobi_step(int64_t n, int nd, const int32_t* off, const TM* U, const TV* dinv, const TV* sd_in, TV* sd_out,
                     TV* sc, hipStream_t s) {
    if (n <= 0) return 0;
    StagedMap sm;
    size_t lds = 0;
    typedef typename Acc<TV>::type T;
    if (const int64_t grid = make_staged_map(n, nd, off, sizeof(T), sm, lds, sizeof(T) == 8 ? 64 : 128)) {
        hipLaunchKernelGGL((k_dias27_staged_jacobi_step<TM, TV>), dim3(grid), dim3(256), lds, s, n, make_offsets(off, nd), sm, U, dinv, sd_in, sd_out, sc);
        UGX_CHECK_LAUNCH();
    }
    UGX_DIA_DISPATCH(k_dias_jacobi_step, n, make_offsets(off, nd), U, dinv, sd_in, sd_out, sc);
    UGX_CHECK_LAUNCH();
}
template int dias_jacobi_step<double, double>(int64_t, int, const int32_t*, const double*, const double*, const double*, double*, double*, hipStream_t);
template int dias_jacobi_step<float, float>(int64_t, int, const int32_t*, const float*, const float*, const float*, float*, float*, hipStream_t);

template <typename T>
int q1mf_planes_jacobi_step(int W, const T* cell, const T* dinv, const T* sd_in, T* sd_out, T* sc, hipStream_t s) {
    MfMap m;
    size_t lds;
    const int64_t grid = make_mf_map(W, sizeof(T), m, lds);
    if (lds > 64 * 1024) return -1;
    hipLaunchKernelGGL(k_q1mf_jacobi_step<T>, dim3(grid), dim3(256), lds, s, m, cell, dinv, sd_in, sd_out, sc);
    UGX_CHECK_LAUNCH();
}
template int q1mf_planes_jacobi_step<float>(int, const float*, const float*, const float*, float*, float*, hipStream_t);
template int q1mf_planes_jacobi_step<double>(int, const double*, const double*, const double*, double*, double*,
                                             hipStream_t);

template <typename T>
int q1mf_planes_apply_sub(int W, const T* cell, const T* x, const T* d_in, T* d_out, hipStream_t s) {
    MfMap m;
    size_t lds;
    const int64_t grid = make_mf_map(W, sizeof(T), m, lds);
    if (lds > 64 * 1024) return -1;
    hipLaunchKernelGGL(k_q1mf_apply_sub<T>, dim3(grid), dim3(256), lds, s, m, cell, x, d_in, d_out);
    UGX_CHECK_LAUNCH();
}
template int q1mf_planes_apply_sub<float>(int, const float*, const float*, const float*, float*, hipStream_t);
template int q1mf_planes_apply_sub<double>(int, const double*, const double*, const double*, double*, hipStream_t);

template <typename T>
int q1mf_planes_axpy(int W, const T* cell, double alpha, const T* v, double beta, const T* x, T* y, hipStream_t s) {
    MfMap m;
    size_t lds;
    const int64_t grid = make_mf_map(W, sizeof(T), m, lds);
    if (lds > 64 * 1024) return -1;
    hipLaunchKernelGGL(k_q1mf_axpy<T>, dim3(grid), dim3(256), lds, s, m, cell, alpha, v, beta, x, y);
    UGX_CHECK_LAUNCH();
}
template int q1mf_planes_axpy<double>(int, const double*, double, const double*, double, const double*, double*,
                                      hipStream_t);

template <typename T>
int q1mf_coeff(int64_t ne, double h, const double* theta, T* c, hipStream_t s) {
    hipLaunchKernelGGL(k_q1mf_coeff<T>, dim3(vec_grid(ne)), dim3(256), 0, s, ne, h, theta, c);
    UGX_CHECK_LAUNCH();
}
template int q1mf_coeff<float>(int64_t, double, const double*, float*, hipStream_t);
template int q1mf_coeff<double>(int64_t, double, const double*, double*, hipStream_t);

template <typename TM, typename TV>
int dia_apply_sub(int64_t n, int nd, const int32_t* off, const TM* A, const TV* x, const TV* d_in, TV* d_out,
                  hipStream_t s) {
    if (n <= 0) return 0;
    UGX_DIA_DISPATCH(k_dia_apply_sub, n, make_offsets(off, nd), A, x, d_in, d_out);
    UGX_CHECK_LAUNCH();
}
template int dia_apply_sub<double, double>(int64_t, int, const int32_t*, const double*, const double*, const double*, double*, hipStream_t);
template int dia_apply_sub<float, float>(int64_t, int, const int32_t*, const float*, const float*, const float*, float*, hipStream_t);

template <typename TM, typename TV>
int dia_axpy(int64_t n, int nd, const int32_t* off, const TM* A, double alpha, const TV* v, double beta, const TV* x,
             TV* y, hipStream_t s) {
    if (n <= 0) return 0;
    UGX_DIA_DISPATCH(k_dia_axpy, n, make_offsets(off, nd), A, alpha, v, beta, x, y);
    UGX_CHECK_LAUNCH();
}
template int dia_axpy<double, double>(int64_t, int, const int32_t*, const double*, double, const double*, double, const double*, double*, hipStream_t);
template int dia_axpy<float, float>(int64_t, int, const int32_t*, const float*, double, const float*, double, const float*, float*, hipStream_t);

template <typename TM, typename TV>
int dia_jacobi_step(int64_t n, int nd, const int32_t* off, const TM* A, const TV* dinv, const TV* sd_in, TV* sd_out,
                    TV* sc, hipStream_t s) {
    if (n <= 0) return 0;
    UGX_DIA_DISPATCH(k_dia_jacobi_step, n, make_offsets(off, nd), A, dinv, sd_in, sd_out, sc);
    UGX_CHECK_LAUNCH();
}
template int dia_jacobi_step<double, double>(int64_t, int, const int32_t*, const double*, const double*, const double*, double*, double*, hipStream_t);
template int dia_jacobi_step<float, float>(int64_t, int, const int32_t*, const float*, const float*, const float*, float*, float*, hipStream_t);

template <typename TV>
int jacobi_accumulate(int64_t n, const TV* dinv, const TV* sd, TV* sc, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_jacobi_accumulate<TV>, dim3(stream_grid(n)), dim3(256), 0, s, n, dinv, sd, sc);
    UGX_CHECK_LAUNCH();
}
template int jacobi_accumulate<double>(int64_t, const double*, const double*, double*, hipStream_t);
template int jacobi_accumulate<float>(int64_t, const float*, const float*, float*, hipStream_t);

template <typename TV>
int jacobi_convert_dot(int64_t n, const TV* dinv, const TV* sd, const TV* sc, double* z, const double* r,
                       double* partial, double* out, hipStream_t s) {
    if (n <= 0) return 0;
    if (!out) {
        hipLaunchKernelGGL(k_jacobi_convert_dot<TV>, dim3(stream_grid(n)), dim3(256), 0, s, n, dinv, sd, sc, z, r,
                           (double*)nullptr);
        UGX_CHECK_LAUNCH();
    }
    const int g = red_grid(n);
    hipLaunchKernelGGL(k_jacobi_convert_dot<TV>, dim3(g), dim3(256), 0, s, n, dinv, sd, sc, z, r, partial);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, g, partial, out, 0);
    UGX_CHECK_LAUNCH();
}
template int jacobi_convert_dot<double>(int64_t, const double*, const double*, const double*, double*, const double*,
                                        double*, double*, hipStream_t);
template int jacobi_convert_dot<float>(int64_t, const float*, const float*, const float*, double*, const double*,
                                       double*, double*, hipStream_t);

template <typename TM, typename TV>
int dia_jacobi_diag(int64_t n, int nd, const TM* dia, double omega, TV* dinv, int* bad, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_dia_jacobi_diag<TM, TV>), dim3(vec_grid(n)), dim3(256), 0, s, n, nd, dia, omega, dinv, bad);
    UGX_CHECK_LAUNCH();
}
template int dia_jacobi_diag<double, double>(int64_t, int, const double*, double, double*, int*, hipStream_t);

template <typename TV>
int prolong_add(int dim, int Wc, int Wf, int64_t n_f, const TV* scc, const uint8_t* dir_f, TV* st, TV* sc,
                hipStream_t s, const TV* dinv_c, const TV* sd_c) {
    if (n_f <= 0) return 0;
    if (n_f >= ((int64_t)1 << 32)) return -1;
    if ((dinv_c == nullptr) != (sd_c == nullptr)) return -1;
    if (dim == 2) return prolong2<TV>(Wc, Wf, scc, dinv_c, sd_c, dir_f, st, sc, s);
    const CoarseCorr<TV> corr{scc, dinv_c, sd_c};
    if (Wf == 2 * Wc - 1) {
        // measured on one MI355X within the 256^3 GMG-CG solve (both kernels
        // with XCD-grouped blocks): 129^3 -> 257^3 FP32 tiled 76 us against
        // 81 us for the per-coarse-point kernel, 65^3 -> 129^3 15 against
        // 13 us, the coarser levels 4.6-5.9 against 7.7-10 us; FP64 tiled
        // 94 us at the top
        constexpr int TY = TransferTile<TV>::TY;
        const size_t lds = prolong3_tiled_lds(Wc, sizeof(TV), TY);
        if (lds <= 64 * 1024) {
            const int nbands = (Wc + TY - 1) / TY;
            hipLaunchKernelGGL(k_prolong3_tiled<TV>, dim3((unsigned)remapped_grid((int64_t)Wf * nbands)), dim3(256), lds, s,
                               Wc, Wf, nbands, corr, st, sc, make_fastdiv((uint32_t)Wf));
            UGX_CHECK_LAUNCH();
        }
        const int64_t n_c = (int64_t)Wc * Wc * Wc;
        hipLaunchKernelGGL(k_prolong_add3<TV>, dim3(remapped_grid((n_c + 255) / 256)), dim3(256), 0, s, Wc, Wf, n_c, corr,
                           dir_f, st,
                           sc, make_fastdiv((uint32_t)Wc));
        UGX_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_prolong_add<TV>, dim3((n_f + 255) / 256), dim3(256), 0, s, Wc, Wf, n_f, corr, dir_f, st,
                       sc, make_fastdiv((uint32_t)Wf));
    UGX_CHECK_LAUNCH();
}
template int prolong_add<double>(int, int, int, int64_t, const double*, const uint8_t*, double*, double*, hipStream_t,
                                 const double*, const double*);
template int prolong_add<float>(int, int, int, int64_t, const float*, const uint8_t*, float*, float*, hipStream_t,
                                const float*, const float*);

// at most this many workgroups per CU are planned for (8 or 10, more and
// shorter chunks, measured 37.3 against 31.6 us at 257^3 -> 129^3)
constexpr int kRzResident = 7;

// plan of k_restrict3_z: 2-line bands (1-line when a staged plane would not
// fit the slots) grouped per XCD, chunks so that the grid is one round;
// returns the grid, 0 when the plan does not apply
template <typename TV>
static int64_t make_rz_map(int Wc, int Wf, RzMap& m, size_t& lds) {
    m = RzMap{};
    m.Wc = Wc;
    m.Wf = Wf;
    m.TY = 5 * (Wf + 2) <= kRzSlots * 256 ? 2 : 1;
    const int64_t PL = (int64_t)(2 * m.TY + 1) * (Wf + 2);
    if (PL > kRzSlots * 256 || Wc < 3) return 0;
    lds = (size_t)(3 * PL) * sizeof(TV);
    if (lds > 64 * 1024) return 0;
    const int64_t nb = (Wc + m.TY - 1) / m.TY;
    int32_t maxg = 0;
    for (int c = 0; c < 8; ++c) {
        const int64_t b0 = c * nb / 8, b1 = (c + 1) * nb / 8;
        m.glo[c] = (int32_t)b0;
        m.gsz[c] = (int32_t)(b1 - b0);
        maxg = m.gsz[c] > maxg ? m.gsz[c] : maxg;
    }
    if (maxg == 0) return 0;
    const int64_t slots = (int64_t)(device_cus() / 8) *
                          std::min(kRzResident, resident_blocks(reinterpret_cast<const void*>(&k_restrict3_z<TV>), lds));
    int64_t nch = slots / maxg;
    nch = std::min<int64_t>(std::max<int64_t>(nch, 1), std::max(1, Wc / 2));
    m.nchunks = (int32_t)nch;
    return 8 * (int64_t)maxg * m.nchunks;
}

template <typename TV>
int restrict_defect(int dim, int Wc, int Wf, int64_t n_c, const TV* sdf, const uint8_t* dir_c, const uint8_t* dir_f,
                    TV* sdc, hipStream_t s, TV* zero_c) {
    if (n_c <= 0) return 0;
    if (n_c >= ((int64_t)1 << 32)) return -1;
    if (dim == 2) return restrict2<TV>(Wc, Wf, sdf, dir_c, dir_f, sdc, zero_c, s);
    if (Wf == 2 * Wc - 1 && Wc >= 65) {
        // large levels: the z-marching restriction (short-lived staging
        // workgroups left the tiled kernel at about 1.1 TB/s at 257^3)
        RzMap rm;
        size_t rlds = 0;
        if (const int64_t grid = make_rz_map<TV>(Wc, Wf, rm, rlds)) {
            hipLaunchKernelGGL(k_restrict3_z<TV>, dim3((unsigned)grid), dim3(256), rlds, s, rm, sdf, sdc, zero_c);
            UGX_CHECK_LAUNCH();
        }
    }
    if (dim == 3 && Wf == 2 * Wc - 1) {
        // measured on one MI355X: 257^3 -> 129^3 FP32 59 / 60 us, FP64 65 / 74 us,
        // 33^3 -> 17^3 about 4 / 8 us against the per-coarse-point kernel
        constexpr int TY = TransferTile<TV>::TY;
        const size_t lds = restrict3_tiled_lds(Wf, sizeof(TV), TY);
        if (lds <= 64 * 1024) {
            const int nbands = (Wc + TY - 1) / TY;
            hipLaunchKernelGGL(k_restrict3_tiled<TV>, dim3((unsigned)remapped_grid((int64_t)Wc * nbands)), dim3(256), lds,
                               s, Wc,
                               Wf, nbands, sdf, sdc, zero_c);
            UGX_CHECK_LAUNCH();
        }
    }
    hipLaunchKernelGGL(k_restrict<TV>, dim3((n_c + 255) / 256), dim3(256), 0, s, Wc, Wf, n_c, sdf, dir_c, dir_f, sdc,
                       make_fastdiv((uint32_t)Wc), zero_c);
    UGX_CHECK_LAUNCH();
}
template int restrict_defect<double>(int, int, int, int64_t, const double*, const uint8_t*, const uint8_t*, double*,
                                     hipStream_t, double*);
template int restrict_defect<float>(int, int, int, int64_t, const float*, const uint8_t*, const uint8_t*, float*,
                                    hipStream_t, float*);

template <typename TV>
int lu_solve(int n, const double* LinvT, const double* UinvT, const int32_t* perm, const TV* b, TV* x, hipStream_t s) {
    if (n <= 0 || n > 4096) return -1;
    hipLaunchKernelGGL(k_lu_solve<TV>, dim3(1), dim3(1024), 2 * n * sizeof(double), s, n, LinvT, UinvT, perm, b, x);
    UGX_CHECK_LAUNCH();
}
template int lu_solve<double>(int, const double*, const double*, const int32_t*, const double*, double*, hipStream_t);

template int lu_solve<float>(int, const double*, const double*, const int32_t*, const float*, float*, hipStream_t);

int invert_map(int64_t n, const int32_t* dof_of_lat, int32_t* lat_of_dof, hipStream_t s) {
    hipLaunchKernelGGL(k_invert_map, dim3(vec_grid(n)), dim3(256), 0, s, n, dof_of_lat, lat_of_dof);
    UGX_CHECK_LAUNCH();
}

int pattern_count(int dim, int W, int64_t n, const int32_t* lat_of_dof, int32_t* cnt, hipStream_t s) {
    hipLaunchKernelGGL(k_pattern_count, dim3(vec_grid(n)), dim3(256), 0, s, dim, W, n, lat_of_dof, cnt);
    UGX_CHECK_LAUNCH();
}

template <typename TM>
int assemble_fv1_tri(int n, double h, const double* theta, int nfine, const double* f_at_dof, const int32_t* dof_of_lat,
                     const int32_t* rowptr, const int32_t* col, TM* csr_val, TM* dia, int64_t dia_n, double* rhs,
                     hipStream_t s) {
    const int hn = (n + 1) / 2;
    const int64_t per = (int64_t)hn * hn;
    for (int color = 0; color < 8; ++color)
        hipLaunchKernelGGL(k_assemble_fv1_tri<TM>, dim3((per + 127) / 128), dim3(128), 0, s, n, color, h, theta, nfine, f_at_dof, dof_of_lat, rowptr, col, csr_val, dia, dia_n, rhs);
    UGX_CHECK_LAUNCH();
}
template int assemble_fv1_tri<double>(int, double, const double*, int, const double*, const int32_t*, const int32_t*, const int32_t*, double*, double*, int64_t, double*, hipStream_t);

template <typename TM>
int dirichlet_csr(int64_t n, int64_t n_inner, const int32_t* rowptr, const int32_t* col, TM* val, double* rhs,
                  hipStream_t s) {
    if (n - n_inner <= 0) return 0;
    hipLaunchKernelGGL(k_dirichlet_csr<TM>, dim3(vec_grid(n - n_inner)), dim3(256), 0, s, n, n_inner, rowptr, col, val, rhs);
    UGX_CHECK_LAUNCH();
}
template int dirichlet_csr<double>(int64_t, int64_t, const int32_t*, const int32_t*, double*, double*, hipStream_t);

template <typename TM>
int dirichlet_dia(int64_t n, int nd, int centre, const uint8_t* dir, TM* dia, hipStream_t s) {
    hipLaunchKernelGGL(k_dirichlet_dia<TM>, dim3(vec_grid(n)), dim3(256), 0, s, n, nd, centre, dir, dia);
    UGX_CHECK_LAUNCH();
}
template int dirichlet_dia<double>(int64_t, int, int, const uint8_t*, double*, hipStream_t);

template <typename TA, typename TB>
int convert(int64_t n, const TA* a, TB* b, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL((k_convert<TA, TB>), dim3(stream_grid(n)), dim3(256), 0, s, n, a, b);
    UGX_CHECK_LAUNCH();
}
template int convert<double, float>(int64_t, const double*, float*, hipStream_t);
template int convert<float, double>(int64_t, const float*, double*, hipStream_t);
template int convert<double, double>(int64_t, const double*, double*, hipStream_t);

template <typename T>
int zero_halos(int64_t n, int64_t h, T* const (&v)[5], hipStream_t s) {
    if (h <= 0) return 0;
    hipLaunchKernelGGL(k_zero_halos<T>, dim3((unsigned)((2 * h + 255) / 256)), dim3(256), 0, s, n, h, v[0], v[1], v[2], v[3],
                       v[4]);
    UGX_CHECK_LAUNCH();
}
template int zero_halos<float>(int64_t, int64_t, float* const (&)[5], hipStream_t);
template int zero_halos<double>(int64_t, int64_t, double* const (&)[5], hipStream_t);

int boundary_flags(int dim, int W, int64_t n, uint8_t* dir, hipStream_t s) {
    hipLaunchKernelGGL(k_boundary_flags, dim3(vec_grid(n)), dim3(256), 0, s, dim, W, n, dir);
    UGX_CHECK_LAUNCH();
}

int sell_widths(int64_t nrows, const int32_t* rowptr, const int32_t* order, int32_t* width, hipStream_t s) {
    const int64_t nsl = (nrows + 63) / 64;
    if (nsl <= 0) return 0;
    hipLaunchKernelGGL(k_sell_widths, dim3((nsl + 255) / 256), dim3(256), 0, s, nrows, rowptr, order, width);
    UGX_CHECK_LAUNCH();
}

template <typename TM>
int sell_fill(int64_t nrows, int64_t ncols, const int32_t* rowptr, const int32_t* col, const TM* val,
              const int32_t* order, const int64_t* slice_ptr, const int32_t* width, int32_t* scol, TM* sval,
              hipStream_t s, bool vals_only) {
    const int64_t nsl = (nrows + 63) / 64;
    if (nsl <= 0) return 0;
    hipLaunchKernelGGL(k_sell_fill<TM>, dim3((unsigned)nsl), dim3(64), 0, s, nrows, ncols, rowptr, col, val, order,
                       slice_ptr, width, scol, sval, vals_only ? 1 : 0);
    UGX_CHECK_LAUNCH();
}
template int sell_fill<double>(int64_t, int64_t, const int32_t*, const int32_t*, const double*, const int32_t*,
                               const int64_t*, const int32_t*, int32_t*, double*, hipStream_t, bool);

// Several waves a slice where the slices do not fill the chip by themselves
// (fewer than 16 waves a CU). Rows of up to 125 entries: 568 slices 23.5 us with
// one wave, 14.9 with four, 18.3 with sixteen; 80 slices 13.0 with four and 11.0
// with sixteen, 12 slices 11.9 and 7.6: sixteen where a CU has at most one slice.
// Rows of up to 27 entries in a cycle: 7.5 - 9.2 us with one wave, 4.0 - 5.5 with
// four; a product keeps one wave there, whose two sums are those of the
// dictionary layout bit for bit.
static int sell_waves(int64_t nslices, int max_width, int min_width) {
    if (nslices >= (int64_t)device_cus() * 16 || max_width <= min_width) return 1;
    return max_width > 32 && nslices <= device_cus() ? 16 : 4;
}

template <typename TM, typename TV, int WAVES>
static void launch_sell_spmv(int64_t nrows, const int64_t* slice_ptr, const int32_t* width, const int32_t* scol,
                             const TM* sval, double alpha, const TV* v1, double beta, const TV* w, TV* dest, int mode,
                             const int32_t* rowptr, const int32_t* order, hipStream_t s) {
    const int64_t nsl = (nrows + 63) / 64, nb = WAVES == 1 ? (nsl + 3) / 4 : nsl;
    hipLaunchKernelGGL((k_sell_spmv<TM, TV, WAVES>), dim3(remapped_grid(nb)), dim3(sell_block(WAVES)), 0, s, nrows,
                       slice_ptr, width, scol, sval, alpha, v1, beta, w, dest, mode, rowptr, order, nb);
}

template <typename TM, typename TV>
int sell_spmv(int64_t nrows, const int64_t* slice_ptr, const int32_t* width, int max_width, const int32_t* scol,
              const TM* sval, double alpha, const TV* v1, double beta, const TV* w, TV* dest, int mode,
              const int32_t* rowptr, const int32_t* order, hipStream_t s) {
    if (nrows <= 0) return 0;
    const int waves = sell_waves((nrows + 63) / 64, max_width, 32);
    auto* f = waves == 16  ? &launch_sell_spmv<TM, TV, 16>
              : waves == 4 ? &launch_sell_spmv<TM, TV, 4>
                           : &launch_sell_spmv<TM, TV, 1>;
    f(nrows, slice_ptr, width, scol, sval, alpha, v1, beta, w, dest, mode, rowptr, order, s);
    UGX_CHECK_LAUNCH();
}
template int sell_spmv<double, double>(int64_t, const int64_t*, const int32_t*, int, const int32_t*, const double*,
                                       double, const double*, double, const double*, double*, int, const int32_t*,
                                       const int32_t*, hipStream_t);

template <int WAVES>
static void launch_sell_cycle(int64_t nrows, const int64_t* slice_ptr, const int32_t* width, const int32_t* scol,
                              const double* sval, const double* w, const int32_t* rowptr, const int32_t* order,
                              const SellEpilogue& e, hipStream_t s) {
    const int64_t nsl = (nrows + 63) / 64, nb = WAVES == 1 ? (nsl + 3) / 4 : nsl;
    hipLaunchKernelGGL(k_sell_cycle<WAVES>, dim3(remapped_grid(nb)), dim3(sell_block(WAVES)), 0, s, nrows, slice_ptr,
                       width, scol, sval, w, rowptr, order, nb, e);
}

int sell_cycle(int64_t nrows, const int64_t* slice_ptr, const int32_t* width, int max_width, const int32_t* scol,
               const double* sval, const double* w, const int32_t* rowptr, const int32_t* order,
               const SellEpilogue& e, hipStream_t s) {
    if (nrows <= 0) return 0;
    const int waves = sell_waves((nrows + 63) / 64, max_width, 8);
    auto* f = waves == 16 ? &launch_sell_cycle<16> : waves == 4 ? &launch_sell_cycle<4> : &launch_sell_cycle<1>;
    f(nrows, slice_ptr, width, scol, sval, w, rowptr, order, e, s);
    UGX_CHECK_LAUNCH();
}

int adjoint_grad_q1_hex(int n, double h, const double* theta, const int32_t* dof_of_lat, int64_t n_inner,
                        const double* u, const double* lambda, double* grad, hipStream_t s) {
    const int64_t ne = (int64_t)n * n * n;
    if (ne <= 0) return 0;
    hipLaunchKernelGGL(k_adjoint_grad_q1_hex, dim3((ne + 127) / 128), dim3(128), 0, s, n, h, theta, dof_of_lat, n_inner, u, lambda, grad);
    UGX_CHECK_LAUNCH();
}

int zero_range(int64_t lo, int64_t hi, double* x, hipStream_t s) {
    if (hi <= lo) return 0;
    hipLaunchKernelGGL(k_zero_range, dim3(vec_grid(hi - lo)), dim3(256), 0, s, lo, hi, x);
    UGX_CHECK_LAUNCH();
}

}  // namespace ugamd
