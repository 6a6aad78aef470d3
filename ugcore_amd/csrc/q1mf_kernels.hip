// Matrix-free Q1 operator of a uniformly refined cube with a coefficient that
// is constant per element (the top level of the hexahedral hierarchy):
// A = sum_e c_e K_ref with c_e = h k_e and the unit-cube Q1 stiffness K_ref
// (diagonal 1/3, face diagonals -1/12, body diagonal -1/12, couplings along
// element edges 0), so for an interior row
//   (A x)_i = sum_{8 cells e at i} c_e (x_i/3 - (x_f1 + x_f2 + x_f3 + x_b)/12)
// with f1..f3 the face-diagonal and b the body-diagonal corner of e seen from
// i. Boundary (Dirichlet) rows are identity rows. The products equal those of
// the Dirichlet-eliminated stored operator on vectors vanishing on Dirichlet
// DoFs, up to rounding (the assembled entries carry quadrature round-off).
//
// The smoothing steps, defect updates and CG operator applications of a solve
// are modes of one row function (Q1Mode) in two schedules:
//   * k_q1mf_march (129^3 and 257^3): workgroups march through planes;
//   * k_q1mf_direct (up to 65^3): one row per thread, straight from the caches.
// 513^3 keeps the plane-by-plane kernels of kernels.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ugx_internal.hpp"

namespace ugamd {

namespace {

// MODE 0: fused Jacobi step (staged st = dinv.*sd; sd_out = sd - A st; sc += st):
//         a = dinv, b = sd, out0 = sd_out, out1 = sc
// MODE 1: d_out = d_in - A x: a = x, c = d_in, out0 = d_out
// MODE 2: y = alpha v + beta A x: a = x, c = v, out0 = y; partials of (y, x)
// MODE 3: the first Jacobi step of a cycle from the FP64 defect d64 and a zero
//         correction: sd = (T)d64, st = dinv.*sd; sd_out = sd - A st; sc = st
// MODE 4: the same from a defect already in T (b = sd)
// MODE 5: the CG direction update fused with the operator: staged
//         p_new = fma(beta, p_old, z) (a = p_old, b = z, beta = *d64, or
//         *d64 / *c where c is given),
//         out1 = p_new, out0 = y = A p_new, partials of (y, p_new)
// MODE 7: the last post-smoothing step of a cycle fused with the correction
//         update that ends it, its conversion and the (z, r) partials: MODE 0
//         (a = dinv, b = sd, c = sc) without storing sd_out or sc, then
//         z64 = (double)(sc_new + dinv .* sd_out) with the arithmetic of
//         k_jacobi_convert_dot (d64 = r)
// MODE 6: the coarse grid correction and the defect update after it: staged
//         t = P c_coarse (a = the coarse correction; with b, c2 its last update
//         a + b .* c2 folded in), d_out = d_in - A t, sc += t: c = d_in,
//         out0 = d_out, out1 = sc (k_q1mf_march only)
// out0 may alias c (MODE 1, 2, 6): every row is read and then written by the same
// thread. Every access is an ordinary one: a line of 257 values begins and ends
// inside a cache line, which the next line's wave completes, and nontemporal
// stores sent it out in parts (1.12 - 1.15 of the bytes; 256^3 solve 8.93 ms, 8.79
// so; 128^3 FP64 2.79 and 2.69; the rows' inputs were nontemporal too).
template <typename T>
struct Q1Args {
    const T* cell;
    const T* a;
    const T* b;
    const T* c;
    T* out0;
    T* out1;
    double alpha, beta;
    double* partial;
    const double* d64;
    double* z64;
    const T* c2;
};

// the value that entry j contributes to its neighbours' rows, from its two
// loaded parts
template <typename T, int MODE>
__device__ __forceinline__ void raw_staged(const Q1Args<T>& q, int64_t j, T& va, T& vb) {
    va = q.a[j];
    if (MODE == 0 || MODE == 4 || MODE == 5 || MODE == 7) vb = q.b[j];
    if (MODE == 3) vb = (T)q.d64[j];
}
template <typename T, int MODE>
__device__ __forceinline__ T combine(T va, T vb, T bcg) {
    if (MODE == 0 || MODE == 3 || MODE == 4 || MODE == 7) return va * vb;
    if (MODE == 5) return (T)fma((double)bcg, (double)va, (double)vb);
    return va;
}

// a row's own inputs
template <typename T>
struct RowIn {
    T u, v, w;
    double r;
};
template <typename T, int MODE>
__device__ __forceinline__ void load_row(const Q1Args<T>& q, int64_t i, bool ok, RowIn<T>& in) {
    if (!ok) return;
    if (MODE == 0) {
        in.u = q.b[i];      // sd
        in.v = q.out1[i];   // sc
    } else if (MODE == 1) {
        in.u = q.c[i];
    } else if (MODE == 6) {
        in.u = q.c[i];
        in.v = q.out1[i];
    } else if (MODE == 2) {
        in.u = q.alpha != 0.0 ? q.c[i] : (T)0;
    } else if (MODE == 3) {
        in.u = (T)q.d64[i];
    } else if (MODE == 4) {
        in.u = q.b[i];
    } else if (MODE == 7) {
        in.u = q.b[i];   // sd
        in.v = q.c[i];   // sc
        in.w = q.a[i];         // dinv
        in.r = q.partial ? q.d64[i] : 0.0;
    }
}
template <typename T, int MODE>
__device__ __forceinline__ void store_row(const Q1Args<T>& q, int64_t i, const RowIn<T>& in, T xi, T s, double& dot) {
    if (MODE == 0 || MODE == 6) {
        q.out0[i] = in.u - s;
        q.out1[i] = in.v + xi;
    } else if (MODE == 3 || MODE == 4) {
        q.out0[i] = in.u - s;
        q.out1[i] = xi;
    } else if (MODE == 1) {
        q.out0[i] = in.u - s;
    } else if (MODE == 7) {
        const T sd = in.u - s, sc = in.v + xi;
        const double z = (double)(T)((double)sc + (double)in.w * (double)sd);
        q.z64[i] = z;
        dot += z * in.r;
    } else {
        const T y = (T)((q.alpha == 0.0 ? 0.0 : q.alpha * (double)in.u) + q.beta * (double)s);
        q.out0[i] = y;
        if (MODE == 5) q.out1[i] = xi;
        dot += (double)y * (double)xi;
    }
}

// The layer of cells between two planes at one column: c[b][a] its four cells
// (y, x), P and Q the 3x3 values around the column on the lower and the upper
// plane. The lower row's neighbours across the layer are Q's, the upper row's
// are P's; both share the eight diagonal products d (body diagonals and
// in-plane face diagonals), and each adds the four face-diagonal products with
// the other plane's edge midpoints (weights: pairs of cells): eq for the lower
// row, ep for the upper one. 21 multiply-adds per row and layer where the row
// sums formed one by one took 43 a row.
template <typename T>
__device__ __forceinline__ void q1_layer(T c00, T c01, T c10, T c11, const T* P0, const T* P1, const T* P2,
                                         const T* Q0, const T* Q1, const T* Q2, T& d, T& ep, T& eq, T& cs) {
    const T x0 = c00 + c10, x1 = c01 + c11, y0 = c00 + c01, y1 = c10 + c11;
    d = c00 * P0[0];
    d = fma(c01, P0[2], d);
    d = fma(c10, P2[0], d);
    d = fma(c11, P2[2], d);
    d = fma(c00, Q0[0], d);
    d = fma(c01, Q0[2], d);
    d = fma(c10, Q2[0], d);
    d = fma(c11, Q2[2], d);
    ep = x0 * P1[0];
    ep = fma(x1, P1[2], ep);
    ep = fma(y0, P0[1], ep);
    ep = fma(y1, P2[1], ep);
    eq = x0 * Q1[0];
    eq = fma(x1, Q1[2], eq);
    eq = fma(y0, Q0[1], eq);
    eq = fma(y1, Q2[1], eq);
    cs = x0 + x1;
}
// the row's value from the sums of the layers below and above it
template <typename T>
__device__ __forceinline__ T q1_row(T off_below, T off_above, T cs_below, T cs_above, T xi) {
    const T off = off_below + off_above, t = (cs_below + cs_above) * xi;
    return fma(t, (T)(1.0 / 3.0), -(off * (T)(1.0 / 12.0)));
}

__device__ __forceinline__ void block_dot(double v, double* partial) {
    __shared__ double sh[4];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}
template <int MODE>
constexpr bool has_dot() {
    return MODE == 2 || MODE == 5 || MODE == 7;
}

// One row per thread: on these lattices (up to 275 k rows, 1 - 17 waves a CU)
// the vectors and coefficients sit in the caches and a launch is one exposed
// latency, while a march is a chain of them, one per plane (65^3, FP32 step:
// 12.8 us marching, 5.2 us here; 33^3: 9.5 and 2.8 us).
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_q1mf_direct(int W, int64_t nblocks, Q1Args<T> q) {
    const int n = W - 1, W2 = W * W;
    // consecutive rows on one XCD
    const int64_t per = nblocks / 8;   // the grid is a multiple of 8
    const int64_t lb = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int i = (int)(lb * 256) + (int)threadIdx.x;
    double dot = 0.0;
    if (i < W2 * W) {
        const T bcg = MODE == 5 ? (T)(q.c ? *q.d64 / (double)*q.c : *q.d64) : (T)0;
        const int yz = i / W, x = i - yz * W, z = yz / W, y = yz - z * W;
        RowIn<T> in{};
        load_row<T, MODE>(q, i, true, in);
        T xi, s;
        if (x == 0 || y == 0 || z == 0 || x == n || y == n || z == n) {
            T va, vb = (T)0;
            raw_staged<T, MODE>(q, i, va, vb);
            xi = combine<T, MODE>(va, vb, bcg);
            s = xi;
        } else {
            T X[3][3][3], B[3][3][3], C[2][2][2];
#pragma unroll
            for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        if (dz == 1 && (dy == 1) != (dx == 1)) continue;   // the row's plane: no edge neighbours
                        raw_staged<T, MODE>(q, i + (dz - 1) * W2 + (dy - 1) * W + dx - 1, X[dz][dy][dx], B[dz][dy][dx]);
                    }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int a = 0; a < 2; ++a) C[c][b][a] = q.cell[((z - 1 + c) * n + y - 1 + b) * n + x - 1 + a];
#pragma unroll
            for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        if (dz == 1 && (dy == 1) != (dx == 1)) X[dz][dy][dx] = (T)0;   // not used
                        else X[dz][dy][dx] = combine<T, MODE>(X[dz][dy][dx], B[dz][dy][dx], bcg);
                    }
            T db, epb, eqb, cb, da, epa, eqa, ca;
            q1_layer<T>(C[0][0][0], C[0][0][1], C[0][1][0], C[0][1][1], X[0][0], X[0][1], X[0][2], X[1][0], X[1][1],
                        X[1][2], db, epb, eqb, cb);
            q1_layer<T>(C[1][0][0], C[1][0][1], C[1][1][0], C[1][1][1], X[1][0], X[1][1], X[1][2], X[2][0], X[2][1],
                        X[2][2], da, epa, eqa, ca);
            xi = X[1][1][1];
            s = q1_row<T>(db + epb, da + eqa, cb, ca, xi);
        }
        store_row<T, MODE>(q, i, in, xi, s, dot);
    }
    if (has_dot<MODE>() && q.partial) block_dot(dot, q.partial);
}

// z-march. A workgroup of 256 threads owns TY lines of a chunk of planes; a
// thread owns the same column x of two neighbouring lines in every plane (x =
// 0 .. NX-1, NX = W - 1 a power of two; the rows at x = NX are identity rows,
// which the first TY threads write). The values of the lower plane around the
// column stay in the thread's registers, so per layer a thread reads the 12
// values and 6 cells of the next plane from LDS for its two rows, and a row
// costs 21 multiply-adds. The loads of the plane after the next and of the
// rows' own inputs are issued before the layer is computed and stored to the
// other LDS buffer after it: one barrier per plane. Bands are grouped per XCD,
// and the planes are split into as many chunks as keep the whole grid resident
// at once (a chunk starts with one extra layer).
// 257^3, one MI355X, against the schedule it replaced (two lines per workgroup
// with rows spread over the threads, 29 LDS reads and 43 multiply-adds a row,
// two barriers a plane): FP32 first step 101 -> 80 us, second 100 -> 99, last with
// its conversion 143 -> 120, d -= A x 87 -> 73, FP64 direction update with the
// operator 186 -> 160.
struct MarchMap {
    int32_t nchunks;
    int32_t glo[8], gsz[8];   // first band and bands of every XCD
};
template <int SH>
struct March {
    static constexpr int NX = 1 << SH, W = NX + 1, G = 256 >> SH, TY = 2 * G, NL = TY + 2, NC = TY + 1;
    static constexpr int SX = (NL * NX + 255) / 256, SC = (NC * NX + 255) / 256;
};

template <typename T, int MODE, int SH>
__global__ __launch_bounds__(256) void k_q1mf_march(MarchMap m, Q1Args<T> q) {
    typedef March<SH> M;
    constexpr int NX = M::NX, W = M::W, G = M::G, TY = M::TY, NL = M::NL, NC = M::NC, SX = M::SX, SC = M::SC;
    constexpr int64_t W2 = (int64_t)W * W;
    __shared__ T xs[2][NL * W];
    __shared__ T cs[2][NC * NX];
    double dot = 0.0;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, g = m.gsz[xcd];
    const int chunk = g == 0 ? 0 : slot / g;
    if (g != 0 && chunk < m.nchunks) {
        const int j0 = (m.glo[xcd] + slot - chunk * g) * TY;
        const int k0 = (int)((int64_t)chunk * W / m.nchunks), k1 = (int)((int64_t)(chunk + 1) * W / m.nchunks);
        const int tid = threadIdx.x, tx = tid & (NX - 1), tg = tid >> SH;
        const T bcg = MODE == 5 ? (T)(q.c ? *q.d64 / (double)*q.c : *q.d64) : (T)0;
        // staging: slot u of a thread is column tx of line tg + u G (lattice
        // line j0 - 1 + that); the lines' last column by the first NL threads
        const int sy = j0 - 1 + tg;
        T va[SX], vb[SX], vc[SC], xa = (T)0, xb = (T)0;
        // MODE 6: the coarse values that the thread's staged points lie between
        // (coarse lines cl0 + j, columns tx/2 and, for odd tx, tx/2 + 1), one new
        // coarse plane for every second fine one: raw parts in flight, and
        // the sums over the columns on the coarse planes below and above
        constexpr int NQ = MODE == 6 ? NL / 2 + 1 : 1;
        constexpr int Wc = NX / 2 + 1;
        T ra[NQ][2], rb[NQ][2], rc[NQ][2], xc = (T)0;
        double lo[NQ], hi[NQ];
        int fetched = -1;   // MODE 6: the plane in flight
        const int cl0 = (j0 >> 1) - 1, cx = tx >> 1, ox = tx & 1;
        auto fetch_coarse = [&](int cp) {
#pragma unroll
            for (int j = 0; j < NQ; ++j)
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const int cy = cl0 + j;
                    const bool in = cy >= 0 && cy < Wc && o <= ox;
                    const int64_t i = ((int64_t)cp * Wc + cy) * Wc + cx + o;
                    ra[j][o] = in ? q.a[i] : (T)0;
                    rb[j][o] = in && q.b ? q.b[i] : (T)0;
                    rc[j][o] = in && q.b ? q.c2[i] : (T)0;
                }
        };
        auto fold_coarse = [&]() {
#pragma unroll
            for (int j = 0; j < NQ; ++j) {
                lo[j] = hi[j];
                const T v0 = q.b ? coarse_fold<T>(ra[j][0], rb[j][0], rc[j][0]) : ra[j][0];
                const T v1 = q.b ? coarse_fold<T>(ra[j][1], rb[j][1], rc[j][1]) : ra[j][1];
                hi[j] = (double)v0 + (double)v1;
            }
        };
        if constexpr (MODE == 6) {
            fetch_coarse((k0 > 0 ? k0 - 1 : 0) >> 1);
            fold_coarse();
            fold_coarse();   // both planes: an even plane takes the upper one over, an odd one replaces it
        }
        auto fetch = [&](int p, int cz) {
            const bool pin = p >= 0 && p < W, cin = cz >= 0 && cz < NX;
            const int64_t base = (int64_t)p * W2;
            if constexpr (MODE == 6) {
                fetched = pin ? p : -1;
                if (pin && (p & 1)) fetch_coarse((p >> 1) + 1);
                xa = xb = xc = (T)0;
                const int ye = j0 - 1 + tid;
                if (pin && !(p & 1) && tid < NL && ye >= 0 && ye < W && !(ye & 1)) {
                    const int64_t i = ((int64_t)(p >> 1) * Wc + (ye >> 1)) * Wc + Wc - 1;
                    xa = q.a[i];
                    xb = q.b ? q.b[i] : (T)0;
                    xc = q.b ? q.c2[i] : (T)0;
                }
            } else {
#pragma unroll
                for (int u = 0; u < SX; ++u) {
                    const int y = sy + u * G;
                    va[u] = vb[u] = (T)0;
                    if (pin && y >= 0 && y < W && tg + u * G < NL)
                        raw_staged<T, MODE>(q, base + (int64_t)y * W + tx, va[u], vb[u]);
                }
                xa = xb = (T)0;
                const int ye = j0 - 1 + tid;
                if (pin && tid < NL && ye >= 0 && ye < W) raw_staged<T, MODE>(q, base + (int64_t)ye * W + NX, xa, xb);
            }
#pragma unroll
            for (int u = 0; u < SC; ++u) {
                const int y = sy + u * G;
                vc[u] = (cin && y >= 0 && y < NX && tg + u * G < NC) ? q.cell[((int64_t)cz * NX + y) * NX + tx] : (T)0;
            }
        };
        auto put = [&](int b) {
            if constexpr (MODE == 6) {
                // plane `fetched`: sums over the planes, then over the lines;
                // the weight is 2^-(odd coordinates), boundary points are zero
                // unless they copy a coarse point
                const int oz = fetched & 1;
                const bool pin = fetched >= 0, pb = fetched == 0 || fetched == W - 1;
                if (pin && oz) fold_coarse();
                if (pin && !oz)
#pragma unroll
                    for (int j = 0; j < NQ; ++j) lo[j] = hi[j];
#pragma unroll
                for (int u = 0; u < SX; ++u) {
                    const int m = tg + u * G, y = j0 - 1 + m;   // y is odd where m is even
                    // between the coarse lines m / 2 and m / 2 + 1 (m even), on
                    // line (m + 1) / 2 (m odd)
                    const bool oy = !(m & 1);
                    auto at = [&](int jj) { return jj < NQ ? (oz ? lo[jj] + hi[jj] : lo[jj]) : 0.0; };
                    double sum;
                    if constexpr (G == 1) sum = (u & 1) ? at((u + 1) / 2) : at(u / 2) + at(u / 2 + 1);
                    else sum = oy ? at(u) + at(u + 1) : at(u + 1);
                    const int nodd = ox + (oy ? 1 : 0) + oz;
                    const double w = nodd == 0 ? 1.0 : nodd == 1 ? 0.5 : nodd == 2 ? 0.25 : 0.125;
                    const bool bnd = tx == 0 || y == 0 || y == W - 1 || pb;
                    const bool zero = !pin || y < 0 || y >= W || (bnd && nodd != 0);
                    if (m < NL) xs[b][m * W + tx] = zero ? (T)0 : (T)(w * sum);
                }
                if (tid < NL) xs[b][tid * W + NX] = q.b ? coarse_fold<T>(xa, xb, xc) : xa;
            } else {
#pragma unroll
                for (int u = 0; u < SX; ++u)
                    if (tg + u * G < NL) xs[b][(tg + u * G) * W + tx] = combine<T, MODE>(va[u], vb[u], bcg);
                if (tid < NL) xs[b][tid * W + NX] = combine<T, MODE>(xa, xb, bcg);
            }
#pragma unroll
            for (int u = 0; u < SC; ++u)
                if (tg + u * G < NC) cs[b][(tg + u * G) * NX + tx] = vc[u];
        };
        const int l0 = 2 * tg, xm = tx > 0 ? tx - 1 : 0;
        auto read = [&](int b, T (&Q)[4][3]) {
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const T* row = xs[b] + (l0 + l) * W;
                Q[l][0] = row[xm];
                Q[l][1] = row[tx];
                Q[l][2] = row[tx + 1];
            }
        };
        fetch(k0 - 1, -1);
        put(0);
        fetch(k0, k0 - 1);
        put(1);
        __syncthreads();
        T P[4][3], off[2], csum[2], pe = (T)0;
        read(0, P);
        off[0] = off[1] = csum[0] = csum[1] = (T)0;
        __syncthreads();
        const int y0 = j0 + l0;
        const bool in0 = y0 < W, in1 = y0 + 1 < W;
        const bool ine = tid < TY && j0 + tid < W;   // the row at x = NX
        const bool side = tx == 0;
        for (int k = k0 - 1; k < k1; ++k) {
            // layer of cells k between planes k and k + 1
            const int b = (k - k0) & 1;   // buffer of plane k + 1: 1 at the first layer
            const bool rows = k >= k0;
            const int64_t i0 = (int64_t)k * W2 + (int64_t)y0 * W + tx;
            const int64_t ie = (int64_t)k * W2 + (int64_t)(j0 + tid) * W + NX;
            fetch(k + 1 < k1 ? k + 2 : -1, k + 1 < k1 ? k + 1 : -1);
            RowIn<T> r0{}, r1{}, re{};
            load_row<T, MODE>(q, i0, rows && in0, r0);
            load_row<T, MODE>(q, i0 + W, rows && in1, r1);
            load_row<T, MODE>(q, ie, rows && ine, re);
            T Q[4][3], c[3][2];
            read(b, Q);
#pragma unroll
            for (int l = 0; l < 3; ++l) {
                c[l][0] = cs[b][(l0 + l) * NX + xm];
                c[l][1] = cs[b][(l0 + l) * NX + tx];
            }
            const T qe = tid < TY ? xs[b][(tid + 1) * W + NX] : (T)0;
            const bool bnd = k == 0 || k == W - 1;
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                T d, ep, eq, cl;
                q1_layer<T>(c[l][0], c[l][1], c[l + 1][0], c[l + 1][1], P[l], P[l + 1], P[l + 2], Q[l], Q[l + 1],
                            Q[l + 2], d, ep, eq, cl);
                const bool in = l == 0 ? in0 : in1;
                if (rows && in) {
                    const int y = y0 + l;
                    const T xi = P[l + 1][1];
                    T s = q1_row<T>(off[l], d + eq, csum[l], cl, xi);
                    if (bnd || side || y == 0 || y == W - 1) s = xi;
                    store_row<T, MODE>(q, i0 + l * W, l == 0 ? r0 : r1, xi, s, dot);
                }
                off[l] = d + ep;
                csum[l] = cl;
            }
            if (rows && ine) store_row<T, MODE>(q, ie, re, pe, pe, dot);
            pe = qe;
#pragma unroll
            for (int l = 0; l < 4; ++l)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) P[l][dx] = Q[l][dx];
            if (k + 1 < k1) put(b ^ 1);
            __syncthreads();
        }
    }
    if (has_dot<MODE>() && q.partial) block_dot(dot, q.partial);
}

// bands of TY lines grouped per XCD (blockIdx % 8), and as many plane chunks
// per band as make the grid resident at once, each at least 4 planes
template <int SH>
int64_t march_grid(const void* kernel, MarchMap& m) {
    const int nb = (March<SH>::W + March<SH>::TY - 1) / March<SH>::TY;
    int maxg = 0;
    for (int c = 0; c < 8; ++c) {
        const int b0 = c * nb / 8, b1 = (c + 1) * nb / 8;
        m.glo[c] = b0;
        m.gsz[c] = b1 - b0;
        maxg = std::max(maxg, b1 - b0);
    }
    const int64_t slots = (int64_t)(device_cus() / 8) * resident_blocks(kernel, 0);
    m.nchunks = (int)std::min<int64_t>(std::max<int64_t>(slots / maxg, 1), March<SH>::W / 4);
    return 8 * (int64_t)maxg * m.nchunks;
}

constexpr int kDirectMaxW = 65;

int64_t direct_grid(int W) {
    const int64_t nb = ((int64_t)W * W * W + 255) / 256;
    return (nb + 7) / 8 * 8;
}

// workgroups of a launch (0: no schedule for this width)
template <typename T, int MODE>
int64_t q1mf_grid(int W, MarchMap& m) {
    if (W <= kDirectMaxW) return direct_grid(W);
    if (W == 129) return march_grid<7>(reinterpret_cast<const void*>(&k_q1mf_march<T, MODE, 7>), m);
    if (W == 257) return march_grid<8>(reinterpret_cast<const void*>(&k_q1mf_march<T, MODE, 8>), m);
    return 0;
}

template <typename T, int MODE>
int q1mf_launch(int W, const Q1Args<T>& q, hipStream_t s, int* n_partial = nullptr) {
    MarchMap m{};
    const int64_t grid = q1mf_grid<T, MODE>(W, m);
    if (!grid) return -1;
    if (q.partial && (!n_partial || grid > *n_partial)) return -1;
    if (W <= kDirectMaxW)
        hipLaunchKernelGGL((k_q1mf_direct<T, MODE>), dim3((unsigned)grid), dim3(256), 0, s, W, grid, q);
    else if (W == 129)
        hipLaunchKernelGGL((k_q1mf_march<T, MODE, 7>), dim3((unsigned)grid), dim3(256), 0, s, m, q);
    else
        hipLaunchKernelGGL((k_q1mf_march<T, MODE, 8>), dim3((unsigned)grid), dim3(256), 0, s, m, q);
    if (n_partial) *n_partial = (int)grid;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

bool q1mf_fused_fits(int W) { return W <= kDirectMaxW || W == 129 || W == 257; }

template <typename T>
int q1mf_jacobi_step(int W, const T* cell, const T* dinv, const T* sd_in, T* sd_out, T* sc, hipStream_t s) {
    if (!q1mf_fused_fits(W)) return q1mf_planes_jacobi_step<T>(W, cell, dinv, sd_in, sd_out, sc, s);
    return q1mf_launch<T, 0>(W, Q1Args<T>{cell, dinv, sd_in, nullptr, sd_out, sc, 0.0, 0.0, nullptr, nullptr, nullptr, nullptr},
                             s);
}
template int q1mf_jacobi_step<float>(int, const float*, const float*, const float*, float*, float*, hipStream_t);
template int q1mf_jacobi_step<double>(int, const double*, const double*, const double*, double*, double*, hipStream_t);

template <typename T>
int q1mf_jacobi_first(int W, const T* cell, const T* dinv, const double* d64, T* sd_out, T* sc, hipStream_t s) {
    return q1mf_launch<T, 3>(W, Q1Args<T>{cell, dinv, nullptr, nullptr, sd_out, sc, 0.0, 0.0, nullptr, d64, nullptr, nullptr},
                             s);
}
template int q1mf_jacobi_first<float>(int, const float*, const float*, const double*, float*, float*, hipStream_t);
template int q1mf_jacobi_first<double>(int, const double*, const double*, const double*, double*, double*, hipStream_t);

template <typename T>
int q1mf_jacobi_first_t(int W, const T* cell, const T* dinv, const T* sd_in, T* sd_out, T* sc, hipStream_t s) {
    return q1mf_launch<T, 4>(W, Q1Args<T>{cell, dinv, sd_in, nullptr, sd_out, sc, 0.0, 0.0, nullptr, nullptr, nullptr, nullptr},
                             s);
}
template int q1mf_jacobi_first_t<float>(int, const float*, const float*, const float*, float*, float*, hipStream_t);

template <typename T>
int q1mf_apply_sub(int W, const T* cell, const T* x, const T* d_in, T* d_out, hipStream_t s) {
    if (!q1mf_fused_fits(W)) return q1mf_planes_apply_sub<T>(W, cell, x, d_in, d_out, s);
    return q1mf_launch<T, 1>(W, Q1Args<T>{cell, x, nullptr, d_in, d_out, nullptr, 0.0, 0.0, nullptr, nullptr, nullptr, nullptr},
                             s);
}
template int q1mf_apply_sub<float>(int, const float*, const float*, const float*, float*, hipStream_t);
template int q1mf_apply_sub<double>(int, const double*, const double*, const double*, double*, hipStream_t);

template <typename T>
int q1mf_jacobi_last(int W, const T* cell, const T* dinv, const T* sd_in, const T* sc, double* z, const double* r,
                     hipStream_t s, double* dot_partial, int* n_partial) {
    if (dot_partial && !n_partial) return -1;
    return q1mf_launch<T, 7>(W, Q1Args<T>{cell, dinv, sd_in, sc, nullptr, nullptr, 0.0, 0.0, dot_partial, r, z, nullptr}, s,
                             n_partial);
}
template int q1mf_jacobi_last<float>(int, const float*, const float*, const float*, const float*, double*,
                                     const double*, hipStream_t, double*, int*);
template int q1mf_jacobi_last<double>(int, const double*, const double*, const double*, const double*, double*,
                                      const double*, hipStream_t, double*, int*);

template <typename T>
int q1mf_axpy(int W, const T* cell, double alpha, const T* v, double beta, const T* x, T* y, hipStream_t s,
              double* dot_partial, int* n_partial) {
    if (!q1mf_fused_fits(W)) {
        if (dot_partial) return -1;   // the fused dot needs one of the schedules here
        return q1mf_planes_axpy<T>(W, cell, alpha, v, beta, x, y, s);
    }
    if (dot_partial && !n_partial) return -1;
    return q1mf_launch<T, 2>(W, Q1Args<T>{cell, x, nullptr, v, y, nullptr, alpha, beta, dot_partial, nullptr, nullptr, nullptr},
                             s, n_partial);
}
template int q1mf_axpy<double>(int, const double*, double, const double*, double, const double*, double*, hipStream_t,
                               double*, int*);

// p_new must not alias p_old (other workgroups still stage p_old)
template <typename T>
int q1mf_direction_axpy(int W, const T* cell, const T* p_old, const T* z, const double* beta_dev, T* p_new, T* y,
                        hipStream_t s, double* dot_partial, int* n_partial, const double* rho_old) {
    if (p_new == p_old || !dot_partial || !n_partial) return -1;
    return q1mf_launch<T, 5>(W, Q1Args<T>{cell, p_old, z, rho_old, y, p_new, 0.0, 1.0, dot_partial, beta_dev, nullptr, nullptr},
                             s, n_partial);
}
template int q1mf_direction_axpy<double>(int, const double*, const double*, const double*, const double*, double*,
                                         double*, hipStream_t, double*, int*, const double*);

// t = P c (the coarse correction, with its last update c += dinv_c .* sd_c
// folded in where given), d -= A t, sc += t on the marching widths in FP32: the
// prolongation's separate pass wrote t and read it back. One MI355X, 129^3 ->
// 257^3: 72 + 73 us in two passes, 111 in this one. FP64 keeps two: the values
// around a column and their sums take the registers of a resident workgroup
// (65^3 -> 129^3 38.6 us in two passes, 38.1 in one).
bool q1mf_prolong_sub_fits(int W) { return W == 129 || W == 257; }
template <typename T>
int q1mf_prolong_sub(int W, const T* cell, const T* c_coarse, const T* dinv_c, const T* sd_c, T* d, T* sc,
                     hipStream_t s) {
    if ((dinv_c == nullptr) != (sd_c == nullptr)) return -1;
    MarchMap m{};
    Q1Args<T> q{cell, c_coarse, dinv_c, d, d, sc, 0.0, 0.0, nullptr, nullptr, nullptr, sd_c};
    if (W == 129) {
        const int64_t grid = march_grid<7>(reinterpret_cast<const void*>(&k_q1mf_march<T, 6, 7>), m);
        hipLaunchKernelGGL((k_q1mf_march<T, 6, 7>), dim3((unsigned)grid), dim3(256), 0, s, m, q);
    } else if (W == 257) {
        const int64_t grid = march_grid<8>(reinterpret_cast<const void*>(&k_q1mf_march<T, 6, 8>), m);
        hipLaunchKernelGGL((k_q1mf_march<T, 6, 8>), dim3((unsigned)grid), dim3(256), 0, s, m, q);
    } else {
        return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int q1mf_prolong_sub<float>(int, const float*, const float*, const float*, const float*, float*, float*,
                                     hipStream_t);

// asks the runtime for the residency of the marching kernels at this width, so
// that no query happens inside a captured cycle
int q1mf_prepare(int W) {
    MarchMap m{};
    q1mf_grid<float, 0>(W, m);
    q1mf_grid<float, 1>(W, m);
    q1mf_grid<float, 3>(W, m);
    q1mf_grid<float, 4>(W, m);
    q1mf_grid<float, 7>(W, m);
    if (W == 129) {
        march_grid<7>(reinterpret_cast<const void*>(&k_q1mf_march<float, 6, 7>), m);
    } else if (W == 257) {
        march_grid<8>(reinterpret_cast<const void*>(&k_q1mf_march<float, 6, 8>), m);
    }
    q1mf_grid<double, 0>(W, m);
    q1mf_grid<double, 1>(W, m);
    q1mf_grid<double, 2>(W, m);
    q1mf_grid<double, 3>(W, m);
    q1mf_grid<double, 5>(W, m);
    q1mf_grid<double, 7>(W, m);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugamd
