// Q2 (triquadratic Lagrange) hexahedron element matrices on gfx950, two
// elements per wavefront by sum factorisation.
//
// Per element (corners X in the reference hexahedron order, coefficient k,
// constant source f): Ke[a][b] = sum_q w_q |det J_q| k grad phi_a . grad phi_b
// and fe[a] = sum_q w_q |det J_q| f phi_a over the 3x3x3 Gauss-Legendre
// points, with the trilinear geometry of the 8 corners. With the symmetric 3x3
// G_q = w_q |det J_q| k J_q^-1 J_q^-T and phi_a = l_i(x) l_j(y) l_m(z),
//   Ke = sum_{d,e} sum_qz sum_qy sum_qx G_q[d][e] (d_d phi_a) (d_e phi_b)
// is summed one direction at a time: 1.5 k multiply-adds for the sums over x
// (54 lanes), 7.7 k for those over y and z (45 lanes: one per unordered pair of
// (i, j), nine entries each), where the contraction over all points at once is
// 64 k on the matrix cores.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ugx_internal.hpp"

namespace ugamd {
namespace {

__device__ __forceinline__ double q2_gauss(int i) {
    // 3-point Gauss-Legendre on [0, 1]: 1/2 -+ sqrt(3/5)/2
    return i == 0 ? 0.11270166537925831 : i == 1 ? 0.5 : 0.8872983346207417;
}
__device__ __forceinline__ double q2_gauss_w(int i) { return i == 1 ? 8.0 / 18.0 : 5.0 / 18.0; }

// Local shape order of LagrangeLSFS<ReferenceHexahedron, 2> (lagrange.cpp:
// 236-253, lagrange.h:2106-2190): multi-indices of the vertices (2 x corner),
// the edge midpoints of edges (0,1) (1,2) (2,3) (3,0) (0,4) (1,5) (2,6) (3,7)
// (4,5) (5,6) (6,7) (7,4), the centres of faces {0,3,2,1} {0,1,5,4} {1,2,6,5}
// {2,3,7,6} {3,0,4,7} {4,5,6,7} (reference_element.cpp), then the interior.
constexpr int8_t kQ2Mi[27][3] = {
    {0, 0, 0}, {2, 0, 0}, {2, 2, 0}, {0, 2, 0}, {0, 0, 2}, {2, 0, 2}, {2, 2, 2}, {0, 2, 2}, {1, 0, 0},
    {2, 1, 0}, {1, 2, 0}, {0, 1, 0}, {0, 0, 1}, {2, 0, 1}, {2, 2, 1}, {0, 2, 1}, {1, 0, 2}, {2, 1, 2},
    {1, 2, 2}, {0, 1, 2}, {1, 1, 0}, {1, 0, 1}, {2, 1, 1}, {1, 2, 1}, {0, 1, 1}, {1, 1, 2}, {1, 1, 1}};
constexpr double q2c_x(int i) { return i == 0 ? 0.11270166537925831 : i == 1 ? 0.5 : 0.8872983346207417; }
constexpr double q2c_l(int i, double x) {
    return i == 0 ? (1.0 - x) * (1.0 - 2.0 * x) : i == 1 ? 4.0 * x * (1.0 - x) : x * (2.0 * x - 1.0);
}
constexpr double q2c_dl(int i, double x) { return i == 0 ? 4.0 * x - 3.0 : i == 1 ? 4.0 - 8.0 * x : 4.0 * x - 1.0; }
// the 1D polynomials and their derivatives at the Gauss points, and the local
// number of the multi-index i + 3 j + 9 m
struct Q2Basis {
    double l[3][3], d[3][3];   // [polynomial][point]
    int8_t num[27];
};
constexpr Q2Basis q2_basis() {
    Q2Basis t{};
    for (int i = 0; i < 3; ++i)
        for (int q = 0; q < 3; ++q) {
            t.l[i][q] = q2c_l(i, q2c_x(q));
            t.d[i][q] = q2c_dl(i, q2c_x(q));
        }
    for (int a = 0; a < 27; ++a) t.num[kQ2Mi[a][0] + 3 * kQ2Mi[a][1] + 9 * kQ2Mi[a][2]] = (int8_t)a;
    return t;
}
__constant__ Q2Basis kQ2Basis = q2_basis();

constexpr int kQ2Waves = 4;   // wavefronts per workgroup, two elements each

// a wavefront's scratch
struct Q2Scratch {
    double X[2][24];       // corners of the two elements
    double G[2][6][27];    // xx, yy, zz, xy, xz, yz at point qx + 3 qy + 9 qz
    double fw[2][27];      // w_q |det J_q| f
    double K[729];         // sums over x, then the element matrix
};
// LDS written by some lanes of a wavefront is read by others: in order, once
// the compiler keeps it so
__device__ __forceinline__ void q2_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// products of two 1D factors at the three points, for the nine pairs of
// polynomials: first derivative on neither, the first, both (x), and all four (y)
struct Q2Tables {
    double x[3][9][3];
    double y[9][12];   // ll, l d, d l, dd
    double l[3][3];
    int mi[27];        // multi-indices of the local shapes, two bits a direction
};
__device__ __forceinline__ void q2_fill_tables(Q2Tables& t) {
    for (int e = threadIdx.x; e < 27; e += blockDim.x) {
        const int p = e / 3, q = e - 3 * p;
        const double l1 = kQ2Basis.l[p / 3][q], l2 = kQ2Basis.l[p % 3][q];
        const double d1 = kQ2Basis.d[p / 3][q], d2 = kQ2Basis.d[p % 3][q];
        t.x[0][p][q] = t.y[p][q] = l1 * l2;
        t.y[p][3 + q] = l1 * d2;
        t.x[1][p][q] = t.y[p][6 + q] = d1 * l2;
        t.x[2][p][q] = t.y[p][9 + q] = d1 * d2;
        if (p < 3) t.l[p][q] = kQ2Basis.l[p][q];
        t.mi[e] = kQ2Mi[e][0] | kQ2Mi[e][1] << 2 | kQ2Mi[e][2] << 4;
    }
    __syncthreads();
}

// a lane's part: its (i, i') and field of the first stage, its (i, j) and
// (i', j') of the second
struct Q2Lane {
    int xrow;      // row of Q2Tables::x
    int g;         // field of G
    int p1, p1t;   // (i, i') and (i', i)
    int py;        // (j, j')
    uint32_t a, b;   // the local shapes (i, j, m) and (i', j', m), m = 0, 1, 2, a byte each
    int mi;          // multi-index of shape l % 32, two bits each
    __device__ __forceinline__ void init(int l) {
        // fields dd Gxx, ll Gyy, ll Gzz, ll Gyz, dl Gxy, dl Gxz of nine pairs each
        const int pair = l < 54 ? l % 9 : 0, field = l < 54 ? l / 9 : 0;
        xrow = (field == 0 ? 2 : field < 4 ? 0 : 1) * 9 + pair;
        g = field == 3 ? 5 : field == 4 ? 3 : field == 5 ? 4 : field;
        int u = 0, v = l < 45 ? l : 0;   // the l-th u <= v of 9
        while (v >= 9 - u) {
            v -= 9 - u;
            ++u;
        }
        v += u;
        a = kQ2Basis.num[u] | kQ2Basis.num[u + 9] << 8 | kQ2Basis.num[u + 18] << 16;
        b = kQ2Basis.num[v] | kQ2Basis.num[v + 9] << 8 | kQ2Basis.num[v + 18] << 16;
        const int s = (l & 31) < 27 ? l & 31 : 0;
        mi = kQ2Mi[s][0] | kQ2Mi[s][1] << 2 | kQ2Mi[s][2] << 4;
        p1 = (u % 3) * 3 + v % 3;
        p1t = (v % 3) * 3 + u % 3;
        py = (u / 3) * 3 + v / 3;
    }
};

// A lane's inputs of the element of its half (l / 32): corner coordinate l % 32
// and the coefficient at Gauss point l % 32 (x fastest); the unit cube for an
// element that is not there
struct Q2In {
    double x, k;
};
template <class Src>
__device__ __forceinline__ Q2In q2_load(int l, const bool (&valid)[2], const Src& src) {
    const int hl = l & 31, c = hl / 3, d = hl - 3 * c;
    const int bit = d == 0 ? (c == 1 || c == 2 || c == 5 || c == 6) : d == 1 ? (c == 2 || c == 3 || c == 6 || c == 7)
                                                                     : (c >= 4);
    const bool mine = l >> 5 ? valid[1] : valid[0];
    Q2In in;
    in.x = mine && hl < 24 ? src.corner(hl) : (double)bit;
    in.k = mine && hl < 27 ? src.k(hl) : 1.0;
    return in;
}

// Two elements by one wavefront (lane l): sink.ke(l, K) with the element matrix K
// in LDS and sink.fe(a, v) for the 27 load entries of each valid element.
template <class Sink>
__device__ __forceinline__ void q2_element_pair(int l, const Q2Lane& L, const Q2Tables& tab, const bool (&valid)[2],
                                                Q2In in, Sink (&sink)[2], double f_const, Q2Scratch& sh,
                                                bool want_fe) {
    // what follows from the lane alone is formed again for every pair of elements:
    // kept across them, it would take the registers of the stages below
    asm volatile("" : "+v"(l));
    const int half = l >> 5, hl = l & 31;
    const bool mine = half ? valid[1] : valid[0];
    q2_wave_sync();   // the elements before are done with the scratch
    if (hl < 24) sh.X[half][hl] = in.x;
    q2_wave_sync();
    // 1. G at point q = hl: the Jacobian of the trilinear map column by column
    if (hl < 27) {
        const double* X = sh.X[half];
        const int qx = hl % 3, qy = (hl / 3) % 3, qz = hl / 9;
        const double x1 = q2_gauss(qx), y1 = q2_gauss(qy), z1 = q2_gauss(qz);
        const double x0 = 1.0 - x1, y0 = 1.0 - y1, z0 = 1.0 - z1;
        double J[3][3];   // J[c][r] = dX_r / dxi_c
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const double X0 = X[r], X1 = X[3 + r], X2 = X[6 + r], X3 = X[9 + r], X4 = X[12 + r], X5 = X[15 + r],
                         X6 = X[18 + r], X7 = X[21 + r];
            J[0][r] = z0 * (y0 * (X1 - X0) + y1 * (X2 - X3)) + z1 * (y0 * (X5 - X4) + y1 * (X6 - X7));
            J[1][r] = z0 * (x0 * (X3 - X0) + x1 * (X2 - X1)) + z1 * (x0 * (X7 - X4) + x1 * (X6 - X5));
            J[2][r] = y0 * (x0 * (X4 - X0) + x1 * (X5 - X1)) + y1 * (x0 * (X7 - X3) + x1 * (X6 - X2));
        }
        double C[3][3];   // rows of det J J^-1
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double* p = J[(d + 1) % 3];
            const double* q = J[(d + 2) % 3];
            C[d][0] = p[1] * q[2] - p[2] * q[1];
            C[d][1] = p[2] * q[0] - p[0] * q[2];
            C[d][2] = p[0] * q[1] - p[1] * q[0];
        }
        const double det = fabs(J[0][0] * C[0][0] + J[0][1] * C[0][1] + J[0][2] * C[0][2]);
        const double w = q2_gauss_w(qx) * q2_gauss_w(qy) * q2_gauss_w(qz);
        const double g = w * in.k / det;
        auto dot = [&](int d, int e) { return g * (C[d][0] * C[e][0] + C[d][1] * C[e][1] + C[d][2] * C[e][2]); };
        sh.G[half][0][hl] = dot(0, 0);
        sh.G[half][1][hl] = dot(1, 1);
        sh.G[half][2][hl] = dot(2, 2);
        sh.G[half][3][hl] = dot(0, 1);
        sh.G[half][4][hl] = dot(0, 2);
        sh.G[half][5][hl] = dot(1, 2);
        if (want_fe) sh.fw[half][hl] = w * det * f_const;
    }
    q2_wave_sync();
    // load vector: fe[a] = sum_q w_q |det J_q| f phi_a(xi_q)
    if (want_fe && hl < 27) {
        const double *lx = tab.l[L.mi & 3], *ly = tab.l[L.mi >> 2 & 3], *lz = tab.l[L.mi >> 4];
        double s = 0.0;
#pragma unroll 1
        for (int qz = 0; qz < 3; ++qz) {
            double sy = 0.0;
#pragma unroll
            for (int qy = 0; qy < 3; ++qy) {
                const double* f = sh.fw[half] + 3 * qy + 9 * qz;
                const double sx = f[0] * lx[0] + f[1] * lx[1] + f[2] * lx[2];
                sy = fma(ly[qy], sx, sy);
            }
            s = fma(lz[qz], sy, s);
        }
        if (mine && half) sink[1].fe(hl, s);
        if (mine && !half) sink[0].fe(hl, s);
    }
#pragma unroll 1
    for (int el = 0; el < 2; ++el) {
        if (!(el ? valid[1] : valid[0])) continue;   // the same for the whole wavefront
        Q2Lane M = L;
        asm volatile("" : "+v"(M.xrow), "+v"(M.g), "+v"(M.p1), "+v"(M.p1t), "+v"(M.py), "+v"(M.a), "+v"(M.b));
        // 2. sums over x: T[field][pair][qy + 3 qz]
        double* T = sh.K;
        q2_wave_sync();
        if (l < 54) {
            const double* G = sh.G[el][M.g];
            const double* c = tab.x[0][0] + 3 * M.xrow;
            const double c0 = c[0], c1 = c[1], c2 = c[2];
            double v[27];
#pragma unroll
            for (int p = 0; p < 27; ++p) v[p] = G[p];
#pragma unroll
            for (int p = 0; p < 9; ++p) T[l * 9 + p] = fma(c2, v[3 * p + 2], fma(c1, v[3 * p + 1], c0 * v[3 * p]));
        }
        q2_wave_sync();
        // 3. sums over y, then over z: V[m][m'] of the lane's (i, j), (i', j')
        double V[3][3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int k = 0; k < 3; ++k) V[m][k] = 0.0;
        double y[12];
#pragma unroll
        for (int q = 0; q < 12; ++q) y[q] = tab.y[M.py][q];
        const double* Txx = T + M.p1 * 9;
        const double* Tyy = T + 81 + M.p1 * 9;
        const double* Tzz = T + 162 + M.p1 * 9;
        const double* Tyz = T + 243 + M.p1 * 9;
        const double* Txy = T + 324 + M.p1 * 9;    // derivative on i
        const double* Tyx = T + 324 + M.p1t * 9;   // derivative on i'
        const double* Txz = T + 405 + M.p1 * 9;
        const double* Tzx = T + 405 + M.p1t * 9;
#pragma unroll
        for (int qz = 0; qz < 3; ++qz) {
            // one plane of T in registers at a time: its offset is known once the
            // plane before is done
            int o = 3 * qz;
            asm volatile("" : "+v"(o) : "v"(V[2][2]));
            double ull = 0.0, uld = 0.0, udl = 0.0, udd = 0.0;   // by the z factors of (a, b)
#pragma unroll
            for (int qy = 0; qy < 3; ++qy) {
                const int p = o + qy;
                const double yz = Tyz[p];
                ull = fma(y[qy], Txx[p], ull);
                ull = fma(y[9 + qy], Tyy[p], ull);
                ull = fma(y[3 + qy], Txy[p], ull);
                ull = fma(y[6 + qy], Tyx[p], ull);
                udd = fma(y[qy], Tzz[p], udd);
                uld = fma(y[qy], Txz[p], uld);
                uld = fma(y[6 + qy], yz, uld);
                udl = fma(y[qy], Tzx[p], udl);
                udl = fma(y[3 + qy], yz, udl);
            }
            // constants that vanish at the middle point drop out
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double lk = q2c_l(k, q2c_x(qz)), dk = q2c_dl(k, q2c_x(qz));
                double A = 0.0, D = 0.0;
                if (lk != 0.0) {
                    A = ull * lk;
                    D = udl * lk;
                }
                if (dk != 0.0) {
                    A = fma(uld, dk, A);
                    D = fma(udd, dk, D);
                }
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    const double lm = q2c_l(m, q2c_x(qz)), dm = q2c_dl(m, q2c_x(qz));
                    if (lm != 0.0) V[m][k] = fma(lm, A, V[m][k]);
                    if (dm != 0.0) V[m][k] = fma(dm, D, V[m][k]);
                }
            }
        }
        q2_wave_sync();   // T is read before its place takes the matrix
        if (l < 45) {
            int a[3], b[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                a[m] = M.a >> (8 * m) & 255u;
                b[m] = M.b >> (8 * m) & 255u;
            }
            // an entry and its transpose take the same value
#pragma unroll
            for (int m = 0; m < 3; ++m)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    sh.K[27 * a[m] + b[k]] = V[m][k];
                    sh.K[27 * b[k] + a[m]] = V[m][k];
                }
        }
        q2_wave_sync();
        if (el) sink[1].ke(l, sh.K);
        else sink[0].ke(l, sh.K);
    }
}

// adds the element matrix to val at slot(i, j): no two entries of an element
// share a slot, so a lane's twelve slots and then its twelve values are in flight
// together
template <class Slot>
__device__ __forceinline__ void q2_add(int l, const double* K, double* val, const Slot& slot) {
    int32_t p[12];
    double v[12];
#pragma unroll
    for (int r = 0; r < 12; ++r) {
        const int e = l + 64 * r < 729 ? l + 64 * r : 728;
        const int i = (int)((unsigned)e * 2428u >> 16);   // e / 27
        p[r] = slot(i, e - 27 * i);
    }
#pragma unroll
    for (int r = 0; r < 12; ++r) v[r] = val[p[r]];
#pragma unroll
    for (int r = 0; r < 12; ++r)
        if (l + 64 * r < 729) val[p[r]] = v[r] + K[l + 64 * r];
}

struct Q2ArraySrc {
    const double* X;
    const double* kc;
    int64_t e;
    __device__ double corner(int l) const { return X[e * 24 + l]; }
    __device__ double k(int) const { return kc ? kc[e] : 1.0; }
};
struct Q2ArraySink {
    double* Kout;
    double* fout;
    __device__ __forceinline__ void ke(int l, const double* K) {
        for (int e = l; e < 729; e += 64) Kout[e] = K[e];
    }
    __device__ void fe(int a, double v) { fout[a] = v; }
};

// Every wavefront takes pairs of elements in turn. Bound by the 5.8 kB that an
// element writes: 64^3 elements (1.64 GB with the inputs) 482 us on one MI355X, 838 us with
// the contraction over all points on the matrix cores (129 kflop an element in
// their 16 x 16 x 4 steps, four of ten of their FP64 rate), Jacobians by 27 of 64
// lanes and every entry stored from where it arose. What is left is latency: three
// waves a SIMD (a fourth would spill: 748 us), each a chain through LDS.
__global__ __launch_bounds__(64 * kQ2Waves, 3) void k_q2_hex_elements(int64_t n, const double* __restrict__ X,
                                                                   const double* __restrict__ kcoef, double f_const,
                                                                   double* __restrict__ Ke, double* __restrict__ fe) {
    __shared__ Q2Scratch sh[kQ2Waves];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    __shared__ Q2Tables tab;
    q2_fill_tables(tab);
    Q2Lane L;
    L.init(l);
    // the next pair's inputs are in flight while a pair is computed
    auto load = [&](int64_t p) {
        const bool valid[2] = {2 * p < n, 2 * p + 1 < n};
        return q2_load(l, valid, Q2ArraySrc{X, kcoef, 2 * p + (l >> 5)});
    };
    const int64_t step = (int64_t)gridDim.x * kQ2Waves;
    int64_t p = (int64_t)blockIdx.x * kQ2Waves + w;
    Q2In in = load(p);
    for (; 2 * p < n; p += step) {
        const bool valid[2] = {true, 2 * p + 1 < n};
        const int64_t e1 = valid[1] ? 2 * p + 1 : 2 * p;
        Q2ArraySink sink[2] = {{Ke + 2 * p * 729, fe ? fe + 2 * p * 27 : nullptr},
                               {Ke + e1 * 729, fe ? fe + e1 * 27 : nullptr}};
        const Q2In next = load(p + step);
        q2_element_pair(l, L, tab, valid, in, sink, f_const, sh[w], fe != nullptr);
        in = next;
    }
}

// ---- assembly on the unit-cube lattice of n^3 elements ----
// Q2 nodes on the (2n+1)^3 lattice, numbered x fastest; element (ex, ey, ez)
// holds the nodes 2 e + m for its local multi-indices m. Two nodes are coupled
// when they share an element, which factorises per direction: an even
// coordinate c (a lattice plane of vertices) reaches c-2 .. c+2, an odd one
// (inside one element) c-1 .. c+1.
__device__ __forceinline__ void q2_range(int c, int W, int& lo, int& hi) {
    const int r = (c & 1) ? 1 : 2;
    lo = c - r < 0 ? 0 : c - r;
    hi = c + r > W - 1 ? W - 1 : c + r;
}

__global__ void k_q2_lattice_count(int W, int64_t N, int32_t* cnt) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % W), y = (int)((i / W) % W), z = (int)(i / ((int64_t)W * W));
        int a, b, c, d, e, f;
        q2_range(x, W, a, b);
        q2_range(y, W, c, d);
        q2_range(z, W, e, f);
        cnt[i] = (b - a + 1) * (d - c + 1) * (f - e + 1);
    }
}

// one wavefront per row: lane l writes entries l, l + 64 of the row's
// (z, y, x)-ordered box of columns, so the row's writes are contiguous
__global__ __launch_bounds__(256) void k_q2_lattice_fill(int W, int64_t N, const int32_t* __restrict__ rowptr,
                                                         int32_t* __restrict__ col) {
    const int64_t i = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6);
    if (i >= N) return;
    const int lane = threadIdx.x & 63;
    const int x = (int)(i % W), y = (int)((i / W) % W), z = (int)(i / ((int64_t)W * W));
    int x0, x1, y0, y1, z0, z1;
    q2_range(x, W, x0, x1);
    q2_range(y, W, y0, y1);
    q2_range(z, W, z0, z1);
    const int nx = x1 - x0 + 1, ny = y1 - y0 + 1, len = nx * ny * (z1 - z0 + 1);
    const int32_t p = rowptr[i];
    for (int e = lane; e < len; e += 64) {
        const int xx = x0 + e % nx, yy = y0 + (e / nx) % ny, zz = z0 + e / (nx * ny);
        col[p + e] = (int32_t)(((int64_t)zz * W + yy) * W + xx);
    }
}

struct Q2LatticeSrc {
    int n;
    double h;
    int ex, ey, ez;
    const double* theta;
    __device__ double corner(int l) const {
        const int c = l / 3, d = l - 3 * c;
        const int bit = d == 0 ? (c == 1 || c == 2 || c == 5 || c == 6) : d == 1 ? (c == 2 || c == 3 || c == 6 || c == 7)
                                                                         : (c >= 4);
        const int e = d == 0 ? ex : d == 1 ? ey : ez;
        return (double)(e + bit) * h;
    }
    __device__ double k(int) const { return theta ? exp(theta[((int64_t)ez * n + ey) * n + ex]) : 1.0; }
};
// Entry (i, j) of element (ex, ey, ez): the row's columns are its box [x0,x1] x
// [y0,y1] x [z0,z1] in (z, y, x) order, so the CSR slot follows from the
// multi-indices; decoding node numbers took eight divisions an entry (a colour of
// 32,768 elements 301 us, 231 so and with a lane's slots in flight together, one
// MI355X)
struct Q2CsrSink {
    int W, ex, ey, ez;
    const int32_t* rowptr;
    double* val;
    double* rhs;
    const int* mi;
    __device__ __forceinline__ int32_t node(int m) const {
        return ((2 * ez + (m >> 4)) * W + 2 * ey + (m >> 2 & 3)) * W + 2 * ex + (m & 3);
    }
    __device__ __forceinline__ int32_t slot(int i, int j) const {
        const int a = mi[i], b = mi[j];
        const int x = 2 * ex + (a & 3), y = 2 * ey + (a >> 2 & 3), z = 2 * ez + (a >> 4);
        const int cx = 2 * ex + (b & 3), cy = 2 * ey + (b >> 2 & 3), cz = 2 * ez + (b >> 4);
        int x0, x1, y0, y1, z0, z1;
        q2_range(x, W, x0, x1);
        q2_range(y, W, y0, y1);
        q2_range(z, W, z0, z1);
        const int nx = x1 - x0 + 1, ny = y1 - y0 + 1;
        return rowptr[(z * W + y) * W + x] + ((cz - z0) * ny + (cy - y0)) * nx + (cx - x0);
    }
    __device__ __forceinline__ void ke(int l, const double* K) {
        q2_add(l, K, val, [&](int i, int j) { return slot(i, j); });
    }
    __device__ __forceinline__ void fe(int a, double v) { rhs[node(mi[a])] += v; }
};

// one colour (element parities px, py, pz): no two of its elements share a node
__global__ __launch_bounds__(64 * kQ2Waves, 3) void k_q2_lattice_assemble(int n, int color, const double* theta,
                                                                       double f_const, const int32_t* rowptr,
                                                                       double* val, double* rhs) {
    const int hn = (n + 1) / 2;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * kQ2Waves + w;
    const int px = color & 1, py = (color >> 1) & 1, pz = color >> 2;
    __shared__ Q2Scratch sh[kQ2Waves];
    __shared__ Q2Tables tab;
    q2_fill_tables(tab);
    Q2Lane L;
    L.init(l);
    Q2LatticeSrc src{n, 1.0 / n, 0, 0, 0, theta};   // of the lane's half
    Q2CsrSink sink[2];
    bool valid[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t t = 2 * p + h;
        const int tx = (int)(t % hn), ty = (int)((t / hn) % hn), tz = (int)(t / ((int64_t)hn * hn));
        const int ex = 2 * tx + px, ey = 2 * ty + py, ez = 2 * tz + pz;
        valid[h] = t < (int64_t)hn * hn * hn && ex < n && ey < n && ez < n;
        if (h == l >> 5) {
            src.ex = ex;
            src.ey = ey;
            src.ez = ez;
        }
        sink[h] = Q2CsrSink{2 * n + 1, ex, ey, ez, rowptr, val, rhs, tab.mi};
    }
    q2_element_pair(l, L, tab, valid, q2_load(l, valid, src), sink, f_const, sh[w],
                    rhs != nullptr);
}

// Dirichlet rows (u = 0 on the boundary of the cube): row := unit row on its
// pattern, rhs := 0
__global__ void k_q2_lattice_dirichlet(int W, int64_t N, const int32_t* __restrict__ rowptr,
                                       const int32_t* __restrict__ col, double* val, double* rhs) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % W), y = (int)((i / W) % W), z = (int)(i / ((int64_t)W * W));
        if (x > 0 && y > 0 && z > 0 && x < W - 1 && y < W - 1 && z < W - 1) continue;
        for (int32_t p = rowptr[i]; p < rowptr[i + 1]; ++p) val[p] = col[p] == (int32_t)i ? 1.0 : 0.0;
        rhs[i] = 0.0;
    }
}

// ---- Q2 hexahedra of a caller-supplied connectivity (ElementDiscretization) ----
struct Q2ElemSrc {
    const double* coords;   // DoF coordinates [N][3]
    const int32_t* dofs;    // [ne][27] in the local shape order
    const double* kel;      // per element or null
    const double* kq;       // per element and Gauss point [ne][27] or null
    int64_t e;
    __device__ double corner(int l) const {
        const int c = l / 3, d = l - 3 * c;
        return coords[(int64_t)dofs[e * 27 + c] * 3 + d];
    }
    __device__ double k(int q) const { return kq ? kq[e * 27 + q] : (kel ? kel[e] : 1.0); }
};
// matrix entries through the per-entry slots (slot[(27 i + j) * ne + pos] for
// the element at colour-sorted position pos), load entries into rhs
struct Q2SlotSink {
    const int32_t* slot;
    const int32_t* dofs;
    int64_t ne, pos, e;
    double* val;
    double* rhs;
    __device__ __forceinline__ void ke(int l, const double* K) {
        if (val) q2_add(l, K, val, [&](int i, int j) { return slot[(int64_t)(27 * i + j) * ne + pos]; });
    }
    __device__ void fe(int a, double v) { rhs[dofs[e * 27 + a]] += v; }
};

// one colour's elements (positions pos0 .. pos0+cnt-1 of the colour order), two
// per wavefront
__global__ __launch_bounds__(64 * kQ2Waves, 3) void k_elem_hex_q2(int64_t ne, const int32_t* __restrict__ order,
                                                               const int32_t* __restrict__ dofs,
                                                               const double* __restrict__ coords,
                                                               const double* __restrict__ kel,
                                                               const double* __restrict__ kq, double f_const,
                                                               const int32_t* __restrict__ slot, double* val,
                                                               double* rhs, int64_t pos0, int64_t cnt) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * kQ2Waves + w;
    __shared__ Q2Scratch sh[kQ2Waves];
    __shared__ Q2Tables tab;
    q2_fill_tables(tab);
    Q2Lane L;
    L.init(l);
    Q2ElemSrc src{coords, dofs, kel, kq, 0};   // of the lane's half
    Q2SlotSink sink[2];
    bool valid[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t t = 2 * p + h;
        valid[h] = t < cnt;
        const int64_t pos = pos0 + (valid[h] ? t : 0);
        const int64_t e = order[pos];
        if (h == l >> 5) src.e = e;
        sink[h] = Q2SlotSink{slot, dofs, ne, pos, e, val, rhs};
    }
    q2_element_pair(l, L, tab, valid, q2_load(l, valid, src), sink, f_const, sh[w],
                    rhs != nullptr);
}

}  // namespace

int q2_hex_elements(int64_t n, const double* X, const double* k, double f_const, double* Ke, double* fe,
                    hipStream_t s) {
    if (n <= 0) return 0;
    if (!X || !Ke || n > (int64_t)INT32_MAX) return -1;
    const int64_t need = (n + 2 * kQ2Waves - 1) / (2 * kQ2Waves);
    const int64_t fit = (int64_t)device_cus() * resident_blocks(reinterpret_cast<const void*>(&k_q2_hex_elements), 0);
    hipLaunchKernelGGL(k_q2_hex_elements, dim3((unsigned)std::min(need, fit)), dim3(64 * kQ2Waves), 0, s, n, X, k,
                       f_const, Ke, fe);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int q2_lattice_count(int n, int32_t* cnt, hipStream_t s) {
    const int W = 2 * n + 1;
    const int64_t N = (int64_t)W * W * W;
    hipLaunchKernelGGL(k_q2_lattice_count, dim3((unsigned)std::min<int64_t>((N + 255) / 256, 65536)), dim3(256), 0, s,
                       W, N, cnt);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
int q2_lattice_fill(int n, const int32_t* rowptr, int32_t* col, hipStream_t s) {
    const int W = 2 * n + 1;
    const int64_t N = (int64_t)W * W * W;
    hipLaunchKernelGGL(k_q2_lattice_fill, dim3((unsigned)((N + 3) / 4)), dim3(256), 0, s, W, N, rowptr, col);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
int q2_lattice_assemble(int n, const double* theta, double f_const, const int32_t* rowptr, const int32_t* col,
                        double* val, double* rhs, hipStream_t s) {
    const int hn = (n + 1) / 2;
    const int64_t per = (int64_t)hn * hn * hn;
    for (int color = 0; color < 8; ++color)
        hipLaunchKernelGGL(k_q2_lattice_assemble, dim3((unsigned)((per + 2 * kQ2Waves - 1) / (2 * kQ2Waves))),
                           dim3(64 * kQ2Waves), 0, s, n, color, theta, f_const, rowptr, val, rhs);
    const int W = 2 * n + 1;
    const int64_t N = (int64_t)W * W * W;
    hipLaunchKernelGGL(k_q2_lattice_dirichlet, dim3((unsigned)std::min<int64_t>((N + 255) / 256, 65536)), dim3(256),
                       0, s, W, N, rowptr, col, val, rhs);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int elem_assemble_q2_colour(int64_t ne, const int32_t* order, const int32_t* dofs, const double* coords,
                            const double* kel, const double* kq, double f_const, const int32_t* slot, double* val,
                            double* rhs, int64_t pos0, int64_t cnt, hipStream_t s) {
    if (cnt <= 0) return 0;
    hipLaunchKernelGGL(k_elem_hex_q2, dim3((unsigned)((cnt + 2 * kQ2Waves - 1) / (2 * kQ2Waves))), dim3(64 * kQ2Waves), 0, s,
                       ne, order, dofs, coords, kel, kq, f_const, slot, val, rhs, pos0, cnt);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugamd
