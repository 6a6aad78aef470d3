// Sliced ELL with a column dictionary per slice: the SpMV layout of
// GPUSparseMatrix when the rows can be grouped into slices of 64 whose entries
// touch at most 255 distinct columns (a 4x4x4 block of lattice points has
// 6x6x6 = 216 neighbours in a 27-point pattern, whatever the DoF numbering).
//
//   * slice t holds rows order[64t .. 64t+63] (-1: an empty lane);
//   * its distinct columns, sorted, are dict[dptr[t] .. dptr[t+1]);
//   * entry k of lane l is value sval[vptr[t] + 2*(64*(k/2) + l) + k%2]
//     (two consecutive entries of a row form one 16-byte load) and the byte
//     k%4 of word sidx[iptr[t] + 64*(k/4) + l], the entry's position in the
//     dictionary; a padded entry has value 0 and position 255, which the
//     product maps to 0 (so non-finite vector entries stay out, as they do in
//     the CSR product);
//   * the product stages x at the dictionary's columns in LDS once per slice
//     (216 gathers instead of 27 per row) and streams 9 bytes per entry.
// Each row is summed as the sliced-ELL kernel sums it (even and odd entries of
// the slice width's groups of four in two sums, the last w % 4 entries into
// the first, in order), so the two layouts agree bit for bit where a row's
// slice has the same width in both placements and to rounding otherwise; only
// the storage of the column indices differs from the CSR, which download_csr
// still returns.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "ugx_internal.hpp"

namespace ugamd {

namespace {

constexpr int kDictSlots = 255;       // dictionary entries per slice (position 255 = zero)
constexpr int kDictMaxWidth = 64;     // longest row of a slice that the layout takes
constexpr int kHashSlots = 512;       // LDS hash of a slice's columns (at most 255 + 64 occupied)
constexpr int kChunk = 8;             // entries per row moved through LDS at a time

typedef double dbl2 __attribute__((ext_vector_type(2)));

inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t > 0 ? (n + t - 1) / t : 1); }

__device__ __forceinline__ int hash_slot(int32_t c) { return (int)(((uint32_t)c * 2654435761u) >> 23); }

// slot of column c, which is in the table
__device__ __forceinline__ int hash_find(const int32_t* hk, int32_t c) {
    int h = hash_slot(c);
    while (hk[h] != c) h = (h + 1) & (kHashSlots - 1);
    return h;
}

// Kernels below run one 64-lane workgroup (one wavefront) per slice. The
// slice's rows: start and length of lane l's row in rbs[l], lens[l] (length 0
// for an empty lane)
__device__ __forceinline__ void slice_rows(int64_t nrows, const int32_t* __restrict__ rowptr,
                                           const int32_t* __restrict__ order, int64_t t, int32_t* rbs, int32_t* lens) {
    const int lane = threadIdx.x;
    const int32_t r = order[t * 64 + lane];
    int32_t rb = 0, len = 0;
    if (r >= 0 && r < nrows) {
        rb = rowptr[r];
        len = rowptr[r + 1] - rb;
    }
    rbs[lane] = rb;
    lens[lane] = len;
}

// inserts the slice's columns into the LDS hash table hk (all -1 on entry;
// *cnt 0): the entries are read row by row (lane e of a round reads entry
// e % w of row e / w), so a round reads contiguous CSR runs. Returns the
// number of distinct columns, or a number above 255 as soon as a round ends
// above it (then the table is incomplete). A round adds at most 64 keys, so
// at most 319 of the 512 slots are ever occupied and every probe ends.
__device__ int slice_hash(int w, const int32_t* rbs, const int32_t* lens, const int32_t* __restrict__ col,
                          int32_t* hk, int* cnt) {
    const int lane = threadIdx.x;
    const int total = 64 * w;
    for (int base = 0; base < total; base += 64) {
        const int e = base + lane;
        if (e < total) {
            const int j = e / w, k = e - j * w;
            if (k < lens[j]) {
                const int32_t c = col[rbs[j] + k];
                int h = hash_slot(c);
                for (;;) {
                    const int32_t old = atomicCAS(&hk[h], -1, c);
                    if (old == -1) {
                        atomicAdd(cnt, 1);
                        break;
                    }
                    if (old == c) break;
                    h = (h + 1) & (kHashSlots - 1);
                }
            }
        }
        __syncthreads();
        const int u = *cnt;
        __syncthreads();
        if (u > kDictSlots) return u;
    }
    return *cnt;
}

__device__ __forceinline__ void cmp_swap(int32_t& a, int32_t& b, bool up) {
    if ((a > b) == up) {
        const int32_t t = a;
        a = b;
        b = t;
    }
}

// bitonic sort of the 256 keys v[0..3] of the wave (key 4*lane + m in v[m]),
// ascending
__device__ __forceinline__ void wave_sort256(int32_t v[4]) {
    const int lane = threadIdx.x;
    for (int size = 2; size <= 256; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            if (stride >= 4) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const int i = 4 * lane + m;
                    const int32_t o = __shfl_xor(v[m], stride >> 2, 64);
                    const bool up = (i & size) == 0, lower = (i & stride) == 0;
                    v[m] = (lower == up) ? min(v[m], o) : max(v[m], o);
                }
            } else {
                const bool up = ((4 * lane) & size) == 0;   // size >= 4 here, or size 2 (both halves alike below)
                if (stride == 2) {
                    cmp_swap(v[0], v[2], up);
                    cmp_swap(v[1], v[3], up);
                } else if (size == 2) {
                    cmp_swap(v[0], v[1], true);
                    cmp_swap(v[2], v[3], false);
                } else {
                    cmp_swap(v[0], v[1], up);
                    cmp_swap(v[2], v[3], up);
                }
            }
        }
    }
}

// distinct columns per slice (above 255, or INT_MAX when the slice is wider
// than the layout takes: the slice does not fit)
__global__ __launch_bounds__(64) void k_dict_count(int64_t nrows, const int32_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ col, const int32_t* __restrict__ order,
                                                   const int32_t* __restrict__ width, int32_t* __restrict__ ucount) {
    __shared__ int32_t hk[kHashSlots];
    __shared__ int32_t rbs[64], lens[64];
    __shared__ int cnt;
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const int w = width[t];
    if (w > kDictMaxWidth) {
        if (lane == 0) ucount[t] = INT_MAX;
        return;
    }
    for (int h = lane; h < kHashSlots; h += 64) hk[h] = -1;
    if (lane == 0) cnt = 0;
    slice_rows(nrows, rowptr, order, t, rbs, lens);
    __syncthreads();
    const int u = slice_hash(w, rbs, lens, col, hk, &cnt);
    if (lane == 0) ucount[t] = u;
}

// moves the slice's values (and, with pb, the dictionary positions of the
// entries) through LDS in chunks of kChunk entries per row: rows are read
// contiguously, the value pairs and position words written contiguously.
// hk/hv: column -> position (used when pb is given)
__device__ void slice_values_out(int w, const int32_t* rbs, const int32_t* lens, const int32_t* __restrict__ col,
                                 const double* __restrict__ val, const int32_t* hk, const int32_t* hv, uint8_t* pb,
                                 double* vt, double* __restrict__ sv, uint32_t* __restrict__ si) {
    const int lane = threadIdx.x;
    const int npairs = (w + 1) >> 1, nwords = (w + 3) >> 2;
    for (int k0 = 0; k0 < w; k0 += kChunk) {
#pragma unroll
        for (int it = 0; it < kChunk; ++it) {
            const int e = it * 64 + lane;
            const int j = e / kChunk, kk = e % kChunk, k = k0 + kk;
            uint32_t pos = 255;
            double v = 0.0;
            if (k < lens[j]) {
                const int64_t a = (int64_t)rbs[j] + k;
                v = val[a];
                if (pb) pos = (uint32_t)hv[hash_find(hk, col[a])];
            }
            if (pb) pb[kk * 64 + j] = (uint8_t)pos;
            vt[(kk >> 1) * 128 + 2 * j + (kk & 1)] = v;
        }
        __syncthreads();
        const int npc = min(kChunk / 2, npairs - k0 / 2);
        for (int o = lane; o < 128 * npc; o += 64) sv[(int64_t)64 * k0 + o] = vt[o];
        if (pb) {
            const int nqc = min(kChunk / 4, nwords - k0 / 4);
            for (int qq = 0; qq < nqc; ++qq) {
                const uint8_t* b = pb + 4 * qq * 64 + lane;
                si[(int64_t)64 * (k0 / 4 + qq) + lane] =
                    (uint32_t)b[0] | ((uint32_t)b[64] << 8) | ((uint32_t)b[128] << 16) | ((uint32_t)b[192] << 24);
            }
        }
        __syncthreads();
    }
}

// the dictionary (sorted distinct columns), positions and values of every
// slice; the count pass has checked that every slice fits
__global__ __launch_bounds__(64) void k_dict_fill(int64_t nrows, const int32_t* __restrict__ rowptr,
                                                  const int32_t* __restrict__ col, const double* __restrict__ val,
                                                  const int32_t* __restrict__ order, const int32_t* __restrict__ width,
                                                  const int32_t* __restrict__ dptr, const int64_t* __restrict__ vptr,
                                                  const int64_t* __restrict__ iptr, int32_t* __restrict__ dict,
                                                  double* __restrict__ sval, uint32_t* __restrict__ sidx) {
    __shared__ int32_t hk[kHashSlots], hv[kHashSlots];
    __shared__ int32_t rbs[64], lens[64], list[256];
    __shared__ int cnt;
    __shared__ uint8_t pb[kChunk * 64];
    __shared__ double vt[kChunk * 64];
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x;
    const int w = width[t];
    for (int h = lane; h < kHashSlots; h += 64) hk[h] = -1;
    if (lane == 0) cnt = 0;
    slice_rows(nrows, rowptr, order, t, rbs, lens);
    __syncthreads();
    const int u = slice_hash(w, rbs, lens, col, hk, &cnt);
    if (u > kDictSlots) return;   // not a slice that fits (the count pass keeps such layouts from being built)
    // compact the table (lane l owns slots 8l .. 8l+7), then sort
    int n = 0;
    for (int i = 0; i < 8; ++i) n += hk[8 * lane + i] >= 0 ? 1 : 0;
    int off = n;
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(off, d, 64);
        if (lane >= d) off += o;
    }
    off -= n;
    for (int i = 0; i < 8; ++i) {
        const int32_t c = hk[8 * lane + i];
        if (c >= 0) list[off++] = c;
    }
    for (int i = u + lane; i < 256; i += 64) list[i] = INT_MAX;
    __syncthreads();
    int32_t v[4] = {list[4 * lane], list[4 * lane + 1], list[4 * lane + 2], list[4 * lane + 3]};
    wave_sort256(v);
    const int32_t d0 = dptr[t];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int i = 4 * lane + m;
        if (i < u) {
            dict[d0 + i] = v[m];
            hv[hash_find(hk, v[m])] = i;
        }
    }
    __syncthreads();
    slice_values_out(w, rbs, lens, col, val, hk, hv, pb, vt, sval + vptr[t], sidx + iptr[t]);
}

// the values alone, for a matrix whose pattern (and so dictionary and
// positions) is unchanged since k_dict_fill: up to 32 columns of all 64 rows
// at a time through LDS, each row's run read once and in one piece (lane e of
// a round reads entry e % wc of row e / wc), the loads of 8 rounds issued
// before their stores; the value pairs then written out contiguously
constexpr int kValCols = 32;
__global__ __launch_bounds__(64) void k_dict_values(int64_t nrows, const int32_t* __restrict__ rowptr,
                                                    const double* __restrict__ val, const int32_t* __restrict__ order,
                                                    const int32_t* __restrict__ width, const int64_t* __restrict__ vptr,
                                                    double* __restrict__ sval) {
    __shared__ int32_t rbs[64], lens[64];
    __shared__ double vt[kValCols * 64];
    const int64_t t = blockIdx.x;
    slice_rows(nrows, rowptr, order, t, rbs, lens);
    __syncthreads();
    const int w = width[t], lane = threadIdx.x;
    double* sv = sval + vptr[t];
    for (int k0 = 0; k0 < w; k0 += kValCols) {
        const int wc = min(kValCols, w - k0), wp = wc + (wc & 1);   // a padded odd entry is written as 0
        const int total = 64 * wp;
        for (int e0 = lane; e0 < total; e0 += 8 * 64) {
            double v[8];
            int o[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = e0 + u * 64;
                const int j = e / wp, kk = e - j * wp, k = k0 + kk;
                o[u] = e < total ? (kk >> 1) * 128 + 2 * j + (kk & 1) : -1;
                v[u] = (e < total && k < lens[j]) ? val[(int64_t)rbs[j] + k] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (o[u] >= 0) vt[o[u]] = v[u];
        }
        __syncthreads();
        for (int q = lane; q < 64 * wp; q += 64) sv[(int64_t)64 * k0 + q] = vt[q];
        __syncthreads();
    }
}

// the sum of a lane's row from entry k (a multiple of 4) to the slice's width w,
// on top of s0 and s1
__device__ __forceinline__ double dict_row_sum(const dbl2* vp, const uint32_t* ip, int w, const double* xs, int k,
                                               double s0, double s1) {
    for (; k + 4 <= w; k += 4) {
        const uint32_t word = __builtin_nontemporal_load(ip + 64 * (k >> 2));
        const dbl2 a = __builtin_nontemporal_load(vp + 64 * (k >> 1));
        const dbl2 b = __builtin_nontemporal_load(vp + 64 * ((k >> 1) + 1));
        s0 = fma(a.x, xs[word & 255u], s0);
        s1 = fma(a.y, xs[(word >> 8) & 255u], s1);
        s0 = fma(b.x, xs[(word >> 16) & 255u], s0);
        s1 = fma(b.y, xs[word >> 24], s1);
    }
    // the last w % 4 entries all go to s0, in order, as in the sliced-ELL
    // kernel, so the two layouts round identically
    if (k < w) {
        const uint32_t word = __builtin_nontemporal_load(ip + 64 * (k >> 2));
        const dbl2 a = __builtin_nontemporal_load(vp + 64 * (k >> 1));
        s0 = fma(a.x, xs[word & 255u], s0);
        if (k + 1 < w) s0 = fma(a.y, xs[(word >> 8) & 255u], s0);
        if (k + 2 < w) {
            const dbl2 b = __builtin_nontemporal_load(vp + 64 * ((k >> 1) + 1));
            s0 = fma(b.x, xs[(word >> 16) & 255u], s0);
        }
    }
    return s0 + s1;
}

// y = alpha*v1 + beta*A*x (mode 0), or y = beta*A*x on rows with entries
// (mode 1); one wave per slice, four slices per workgroup.
// Bound by HBM: 9 bytes per entry and the dictionaries (257^3 Q1 operator 988 us
// on one MI355X). A kernel of its own: as one template with the form below its
// further arguments cost the products that stay in the caches (33^3 Q1 6.35 us
// against 6.15, 65^3 17.15 and 16.99, 49^3 tetrahedral rows 8.09 and 7.92).
__global__ __launch_bounds__(256) void k_dict_spmv(int64_t nrows, int64_t nslices, const int32_t* __restrict__ width,
                                                   const int32_t* __restrict__ dptr, const int32_t* __restrict__ dict,
                                                   const int64_t* __restrict__ vptr, const int64_t* __restrict__ iptr,
                                                   const double* __restrict__ sval, const uint32_t* __restrict__ sidx,
                                                   const int32_t* __restrict__ order, double alpha, const double* v1,
                                                   double beta, const double* __restrict__ x, double* y, int mode,
                                                   const int32_t* __restrict__ rowptr) {
    __shared__ double xl[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + wave;
    double* xs = xl[wave];
    int w = 0;
    if (t < nslices) {
        const int32_t d0 = dptr[t], nd = dptr[t + 1] - d0;
        for (int j = lane; j < nd; j += 64) xs[j] = x[dict[d0 + j]];
        if (lane == 0) xs[255] = 0.0;
        w = width[t];
    }
    __syncthreads();
    if (t >= nslices) return;
    const dbl2* vp = reinterpret_cast<const dbl2*>(sval + vptr[t]) + lane;
    const uint32_t* ip = sidx + iptr[t] + lane;
    const double sum = dict_row_sum(vp, ip, w, xs, 0, 0.0, 0.0);
    const int32_t r = order[t * 64 + lane];
    if (r < 0 || r >= nrows) return;
    if (mode == 1) {
        if (rowptr[r + 1] > rowptr[r]) y[r] = beta * sum;
    } else {
        const double base = (alpha == 0.0) ? 0.0 : alpha * v1[r];
        y[r] = base + beta * sum;
    }
}

// y = A x with the workgroup's partial sums of (y, u) and (y, y), in part[block]
// and part[blocks + block]. x may be FP32 (converted as it is staged); dict and
// order may number the columns and rows differently from the matrix's own
// numbering (order and x, y then share that numbering). These are the products
// of a solver's step on operators that stay in the caches, where latency counts:
// the first kPre entries of every row and the row numbers are requested before
// the dictionary and x (a chain of three dependent loads and a barrier that the
// values do not depend on), and consecutive slices run on one XCD, whose L2 then
// holds the x values that neighbouring lattice blocks share (97^3 tetrahedral
// rows, one MI355X: 41 us without the two, 37 us with them and the partials; the
// product at the stream's rate loses by them, 988 -> 995 us, so k_dict_spmv has
// neither).
template <typename XT>
__global__ __launch_bounds__(256) void k_dict_spmv_dots(int64_t nrows, int64_t nslices,
                                                        const int32_t* __restrict__ width,
                                                        const int32_t* __restrict__ dptr,
                                                        const int32_t* __restrict__ dict,
                                                        const int64_t* __restrict__ vptr,
                                                        const int64_t* __restrict__ iptr,
                                                        const double* __restrict__ sval,
                                                        const uint32_t* __restrict__ sidx,
                                                        const int32_t* __restrict__ order,
                                                        const XT* __restrict__ x, double* __restrict__ y,
                                                        int64_t per_xcd, const double* __restrict__ u,
                                                        double* __restrict__ part) {
    __shared__ double xl[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t lb = per_xcd ? (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : (int64_t)blockIdx.x;
    const int64_t t = lb * 4 + wave;
    double* xs = xl[wave];
    const bool live = t < nslices;
    int w = 0;
    const dbl2* vp = reinterpret_cast<const dbl2*>(sval) + lane;
    const uint32_t* ip = sidx + lane;
    int32_t r = -1;
    if (live) {
        w = width[t];
        vp = reinterpret_cast<const dbl2*>(sval + vptr[t]) + lane;
        ip += iptr[t];
        r = order[t * 64 + lane];
    }
    constexpr int kPre = 8;
    uint32_t pw[kPre / 4];
    dbl2 pv[kPre / 2];
    const bool pre = w >= kPre;   // the same for every lane of the wave
    if (pre) {
#pragma unroll
        for (int q = 0; q < kPre / 4; ++q) pw[q] = __builtin_nontemporal_load(ip + 64 * q);
#pragma unroll
        for (int q = 0; q < kPre / 2; ++q) pv[q] = __builtin_nontemporal_load(vp + 64 * q);
    }
    if (live) {
        const int32_t d0 = dptr[t], nd = dptr[t + 1] - d0;
        for (int j = lane; j < nd; j += 64) xs[j] = (double)x[dict[d0 + j]];
        if (lane == 0) xs[255] = 0.0;
    }
    const bool mine = r >= 0 && r < nrows;
    const double ur = mine ? u[r] : 0.0;
    __syncthreads();
    double s0 = 0.0, s1 = 0.0;
    int k = 0;
    if (pre) {
#pragma unroll
        for (int q = 0; q < kPre / 4; ++q) {
            const uint32_t word = pw[q];
            s0 = fma(pv[2 * q].x, xs[word & 255u], s0);
            s1 = fma(pv[2 * q].y, xs[(word >> 8) & 255u], s1);
            s0 = fma(pv[2 * q + 1].x, xs[(word >> 16) & 255u], s0);
            s1 = fma(pv[2 * q + 1].y, xs[word >> 24], s1);
        }
        k = kPre;
    }
    const double sum = dict_row_sum(vp, ip, w, xs, k, s0, s1);
    const double yr = mine ? 0.0 + sum : 0.0;
    double yu = yr * ur, yy = yr * yr;
    if (mine) y[r] = yr;
    for (int o = 32; o > 0; o >>= 1) {
        yu += __shfl_down(yu, o, 64);
        yy += __shfl_down(yy, o, 64);
    }
    __shared__ double sh[2][4];
    if (lane == 0) {
        sh[0][wave] = yu;
        sh[1][wave] = yy;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const double* q = sh[threadIdx.x];
        part[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = (q[0] + q[1]) + (q[2] + q[3]);
    }
}

// Q1 values (and load vector) of a lattice operator whose pattern and
// dictionary are in place, into the CSR and the dictionary layout in one pass,
// one wave per slice, one row per lane. A lane forms the 27 entries of its row
// in registers (64 multiply-adds; the same order as k_q1_lattice_csr, so the
// same bits) and leaves them in LDS by direction. The row's entries are the
// slice's dictionary positions, so the direction of entry k is the lattice
// difference between that dictionary column and the row: the layout's pairs are
// written from there in entry order, and the CSR rows, two at a time, by lanes
// that own a direction and its rank in the row. Boundary rows are identity
// rows with a zero load.
// Bound by the two writes of 8 bytes per entry. One pass for the CSR with 32
// lanes a row (ranks by shuffles, every lane testing all 8 elements), one for
// the Dirichlet rows and one that read the CSR back for the layout took 695 us
// at 129^3 (57,066,625 entries) on one MI355X; this pass 325 us.
__global__ __launch_bounds__(64) void k_dict_q1_values(int n, int64_t nslices, double h, double fh3,
                                                       const double* __restrict__ tab,
                                                       const double* __restrict__ kel,
                                                       const int32_t* __restrict__ lat_of_dof,
                                                       const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ width,
                                                       const int32_t* __restrict__ dptr,
                                                       const int32_t* __restrict__ dict,
                                                       const int64_t* __restrict__ vptr,
                                                       const int64_t* __restrict__ iptr,
                                                       const uint32_t* __restrict__ sidx, double* __restrict__ sval,
                                                       double* __restrict__ val, double* __restrict__ rhs) {
    constexpr int P = 65;   // row pitch of a direction: the reads along a row hit different banks
    __shared__ double v[27 * P];
    __shared__ uint8_t rank[27 * 64];
    __shared__ int32_t code[256], rb[64];
    const int lane = threadIdx.x, W = n + 1;
    const int64_t per = (nslices + 7) / 8;
    const int64_t t = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);   // consecutive slices on one XCD
    if ((blockIdx.x >> 3) >= per || t >= nslices) return;
    auto point = [&](int32_t l, int& x, int& y, int& z) {
        const int yz = l / W;
        x = l - yz * W;
        z = yz / W;
        y = yz - z * W;
    };
    const int32_t r = order[t * 64 + lane];
    const int w = width[t];
    const int32_t d0 = dptr[t], nd = dptr[t + 1] - d0;
    // everything that the chains of dependent loads below end in is requested
    // up front: positions, dictionary, rows
    const uint32_t* ip = sidx + iptr[t] + lane;
    uint32_t word[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) word[j] = 4 * j < w ? __builtin_nontemporal_load(ip + 64 * j) : 0u;
    int32_t lp[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) lp[j] = nd > 0 ? dict[d0 + (lane + 64 * j < nd ? lane + 64 * j : 0)] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) lp[j] = lat_of_dof[lp[j]];
    // lattice points as x | y << 10 | z << 20
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        int x, y, z;
        point(lp[j], x, y, z);
        if (lane + 64 * j < nd) code[lane + 64 * j] = x | y << 10 | z << 20;
    }
    for (int i = lane; i < 27 * 64; i += 64) rank[i] = 255;
    int x = 0, y = 0, z = 0, len = 0;
    rb[lane] = 0;
    if (r >= 0) {
        point(lat_of_dof[r], x, y, z);
        rb[lane] = rowptr[r];
        len = rowptr[r + 1] - rowptr[r];
    }
    const bool inner = r >= 0 && x > 0 && y > 0 && z > 0 && x < n && y < n && z < n;
    double e[27], f = 0.0;
#pragma unroll
    for (int d = 0; d < 27; ++d) e[d] = 0.0;
    if (inner) {
#pragma unroll
        for (int o = 0; o < 8; ++o) {
            const int ox = o & 1, oy = (o >> 1) & 1, oz = o >> 2;
            // local index of a corner in the reference hexahedron
            auto local = [](int cx, int cy, int cz) { return 4 * cz + (cy ? 3 - cx : cx); };
            const int a = local(1 - ox, 1 - oy, 1 - oz);
            const double k = kel ? kel[((int64_t)(z - 1 + oz) * n + y - 1 + oy) * n + x - 1 + ox] : 1.0;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int bx = c & 1, by = (c >> 1) & 1, bz = c >> 2;
                const int d = (oz + bz) * 9 + (oy + by) * 3 + ox + bx;
                e[d] = fma(k, tab[512 + 8 * a + local(bx, by, bz)], e[d]);
            }
            f += tab[576 + a];
        }
#pragma unroll
        for (int d = 0; d < 27; ++d) e[d] *= h;
    } else {
        e[13] = 1.0;
    }
#pragma unroll
    for (int d = 0; d < 27; ++d) v[d * P + lane] = e[d];
    if (rhs && r >= 0) rhs[r] = inner ? fh3 * f : 0.0;
    __syncthreads();
    // the layout's pairs in entry order, and the rank of every direction
    dbl2* vp = reinterpret_cast<dbl2*>(sval + vptr[t]) + lane;
    const int own = (x | y << 10 | z << 20) - (1 | 1 << 10 | 1 << 20);
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        const int k = 4 * j;
        if (k >= w) break;
        double q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            q[u] = 0.0;
            if (k + u < len) {
                const int df = code[(word[j] >> (8 * u)) & 255u] - own;
                const int d = ((df >> 20) & 3) * 9 + ((df >> 10) & 3) * 3 + (df & 3);
                q[u] = v[d * P + lane];
                rank[d * 64 + lane] = (uint8_t)(k + u);
            }
        }
        const dbl2 p0 = {q[0], q[1]}, p1 = {q[2], q[3]};
        __builtin_nontemporal_store(p0, vp + 64 * (k >> 1));
        if (k + 2 < w) __builtin_nontemporal_store(p1, vp + 64 * ((k >> 1) + 1));
    }
    __syncthreads();
    const int d = lane & 31, half = lane >> 5;
    if (d < 27)
#pragma unroll 8
        for (int j = half; j < 64; j += 2) {
            const int k = rank[d * 64 + j];
            if (k != 255) val[(int64_t)rb[j] + k] = v[d * P + j];
        }
}

// the rows of a lattice in blocks of 64 points: 4x4x4 (3D) or 8x8 (2D). Slot
// 64*b + l of block b (x fastest over the blocks) holds the DoF of the block's
// point l (x fastest inside the block), -1 where the block extends past the
// lattice
__global__ void k_block_order(int dim, int W, const int32_t* __restrict__ dof_of_lat, int32_t* __restrict__ order) {
    const int e = dim == 3 ? 4 : 8;
    const int nb = (W + e - 1) / e;
    const int64_t nblocks = dim == 3 ? (int64_t)nb * nb * nb : (int64_t)nb * nb;
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= nblocks * 64) return;
    const int64_t b = s >> 6;
    const int l = (int)(s & 63);
    if (dim == 3) {
        const int bx = (int)(b % nb), by = (int)((b / nb) % nb), bz = (int)(b / ((int64_t)nb * nb));
        const int x = 4 * bx + (l & 3), y = 4 * by + ((l >> 2) & 3), z = 4 * bz + (l >> 4);
        order[s] = (x < W && y < W && z < W) ? dof_of_lat[((int64_t)z * W + y) * W + x] : -1;
    } else {
        const int bx = (int)(b % nb), by = (int)(b / nb);
        const int x = 8 * bx + (l & 7), y = 8 * by + (l >> 3);
        order[s] = (x < W && y < W) ? dof_of_lat[(int64_t)y * W + x] : -1;
    }
}

__global__ void k_dict_widths(int64_t nslices, int64_t nrows, const int32_t* __restrict__ rowptr,
                              const int32_t* __restrict__ order, int32_t* __restrict__ width) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= nslices) return;
    int32_t w = 0;
    for (int l = 0; l < 64; ++l) {
        const int32_t r = order[t * 64 + l];
        if (r >= 0 && r < nrows) {
            const int32_t len = rowptr[r + 1] - rowptr[r];
            w = len > w ? len : w;
        }
    }
    width[t] = w;
}

}  // namespace

int dict_widths(int64_t nslices, int64_t nrows, const int32_t* rowptr, const int32_t* order, int32_t* width,
                hipStream_t s) {
    if (nslices <= 0) return 0;
    hipLaunchKernelGGL(k_dict_widths, dim3(nblk(nslices, 256)), dim3(256), 0, s, nslices, nrows, rowptr, order, width);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int dict_count(int64_t nslices, int64_t nrows, const int32_t* rowptr, const int32_t* col, const int32_t* order,
               const int32_t* width, int32_t* ucount, hipStream_t s) {
    if (nslices <= 0) return 0;
    hipLaunchKernelGGL(k_dict_count, dim3((unsigned)nslices), dim3(64), 0, s, nrows, rowptr, col, order, width,
                       ucount);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int dict_fill(int64_t nslices, int64_t nrows, const int32_t* rowptr, const int32_t* col, const double* val,
              const int32_t* order, const int32_t* width, const int32_t* dptr, const int64_t* vptr,
              const int64_t* iptr, int32_t* dict, double* sval, uint32_t* sidx, hipStream_t s) {
    if (nslices <= 0) return 0;
    hipLaunchKernelGGL(k_dict_fill, dim3((unsigned)nslices), dim3(64), 0, s, nrows, rowptr, col, val, order, width,
                       dptr, vptr, iptr, dict, sval, sidx);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int dict_values(int64_t nslices, int64_t nrows, const int32_t* rowptr, const double* val, const int32_t* order,
                const int32_t* width, const int64_t* vptr, double* sval, hipStream_t s) {
    if (nslices <= 0) return 0;
    hipLaunchKernelGGL(k_dict_values, dim3((unsigned)nslices), dim3(64), 0, s, nrows, rowptr, val, order, width, vptr,
                       sval);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int dict_spmv(int64_t nrows, int64_t nslices, const int32_t* width, const int32_t* dptr, const int32_t* dict,
              const int64_t* vptr, const int64_t* iptr, const double* sval, const uint32_t* sidx,
              const int32_t* order, double alpha, const double* v1, double beta, const double* x, double* y, int mode,
              const int32_t* rowptr, hipStream_t s) {
    if (nslices <= 0) return 0;
    hipLaunchKernelGGL(k_dict_spmv, dim3(nblk(nslices, 4)), dim3(256), 0, s, nrows, nslices, width, dptr, dict, vptr,
                       iptr, sval, sidx, order, alpha, v1, beta, x, y, mode, rowptr);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int64_t dict_spmv_blocks(int64_t nslices) {
    const int64_t nb = (nslices + 3) / 4;
    return nb >= 64 ? (nb + 7) / 8 * 8 : nb;
}

template <typename XT>
int dict_spmv_dots(int64_t nrows, int64_t nslices, const int32_t* width, const int32_t* dptr, const int32_t* dict,
                   const int64_t* vptr, const int64_t* iptr, const double* sval, const uint32_t* sidx,
                   const int32_t* order, const XT* x, double* y, const double* u, double* part, hipStream_t s) {
    if (nslices <= 0) return -1;
    const int64_t nb = (nslices + 3) / 4, per = nb >= 64 ? (nb + 7) / 8 : 0;
    hipLaunchKernelGGL(k_dict_spmv_dots<XT>, dim3((unsigned)dict_spmv_blocks(nslices)), dim3(256), 0, s, nrows,
                       nslices, width, dptr, dict, vptr, iptr, sval, sidx, order, x, y, per, u, part);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int dict_spmv_dots<float>(int64_t, int64_t, const int32_t*, const int32_t*, const int32_t*, const int64_t*,
                                   const int64_t*, const double*, const uint32_t*, const int32_t*, const float*,
                                   double*, const double*, double*, hipStream_t);
template int dict_spmv_dots<double>(int64_t, int64_t, const int32_t*, const int32_t*, const int32_t*, const int64_t*,
                                    const int64_t*, const double*, const uint32_t*, const int32_t*, const double*,
                                    double*, const double*, double*, hipStream_t);

int dict_q1_values(int n, int64_t nslices, double h, double f_const, const double* tab, const double* kel,
                   const int32_t* lat_of_dof, const int32_t* order, const int32_t* rowptr, const int32_t* width,
                   const int32_t* dptr, const int32_t* dict, const int64_t* vptr, const int64_t* iptr,
                   const uint32_t* sidx, double* sval, double* val, double* rhs, hipStream_t s) {
    if (n <= 0 || n >= 1023 || nslices <= 0) return -1;
    const int64_t per = (nslices + 7) / 8;
    hipLaunchKernelGGL(k_dict_q1_values, dim3((unsigned)(8 * per)), dim3(64), 0, s, n, nslices, h, f_const * h * h * h,
                       tab, kel, lat_of_dof, order, rowptr, width, dptr, dict, vptr, iptr, sidx, sval, val, rhs);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int64_t lattice_block_slots(int dim, int W) {
    const int e = dim == 3 ? 4 : 8;
    const int64_t nb = (W + e - 1) / e;
    return (dim == 3 ? nb * nb * nb : nb * nb) * 64;
}

int lattice_block_order(int dim, int W, const int32_t* dof_of_lat, int32_t* order, hipStream_t s) {
    const int64_t n = lattice_block_slots(dim, W);
    hipLaunchKernelGGL(k_block_order, dim3(nblk(n, 256)), dim3(256), 0, s, dim, W, dof_of_lat, order);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugamd
