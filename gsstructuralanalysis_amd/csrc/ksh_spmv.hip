// ksh_spmv.hip -- symmetric band mat-vec y = K x and batched refinement residuals r = b - K x.
//
// K is stored as its lower band, column major: ab[j*ld + (i-j)], ld = bw+1.  The single mat-vec goes by
// rows: a workgroup of 256 threads owns a block of 64 consecutive rows:
//   lower part  sum_{j<=i} K[i][j] x[j]: lanes = the block's rows, so each band column contributes
//               one contiguous 64-entry run (coalesced); the four waves take every fourth column and
//               issue 8 independent loads per lane before accumulating;
//   upper part  sum_{j>i} K[j][i] x[j] = sum_d ab[i*ld + d] x[i+d]: one wave per 16 rows, lanes along
//               the contiguous column of row i, wave reductions.
// Every band entry is read twice (once for each triangle), one launch, no scratch.  The batched
// residuals go by columns (below), each entry read once; their norms are reduced per block, then
// per matrix in block order (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>
#include <vector>

#include "ksh_devutil.hpp"
#include "ksh_internal.hpp"
#include "ksh_profile.hpp"
#include "ksh_vec.hpp"

namespace ksh {

namespace {

constexpr int kRows = 64;
constexpr int kT = 256;
constexpr int kU = 8;

// (K x)[i0 + lane] for NR vectors x[0..NR-1] at once: the band entries are loaded once and used
// for every vector.  Returns the products in y (valid in lanes 0..63 of every wave).
template <typename T, int NR>
__device__ __forceinline__ void symv_row_block(const T *__restrict__ ab, int n, int bw, const double *const (&x)[NR], int i0,
                                               double (&y)[NR])
{
    __shared__ double part[NR][4][kRows];
    __shared__ double up[NR][kRows];
    const size_t ld = (size_t)bw + 1;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int i = i0 + lane;
    const bool ok = i < n;
    // lower triangle incl. diagonal
    {
        const int jlo = max(0, i0 - bw), jhi = min(n - 1, i0 + kRows - 1);
        double acc[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) acc[q] = 0.0;
        for (int jb = jlo + wave; jb <= jhi; jb += 4 * kU) {
            double v[kU], xv[NR][kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                int j = jb + 4 * u;
                bool in = ok && j <= jhi && j <= i && i - j <= bw;
                v[u] = in ? (double)ab[(size_t)j * ld + (i - j)] : 0.0;
#pragma unroll
                for (int q = 0; q < NR; ++q) xv[q][u] = (j <= jhi) ? x[q][j] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int q = 0; q < NR; ++q) acc[q] += v[u] * xv[q][u];
        }
#pragma unroll
        for (int q = 0; q < NR; ++q) part[q][wave][lane] = acc[q];
    }
    // strict upper triangle: rows 16*wave .. 16*wave+15 of the block
    for (int rr = 0; rr < 16; ++rr) {
        const int row = i0 + 16 * wave + rr;
        double acc[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) acc[q] = 0.0;
        if (row < n) {
            const int dmax = min(bw, n - 1 - row);
            for (int d0 = 1; d0 <= dmax; d0 += 64 * 4) {
                double v[4], xv[NR][4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    int d = d0 + lane + 64 * u;
                    bool in = d <= dmax;
                    v[u] = in ? (double)ab[(size_t)row * ld + d] : 0.0;
#pragma unroll
                    for (int q = 0; q < NR; ++q) xv[q][u] = in ? x[q][row + d] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int q = 0; q < NR; ++q) acc[q] += v[u] * xv[q][u];
            }
        }
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            for (int off = 32; off > 0; off >>= 1) acc[q] += __shfl_xor(acc[q], off);
            if (lane == 0) up[q][16 * wave + rr] = acc[q];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NR; ++q) y[q] = part[q][0][lane] + part[q][1][lane] + part[q][2][lane] + part[q][3][lane] + up[q][lane];
    __syncthreads();  // part/up are reused by the next call
}

template <typename T>
__global__ __launch_bounds__(kT) void k_symv_rows(const T *ab, int n, int bw, const double *x, double *y)
{
    const int i0 = blockIdx.x * kRows;
    const double *xs[1] = {x};
    double v[1];
    symv_row_block<T, 1>(ab, n, bw, xs, i0, v);
    if (threadIdx.x < kRows && i0 + threadIdx.x < n) y[i0 + threadIdx.x] = v[0];
}

// the descriptor that row block blk belongs to, its pointers stated to be global memory
__device__ inline RefDesc find_block(const RefDesc *d, int n, int blk)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (d[mid].blk0 <= blk) lo = mid;
        else hi = mid - 1;
    }
    RefDesc r = d[lo];
    r.ab = global_ptr(r.ab);
    r.b = global_ptr(r.b);
    r.x = global_ptr(r.x);
    r.r = global_ptr(r.r);
    r.part = global_ptr(r.part);
    r.b2 = global_ptr(r.b2);
    r.x2 = global_ptr(r.x2);
    r.r2 = global_ptr(r.r2);
    r.part2 = global_ptr(r.part2);
    r.prod = global_ptr(r.prod);
    r.prod2 = global_ptr(r.prod2);
    return r;
}

// ---- K x by column blocks, for the refinement residuals ----
// A workgroup takes 64 columns of one matrix, wave w columns 16 w .. 16 w + 15, and walks down their band
// by chunks of 64 rows (lane = row: every load is a contiguous run of one column).  An entry K[i][j] is
// read once for both of its products: K[i][j] x_j goes to the chunk's partial sum of rows i, summed over
// the block's columns and stored (prod: per column block its chunks' 64 sums), and K[i][j] x_i to
// column j's own sum, complete at the end of the walk (prod's first n entries).  k_refine_sum then adds a
// row's at most bw / 64 + 2 partial sums, in the order of the column blocks.  The band is read once
// instead of twice and the partial sums are 1 / 32 of it: HBM bound.  256 bands of half-width 182..470 in
// FP64 (3.1 GB), two vectors each: 1.61 ms by rows (every entry read for its row and again for its
// column), 0.72 ms by columns (4.4 TB/s) and 0.04 ms for the sums.
constexpr int kCols = kRows / 4;

// chunks of 64 rows that a block of 64 columns of half-width bw reaches
__host__ __device__ inline int col_chunks(int bw) { return (bw + 2 * kRows - 1) / kRows; }
__host__ __device__ inline size_t prod_doubles(int n, int bw)
{
    const size_t nblk = ((size_t)n + kRows - 1) / kRows;
    return nblk * kRows * (1 + (size_t)col_chunks(bw));
}

template <typename T, int NR>
__device__ __forceinline__ void column_block(const RefDesc &d, int lb)
{
    __shared__ double red[2][NR][4][kRows];
    const int n = d.n, bw = d.bw, j0 = lb * kRows, lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), jw = j0 + kCols * wv;
    const size_t ld = (size_t)bw + 1;
    const T *ab = (const T *)d.ab;
    const double *x[NR];
    double *prod[NR];
    x[0] = d.x;
    prod[0] = d.prod;
    if constexpr (NR > 1) {
        x[1] = d.x2;
        prod[1] = d.prod2;
    }
    double xj[NR][kCols], up[NR][kCols];
#pragma unroll
    for (int q = 0; q < NR; ++q)
#pragma unroll
        for (int u = 0; u < kCols; ++u) {
            xj[q][u] = jw + u < n ? x[q][jw + u] : 0.0;
            up[q][u] = 0.0;
        }
    const int nch = (min(n - j0, kRows + bw) + kRows - 1) / kRows;
    for (int c = 0; c < nch; ++c) {
        const int i = j0 + kRows * c + lane;
        double v[kCols], xi[NR], low[NR];
#pragma unroll
        for (int u = 0; u < kCols; ++u) {
            const int j = jw + u, o = i - j;
            const bool in = o >= 0 && o <= bw && i < n;
            const T e = ab[in ? (size_t)j * ld + (unsigned)o : 0];
            v[u] = in ? (double)e : 0.0;
        }
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            xi[q] = i < n ? x[q][i] : 0.0;
            low[q] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < kCols; ++u)
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                low[q] += v[u] * xj[q][u];
                up[q][u] += (i == jw + u ? 0.0 : v[u]) * xi[q];
            }
#pragma unroll
        for (int q = 0; q < NR; ++q) red[c & 1][q][wv][lane] = low[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NR; ++q)
            if (wv == ((c + q) & 3))
                prod[q][((size_t)d.nblk + (size_t)lb * col_chunks(bw) + c) * kRows + lane] =
                    (red[c & 1][q][0][lane] + red[c & 1][q][1][lane]) + (red[c & 1][q][2][lane] + red[c & 1][q][3][lane]);
    }
#pragma unroll
    for (int q = 0; q < NR; ++q) {
        const double t = sum_lanes(up[q], lane);
        if ((lane & 3) == 0) prod[q][jw + (lane >> 2)] = t;
    }
}

__global__ __launch_bounds__(kT) void k_refine_cols(const RefDesc *__restrict__ descs, int ninst)
{
    const RefDesc d = find_block(descs, ninst, blockIdx.x);
    if (!d.active) return;
    const int lb = blockIdx.x - d.blk0;
    if (d.sprec == KSH_FP64) {
        if (d.x2) column_block<double, 2>(d, lb);
        else column_block<double, 1>(d, lb);
    } else {
        if (d.x2) column_block<float, 2>(d, lb);
        else column_block<float, 1>(d, lb);
    }
}

// r = b - K x on one block of 64 rows, K x from the column blocks' sums, and the block's partial norms
// (||r||^2, ||b||^2); workgroup y: the first or the second vector of the descriptor
__global__ __launch_bounds__(64) void k_refine_sum(const RefDesc *__restrict__ descs, int ninst)
{
    const RefDesc d = find_block(descs, ninst, blockIdx.x);
    const bool second = blockIdx.y != 0;
    if (!d.active || (second && !d.x2)) return;
    const double *prod = second ? d.prod2 : d.prod, *b = second ? d.b2 : d.b;
    double *r = second ? d.r2 : d.r, *part = second ? d.part2 : d.part;
    const int lb = blockIdx.x - d.blk0, lane = (int)threadIdx.x, i = lb * kRows + lane;
    const int nch = col_chunks(d.bw), first = max(0, lb - nch + 1);
    const double own = prod[i];
    double y = 0.0;
    for (int J0 = first; J0 <= lb; J0 += kU) {
        double v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int J = min(J0 + u, lb);
            v[u] = prod[((size_t)d.nblk + (size_t)J * nch + (lb - J)) * kRows + lane];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (J0 + u <= lb) y += v[u];
    }
    double ri = 0.0, bi = 0.0;
    if (i < d.n) {
        bi = b[i];
        ri = bi - (y + own);
        r[i] = ri;
    }
    double rr = ri * ri, bb = bi * bi;
    for (int off = 32; off > 0; off >>= 1) {
        rr += __shfl_xor(rr, off);
        bb += __shfl_xor(bb, off);
    }
    if (lane == 0) {
        part[2 * lb] = rr;
        part[2 * lb + 1] = bb;
    }
}

// per-matrix norms from the block partials (block order), one workgroup per matrix
__global__ __launch_bounds__(64) void k_refine_norms_batched(const RefDesc *descs)
{
    const RefDesc &d = descs[blockIdx.x];
    if (!d.active) return;
    if (threadIdx.x < 2) {
        const double *part = global_ptr(threadIdx.x == 0 ? d.part : d.part2);
        double *norms = global_ptr(threadIdx.x == 0 ? d.norms : d.norms2);
        if (!part) return;
        double rr = 0.0, bb = 0.0;
        const int last = d.nblk - 1;
        for (int k0 = 0; k0 <= last; k0 += kU) {  // kU blocks' loads in flight, added in block order
            double v[kU], w[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                v[u] = part[2 * min(k0 + u, last)];
                w[u] = part[2 * min(k0 + u, last) + 1];
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (k0 + u <= last) {
                    rr += v[u];
                    bb += w[u];
                }
        }
        norms[0] = rr;
        norms[1] = bb;
    }
}

__global__ __launch_bounds__(kT) void k_refine_update_batched(const RefDesc *__restrict__ descs, int ninst)
{
    const RefDesc d = find_block(descs, ninst, blockIdx.x);
    if (!d.active) return;
    const int i = (blockIdx.x - d.blk0) * kRows + threadIdx.x;
    if (threadIdx.x < kRows && i < d.n) d.x[i] += d.r[i];
}

inline unsigned nblocks(int n) { return (unsigned)((n + kRows - 1) / kRows); }

int prefix_blocks(std::vector<RefDesc> &h)
{
    int tot = 0;
    for (auto &d : h) {
        d.blk0 = tot;
        d.nblk = (int)nblocks(d.n);
        tot += d.nblk;
    }
    return tot;
}

}  // namespace

int band_symv(const Matrix &K, const double *x_dev, double *y_dev)
{
    Problem &pb = *K.pb;
    ProfScope ps("band_symv", pb.stream);
    ps.set_work(K.n * (2.0 * K.bw + 1.0) * (K.sprec == KSH_FP64 ? 8.0 : 4.0) + 16.0 * K.n);
    if (K.sprec == KSH_FP64)
        hipLaunchKernelGGL(k_symv_rows<double>, dim3(nblocks(K.n)), dim3(kT), 0, pb.stream, (const double *)K.ab, K.n, K.bw,
                           x_dev, y_dev);
    else
        hipLaunchKernelGGL(k_symv_rows<float>, dim3(nblocks(K.n)), dim3(kT), 0, pb.stream, (const float *)K.ab, K.n, K.bw,
                           x_dev, y_dev);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

// most of the products' scratch that one launch uses; larger batches go by several launches, one after
// the other on the stream, over the same scratch
constexpr size_t kProdBytes = 512ull << 20;

int refine_residual_batch(hipStream_t s, RefDesc *d_descs, const std::vector<RefDesc> &hin, DevScratch &prod)
{
    if (hin.empty()) return KSH_SUCCESS;
    // two active jobs on the same matrix (the arc-length solves' two right-hand sides) share one
    // descriptor, so that their band is read once for both products
    std::vector<RefDesc> h;
    h.reserve(hin.size());
    std::vector<char> taken(hin.size(), 0);
    for (size_t i = 0; i < hin.size(); ++i) {
        if (taken[i]) continue;
        RefDesc d = hin[i];
        d.b2 = nullptr;
        d.x2 = d.r2 = d.norms2 = d.part2 = nullptr;
        if (d.active)
            for (size_t j = i + 1; j < hin.size(); ++j) {
                const RefDesc &e = hin[j];
                if (taken[j] || !e.active || e.ab != d.ab || e.sprec != d.sprec || e.n != d.n || e.bw != d.bw) continue;
                d.b2 = e.b;
                d.x2 = e.x;
                d.r2 = e.r;
                d.norms2 = e.norms;
                d.part2 = e.part;
                taken[j] = 1;
                break;
            }
        h.push_back(d);
    }
    // groups of descriptors [g0, g1) with their own offsets into the scratch and launch blocks
    std::vector<std::pair<size_t, size_t>> groups;
    std::vector<size_t> off(h.size());
    size_t most = 0;
    for (size_t g0 = 0; g0 < h.size();) {
        size_t used = 0, g1 = g0;
        for (; g1 < h.size(); ++g1) {
            const size_t w = h[g1].active ? prod_doubles(h[g1].n, h[g1].bw) * (h[g1].x2 ? 2 : 1) * sizeof(double) : 0;
            if (g1 > g0 && used + w > kProdBytes) break;
            off[g1] = used;
            used += w;
        }
        most = std::max(most, used);
        groups.push_back({g0, g1});
        g0 = g1;
    }
    int rc;
    if ((rc = prod.ensure(most))) return rc;
    std::vector<int> tot;
    for (const auto &g : groups) {
        int t = 0;
        for (size_t i = g.first; i < g.second; ++i) {
            RefDesc &d = h[i];
            d.blk0 = t;
            d.nblk = (int)nblocks(d.n);
            t += d.nblk;
            d.prod = (double *)((char *)prod.p + off[i]);
            d.prod2 = d.x2 ? d.prod + prod_doubles(d.n, d.bw) : nullptr;
        }
        tot.push_back(t);
    }
    KSH_HIP(hipMemcpyAsync(d_descs, h.data(), sizeof(RefDesc) * h.size(), hipMemcpyHostToDevice, s));
    {
        ProfScope ps("refine_residual_batch", s);
        double work = 0.0;  // the band read once, x and b read, r written (per vector)
        for (const auto &d : h)
            if (d.active) work += d.n * (d.bw + 1.0) * (d.sprec == KSH_FP64 ? 8.0 : 4.0) + (d.x2 ? 48.0 : 24.0) * d.n;
        ps.set_work(work);
        for (size_t g = 0; g < groups.size(); ++g) {
            const RefDesc *dd = (const RefDesc *)d_descs + groups[g].first;
            const int cnt = (int)(groups[g].second - groups[g].first);
            hipLaunchKernelGGL(k_refine_cols, dim3((unsigned)tot[g]), dim3(kT), 0, s, dd, cnt);
            hipLaunchKernelGGL(k_refine_sum, dim3((unsigned)tot[g], 2), dim3(64), 0, s, dd, cnt);
        }
    }
    KSH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_refine_norms_batched, dim3((unsigned)h.size()), dim3(64), 0, s, (const RefDesc *)d_descs);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

int refine_update_batch(hipStream_t s, RefDesc *d_descs, const std::vector<RefDesc> &hin)
{
    if (hin.empty()) return KSH_SUCCESS;
    std::vector<RefDesc> h = hin;
    int tot = prefix_blocks(h);
    KSH_HIP(hipMemcpyAsync(d_descs, h.data(), sizeof(RefDesc) * h.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_refine_update_batched, dim3((unsigned)tot), dim3(kT), 0, s, (const RefDesc *)d_descs, (int)h.size());
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

}  // namespace ksh
