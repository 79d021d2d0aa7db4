// ksh_solve_tiled.hip -- L D L^T solve of one large band spread over many workgroups.
//
// For bands too long for the LDS-resident kernel (vector over 160 KB) or wider than its 512
// prefetched columns -- e.g. the 128 x 128 degree-3 plate, n = 51k, bw = 1190, whose band is
// about 0.5 GB in FP64 -- a single workgroup would stream the band at one CU's bandwidth.  Here
// each 64-row step of a sweep is one launch whose workgroups share the rows the step touches:
//   forward, block c0..c0+63 (rows after it already hold b - L y of the earlier blocks):
//     every workgroup solves the unit-lower diagonal block for y (wave 0, lane = row,
//     v_readlane broadcasts; the block is read from L2), workgroup 0 stores z = D^-1 y, and each
//     workgroup takes 64 of the following bw rows: b[r] -= sum_k L[r][c0+k] y_k (lanes = rows,
//     so each load reads 64 consecutive entries of a band column);
//   backward, block c0..c0+63 from the last block down (z of the block already holds
//     D^-1 y - sum over later blocks): every workgroup solves the transposed diagonal block for
//     x, workgroup 0 stores it, and each workgroup takes 64 of the preceding bw rows:
//     z[i] -= sum_k L[c0+k][i] x_k (lanes = k, so each load reads 64 consecutive entries of
//     column i; the 64 x 64 products are summed per row through LDS).
// Rows touched by one launch belong to one workgroup, and the block rows are read but not
// written, so launches on one stream need no other synchronization.  HBM traffic: the band once
// per sweep, 2 n (bw+1) entries per solve.  Single bands take the resident teams (ksh_solve_team.hip: one
// launch, 2.3 ms against 11.2 on that plate); these launches serve a device without room for
// the team's workspace, and KSH_BAND_PATH=tiled.  Replaces
// SimplicialLDLT::solve
// (src/gsEigenSolvers/gsEigenProblemBase.hpp:152-216 drives it through the shift-invert operator).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ksh_devutil.hpp"
#include "ksh_internal.hpp"

namespace ksh {

namespace {

constexpr int kSB = 64;  // rows per step = threads per workgroup

// Band entries of one step: they do not depend on the solution, so all of a step's loads are issued
// together.
template <typename T>
struct StepRegs {
    T l[kSB];  // diagonal block (forward: row lane; backward: column lane)
    T u[kSB];  // this workgroup's off-diagonal rows / columns
    T d;       // pivot (forward)
};

// forward, block c0: lane ii holds row c0+ii of the diagonal block, L[c0+ii][c0+jj] for jj < ii;
// the workgroup's rows c0+r, r = w + 64 wg + lane, their entries L[c0+r][c0+kk]
template <typename T>
__device__ __forceinline__ void fwd_load_diag(const T *fac, int n, int bw, int c0, StepRegs<T> &q)
{
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0);
#pragma unroll
    for (int jj = 0; jj < kSB; ++jj) {
        const bool ok = jj < lane && lane < w && lane - jj <= bw;
        q.l[jj] = load_if<T>(ok, rs, ((unsigned)(c0 + jj) * ldu + (unsigned)(lane - jj)) * es);
    }
    q.d = load_if<T>(lane < w, rs, (unsigned)(c0 + lane) * ldu * es);
}

template <typename T>
__device__ __forceinline__ void fwd_load_rows(const T *fac, int n, int bw, int c0, int wg, StepRegs<T> &q)
{
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0), nr = min(n - c0, w + bw);
    const int r = w + kSB * wg + lane;
#pragma unroll
    for (int kk = 0; kk < kSB; ++kk) {
        const bool ok = kk < w && r < nr && r - kk <= bw;
        q.u[kk] = load_if<T>(ok, rs, ((unsigned)(c0 + kk) * ldu + (unsigned)(r - kk)) * es);
    }
}

template <typename T>
__device__ __forceinline__ void fwd_load(const T *fac, int n, int bw, int c0, int wg, StepRegs<T> &q)
{
    fwd_load_diag<T>(fac, n, bw, c0, q);
    fwd_load_rows<T>(fac, n, bw, c0, wg, q);
}

template <typename T>
__device__ __forceinline__ void fwd_compute(int n, int bw, int c0, double *b, double *z, int wg, const StepRegs<T> &q)
{
    __shared__ double ys[kSB];
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0), nr = min(n - c0, w + bw);
    const int r = w + kSB * wg + lane;
    const double rb = r < nr ? b[c0 + r] : 0.0;
    double y = lane < w ? b[c0 + lane] : 0.0;
#pragma unroll
    for (int jj = 0; jj < kSB - 1; ++jj) y -= (double)q.l[jj] * readlane_f64(y, jj);  // l = 0 on and above the diagonal
    ys[lane] = y;
    if (wg == 0 && lane < w) z[c0 + lane] = y / (double)q.d;
    __syncthreads();
    double acc = 0.0;
#pragma unroll
    for (int kk = 0; kk < kSB; ++kk) acc += (double)q.u[kk] * ys[kk];
    if (r < nr) b[c0 + r] = rb - acc;
}

template <typename T>
__global__ __launch_bounds__(kSB) void k_band_fwd_step(const T *fac, int n, int bw, int c0, double *b, double *z)
{
    StepRegs<T> q;
    fwd_load<T>(fac, n, bw, c0, (int)blockIdx.x, q);
    fwd_compute<T>(n, bw, c0, b, z, (int)blockIdx.x, q);
}

// backward, block c0: lane jj holds column c0+jj of the transposed diagonal block,
// L[c0+kk][c0+jj] for kk > jj; rows i = c0 - 1 - (64 wg + q) above the block, L[c0+k][i] (lane = k)
template <typename T>
__device__ __forceinline__ void bwd_load_diag(const T *fac, int n, int bw, int c0, StepRegs<T> &q)
{
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0);
#pragma unroll
    for (int kk = 0; kk < kSB; ++kk) {
        const bool ok = kk > lane && kk < w && kk - lane <= bw;
        q.l[kk] = load_if<T>(ok, rs, ((unsigned)(c0 + lane) * ldu + (unsigned)(kk - lane)) * es);
    }
}

template <typename T>
__device__ __forceinline__ void bwd_load_rows(const T *fac, int n, int bw, int c0, int wg, StepRegs<T> &q)
{
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0);
    const int lo = max(0, c0 - bw);
#pragma unroll
    for (int qq = 0; qq < kSB; ++qq) {
        const int i = c0 - 1 - (kSB * wg + qq);
        const bool ok = i >= lo && lane < w && c0 + lane - i <= bw;
        q.u[qq] = load_if<T>(ok, rs, ((unsigned)max(i, 0) * ldu + (unsigned)(c0 + lane - max(i, 0))) * es);
    }
}

template <typename T>
__device__ __forceinline__ void bwd_load(const T *fac, int n, int bw, int c0, int wg, StepRegs<T> &q)
{
    bwd_load_diag<T>(fac, n, bw, c0, q);
    bwd_load_rows<T>(fac, n, bw, c0, wg, q);
}

template <typename T>
__device__ __forceinline__ void bwd_compute(int n, int bw, int c0, double *z, double *x, int wg, const StepRegs<T> &q)
{
    __shared__ double prod[kSB][kSB + 1];
    const int lane = threadIdx.x;
    const int w = min(kSB, n - c0);
    const int lo = max(0, c0 - bw);
    double xv = lane < w ? z[c0 + lane] : 0.0;
#pragma unroll
    for (int kk = kSB - 1; kk > 0; --kk) xv -= (double)q.l[kk] * readlane_f64(xv, kk);  // l = 0 on and below the diagonal
    if (wg == 0 && lane < w) x[c0 + lane] = xv;
#pragma unroll
    for (int qq = 0; qq < kSB; ++qq) prod[qq][lane] = (double)q.u[qq] * xv;  // masked entries loaded as 0
    __syncthreads();
    const int i = c0 - 1 - (kSB * wg + lane);
    double s = 0.0;
#pragma unroll 16
    for (int k = 0; k < kSB; ++k) s += prod[lane][k];
    if (i >= lo) z[i] -= s;
}

template <typename T>
__global__ __launch_bounds__(kSB) void k_band_bwd_step(const T *fac, int n, int bw, int c0, double *z, double *x)
{
    StepRegs<T> q;
    bwd_load<T>(fac, n, bw, c0, (int)blockIdx.x, q);
    bwd_compute<T>(n, bw, c0, z, x, (int)blockIdx.x, q);
}

template <typename T>
int run_solve(hipStream_t s, const T *fac, int n, int bw, double *x, double *z)
{
    for (int c0 = 0; c0 < n; c0 += kSB) {
        const int w = std::min(kSB, n - c0), nr = std::min(n - c0, w + bw);
        const unsigned grid = (unsigned)std::max(1, (nr - w + kSB - 1) / kSB);
        hipLaunchKernelGGL(k_band_fwd_step<T>, dim3(grid), dim3(kSB), 0, s, fac, n, bw, c0, x, z);
    }
    for (int c0 = ((n - 1) / kSB) * kSB; c0 >= 0; c0 -= kSB) {
        const int above = std::min(c0, bw);
        const unsigned grid = (unsigned)std::max(1, (above + kSB - 1) / kSB);
        hipLaunchKernelGGL(k_band_bwd_step<T>, dim3(grid), dim3(kSB), 0, s, fac, n, bw, c0, z, x);
    }
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

}  // namespace

int band_solve_tiled(hipStream_t s, const void *fac, int prec, int n, int bw, double *x, double *z)
{
    const size_t es = prec == KSH_FP64 ? sizeof(double) : sizeof(float);
    if ((size_t)n * (size_t)(bw + 1) * es >= 0x80000000ull)
        return fail(KSH_SOLVER_ERROR, "band of 2 GiB or more: beyond the band kernels' 32-bit offsets");
    return prec == KSH_FP64 ? run_solve<double>(s, (const double *)fac, n, bw, x, z)
                            : run_solve<float>(s, (const float *)fac, n, bw, x, z);
}

}  // namespace ksh
