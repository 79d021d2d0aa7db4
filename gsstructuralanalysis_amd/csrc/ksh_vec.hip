// ksh_vec.hip -- batched vector kernels of the path engine: dot products, linear combinations,
// and the learned predictor's modal projection / decode.
//
// Every vector of every instance of a batch lives in device memory; the engine's host logic only
// ever sees scalars.  One launch serves all instances of a round:
//   k_dots      one workgroup per instance and dot product of length n (up to kMaxDots);
//               lanes stride over the entries, then a fixed-order reduction (wave shuffles, then
//               the four wave sums in order), so results are bit-reproducible run to run;
//   k_vecops    per instance a short program of 3-term combinations dst = a x + b y + c z,
//               applied in order by each thread to its entry (so an op may read what an earlier op
//               of the same program wrote, and dst may alias x, y or z);
//   k_features  the 66 predictor features of a state: lambda, ||U||, and the 64 least-squares
//               coefficients of the out-of-plane control displacements in the analytic modes
//               (P [64][ncp] times the gathered z values);
//   k_decode    dU[z dof of cp] += scale * sum_r Phi[cp][r] coef[r];
//   k_dr        one explicit dynamic-relaxation update of an instance with its four norms.
// All are HBM / latency bound and tiny next to the assembly and the factor.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ksh_devutil.hpp"
#include "ksh_internal.hpp"
#include "ksh_vec.hpp"

namespace ksh {

namespace {

constexpr int kT = 256;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Latency bound: a workgroup holds kDots entries a lane in flight, and every product has its own
// workgroup: 18 us for the up to ten products of 256 roofs of 16..48 elements a side, 61 us with all
// of an instance's products in one workgroup, one entry a lane at a time.
constexpr int kDots = 8;

__global__ __launch_bounds__(kT) void k_dots(const DotDesc *__restrict__ descs)
{
    const DotDesc &D = descs[blockIdx.x];
    const int k = blockIdx.y, n = D.n;
    if (k >= D.npairs) return;
    const double *a = global_ptr(D.a[k]), *b = global_ptr(D.b[k]);
    double acc = 0.0;
    for (int i0 = threadIdx.x; i0 < n; i0 += kDots * kT) {
        double va[kDots], vb[kDots];
#pragma unroll
        for (int q = 0; q < kDots; ++q) {
            const int i = min(i0 + q * kT, n - 1);
            va[q] = a[i];
            vb[q] = b[i];
        }
#pragma unroll
        for (int q = 0; q < kDots; ++q)
            if (i0 + q * kT < n) acc += va[q] * vb[q];
    }
    __shared__ double part[kT / 64];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    acc = wave_sum(acc);
    if (lane == 0) part[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kT / 64; ++w) s += part[w];
        global_ptr(D.out)[k] = s;
    }
}

__global__ __launch_bounds__(kT) void k_vecops(const VecDesc *__restrict__ descs)
{
    const VecDesc &D = descs[blockIdx.y];
    const int i = blockIdx.x * kT + threadIdx.x;
    if (i >= D.n) return;
    for (int k = 0; k < D.nops; ++k) {
        const VecOp o = D.op[k];
        double v = 0.0;
        if (o.x) v = o.a * global_ptr(o.x)[i];
        if (o.y) v += o.b * global_ptr(o.y)[i];
        if (o.z) v += o.c * global_ptr(o.z)[i];
        global_ptr(o.dst)[i] = v;
    }
}

constexpr int kChunk = 2048;  // control points staged in LDS per pass

__global__ __launch_bounds__(kT) void k_features(const FeatDesc *__restrict__ descs)
{
    FeatDesc D = descs[blockIdx.x];
    D.P = global_ptr(D.P);
    D.zfree = global_ptr(D.zfree);
    D.U = global_ptr(D.U);
    D.out = global_ptr(D.out);
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    __shared__ double z[kChunk];
    __shared__ double red[kT / 64];
    // ||U||
    double acc = 0.0;
    for (int i = threadIdx.x; i < D.nfree; i += kT) acc += D.U[i] * D.U[i];
    acc = wave_sum(acc);
    if (lane == 0) red[wave] = acc;
    // coefficients: wave w owns r = w, w + 4, ... (16 of the 64)
    double coef[kModalCoef / 4];
#pragma unroll
    for (int q = 0; q < kModalCoef / 4; ++q) coef[q] = 0.0;
    for (int c0 = 0; c0 < D.ncp; c0 += kChunk) {
        const int cn = min(kChunk, D.ncp - c0);
        __syncthreads();
        for (int c = threadIdx.x; c < cn; c += kT) {
            const int f = D.zfree[c0 + c];
            z[c] = f >= 0 ? D.U[f] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kModalCoef / 4; ++q) {
            const int r = wave + 4 * q;
            const double *P = D.P + (size_t)r * D.ncp + c0;
            double s = 0.0;
            for (int c = lane; c < cn; c += 64) s += P[c] * z[c];
            coef[q] += s;
        }
    }
#pragma unroll
    for (int q = 0; q < kModalCoef / 4; ++q) {
        const double s = wave_sum(coef[q]);
        if (lane == 0) D.out[2 + wave + 4 * q] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kT / 64; ++w) s += red[w];
        D.out[0] = D.lambda;
        D.out[1] = sqrt(s);
    }
}

__global__ __launch_bounds__(kT) void k_decode(const DecDesc *__restrict__ descs)
{
    DecDesc D = descs[blockIdx.y];
    D.Phi = global_ptr(D.Phi);
    D.zfree = global_ptr(D.zfree);
    D.coef = global_ptr(D.coef);
    D.dU = global_ptr(D.dU);
    const int c = blockIdx.x * kT + threadIdx.x;
    if (c >= D.ncp) return;
    const int f = D.zfree[c];
    if (f < 0) return;
    const double *phi = D.Phi + (size_t)c * kModalCoef;
    double s = 0.0;
#pragma unroll 8
    for (int r = 0; r < kModalCoef; ++r) s += phi[r] * D.coef[r];
    D.dU[f] += D.scale * s;
}

// One workgroup per instance (its norms need no second launch), so the largest instance's chain of
// memory latencies is its time: each lane has kDr entries of every vector in flight.  Over 64 roofs
// of 16..48 elements a side, one entry at a time took 51 us; 14 us.
constexpr int kDr = 8;

__global__ __launch_bounds__(kT) void k_dr(const DrDesc *__restrict__ descs)
{
    const DrDesc D = descs[blockIdx.x];
    const double *R = global_ptr(D.R), *m = global_ptr(D.m), *minv = global_ptr(D.minv), *damp = global_ptr(D.damp);
    const double *U = global_ptr(D.U);
    double *gv = global_ptr(D.v), *gdU = global_ptr(D.dU), *gDU = global_ptr(D.DU), *X = global_ptr(D.X);
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    __shared__ double red[4][kT / 64];
    const double dt = D.dt;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i0 = threadIdx.x; i0 < D.n; i0 += kDr * kT) {
        double lr[kDr], lv[kDr], lmi[kDr], lm[kDr], ld[kDr], lU[kDr], lD[kDr];
#pragma unroll
        for (int q = 0; q < kDr; ++q) {
            const int i = min(i0 + q * kT, D.n - 1);
            lr[q] = R[i];
            lv[q] = gv[i];
            lmi[q] = minv[i];
            lm[q] = m[i];
            ld[q] = D.mode != 0 ? damp[i] : 0.0;
            lU[q] = U[i];
            lD[q] = gDU[i];
        }
#pragma unroll
        for (int q = 0; q < kDr; ++q) {
            const int i = i0 + q * kT;
            if (i >= D.n) break;
            double r = lr[q], v = lv[q], du;
            if (D.mode == 0) {
                du = 0.5 * dt * dt * lmi[q] * r;
                v = du / dt;
            } else if (D.mode == 1) {
                r -= ld[q] * v;
                v += dt * lmi[q] * r;
                du = dt * v;
            } else {
                r -= ld[q] * v;
                du = -1.5 * dt * v + 0.5 * dt * dt * lmi[q] * r;
                v = 0.0;
            }
            const double DU = lD[q] + du;
            gv[i] = v;
            gdU[i] = du;
            gDU[i] = DU;
            X[i] = lU[q] + DU;
            s[0] += r * r;
            s[1] += v * (lm[q] * v);
            s[2] += du * du;
            s[3] += DU * DU;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const double w = wave_sum(s[q]);
        if (lane == 0) red[q][wave] = w;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < kT / 64; ++w) t += red[threadIdx.x][w];
        global_ptr(D.out)[threadIdx.x] = t;
    }
}

template <typename Desc>
int upload_descs(hipStream_t s, DevScratch &buf, const std::vector<Desc> &h)
{
    int rc;
    if ((rc = buf.ensure(h.size() * sizeof(Desc)))) return rc;
    KSH_HIP(hipMemcpyAsync(buf.p, h.data(), h.size() * sizeof(Desc), hipMemcpyHostToDevice, s));
    return KSH_SUCCESS;
}

}  // namespace

int DevScratch::ensure(size_t b)
{
    if (b <= bytes) return KSH_SUCCESS;
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    KSH_HIP(hipMalloc(&p, b));
    bytes = b;
    return KSH_SUCCESS;
}

DevScratch::~DevScratch()
{
    if (p) (void)hipFree(p);
}

int batch_dots(hipStream_t s, DevScratch &desc_buf, const std::vector<DotDesc> &h)
{
    if (h.empty()) return KSH_SUCCESS;
    for (const DotDesc &d : h)
        if (d.npairs < 0 || d.npairs > kMaxDots || d.n < 0 || !d.out) return fail(KSH_OTHER_ERROR, "dot descriptor");
    int rc;
    if ((rc = upload_descs(s, desc_buf, h))) return rc;
    int most = 1;
    for (const DotDesc &d : h) most = std::max(most, d.npairs);
    hipLaunchKernelGGL(k_dots, dim3((unsigned)h.size(), (unsigned)most), dim3(kT), 0, s, (const DotDesc *)desc_buf.p);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

int batch_vecops(hipStream_t s, DevScratch &desc_buf, const std::vector<VecDesc> &h)
{
    if (h.empty()) return KSH_SUCCESS;
    int nmax = 0;
    for (const VecDesc &d : h) {
        if (d.nops < 0 || d.nops > kMaxVecOps) return fail(KSH_OTHER_ERROR, "vector program too long");
        nmax = std::max(nmax, d.n);
    }
    if (nmax == 0) return KSH_SUCCESS;
    int rc;
    if ((rc = upload_descs(s, desc_buf, h))) return rc;
    hipLaunchKernelGGL(k_vecops, dim3((unsigned)((nmax + kT - 1) / kT), (unsigned)h.size()), dim3(kT), 0, s,
                       (const VecDesc *)desc_buf.p);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

int batch_dr(hipStream_t s, DevScratch &desc_buf, const std::vector<DrDesc> &h)
{
    if (h.empty()) return KSH_SUCCESS;
    for (const DrDesc &d : h)
        if (d.n < 0 || d.mode < 0 || d.mode > 2 || !d.out) return fail(KSH_OTHER_ERROR, "dynamic relaxation descriptor");
    int rc;
    if ((rc = upload_descs(s, desc_buf, h))) return rc;
    hipLaunchKernelGGL(k_dr, dim3((unsigned)h.size()), dim3(kT), 0, s, (const DrDesc *)desc_buf.p);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

int batch_features(hipStream_t s, DevScratch &desc_buf, const std::vector<FeatDesc> &h)
{
    if (h.empty()) return KSH_SUCCESS;
    int rc;
    if ((rc = upload_descs(s, desc_buf, h))) return rc;
    hipLaunchKernelGGL(k_features, dim3((unsigned)h.size()), dim3(kT), 0, s, (const FeatDesc *)desc_buf.p);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

int batch_decode(hipStream_t s, DevScratch &desc_buf, const std::vector<DecDesc> &h)
{
    if (h.empty()) return KSH_SUCCESS;
    int cmax = 0;
    for (const DecDesc &d : h) cmax = std::max(cmax, d.ncp);
    if (cmax == 0) return KSH_SUCCESS;
    int rc;
    if ((rc = upload_descs(s, desc_buf, h))) return rc;
    hipLaunchKernelGGL(k_decode, dim3((unsigned)((cmax + kT - 1) / kT), (unsigned)h.size()), dim3(kT), 0, s,
                       (const DecDesc *)desc_buf.p);
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

}  // namespace ksh
