// ksh_solve_team.hip -- L D L^T solve of one band by a team of workgroups.
//
// A band solve is a chain: 64-row block k needs the solution of the block before it.  One workgroup
// per band (ksh_solve.hip) streams the whole band through one CU, 5 us per block and sweep at half-width
// 326; a launch per block (ksh_solve_tiled.hip) costs 7 us a block.  Here a team stays resident for
// the whole solve: its leader walks the chain, its helpers form what does not sit on it.
//   forward, block k:  y_k = c_k - Q_k y_{k-1}, Q_k = M_k L_{k,k-1}, M_k = L_kk^-1;
//     c_k = M_k (b_k - sum over j <= k - 2 of L_kj y_j), by a helper;
//   backward, block k: x_k = c_k - P_k x_{k+1}, P_k = M_k^T L_{k+1,k}^T;
//     c_k = M_k^T (y_k / d_k - sum over i >= k + 2 of L_ik^T x_i), by a helper.
// M_k, Q_k and P_k (64 x 64) are formed beforehand by k_team_prep, all blocks at once.  A leader step is
// one 64 x 64 product spread over its four waves with one LDS exchange: no recurrence over single
// rows, and 32 KB to load (loaded three blocks ahead; 1,400-1,600 cycles a step when nothing else holds it).
// Helper h takes blocks h, h + H, ...; it runs ahead of the chain, its band
// entries loaded four blocks ahead, and waits only for the last solution blocks.
//
// Solution blocks and the helpers' c_k travel through memory by relaxed device-scope atomics that carry the
// data itself: every slot starts as a sentinel (a signalling NaN pattern no arithmetic produces), and a
// reader polls its slot until the value is there, so one store and one load pass a block on, with
// no flag, fence or cache write-back.  A team's workgroups are placed on one XCD (workgroup ids equal
// mod 8), whose L2 passes the blocks on; placement is for speed only, the atomics are correct from
// any CU.
//
// Progress.  Nothing waits for a workgroup that is not running: workgroups register as they start, the
// leader (the first) waits a bounded time for S of them and closes the team with those it has, and
// later ones leave at once.  A leader without helpers forms the c_k itself.  Every poll is bounded
// all the same.  Past the bound a workgroup goes on with NaN, which reaches every later block of the chain:
// a leader that ends with NaN does the whole solve again without helpers, over slots of its own: later,
// and with the same bits (or with the NaN that the right-hand side or the factor holds).
//
// Replaces SimplicialLDLT::solve (src/gsALMSolvers/gsALMBase.hpp:200-211,
// src/gsStaticSolvers/gsStaticNewton.hpp:215-240, src/gsEigenSolvers/gsEigenProblemBase.hpp:152-216).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "ksh_devutil.hpp"
#include "ksh_internal.hpp"
#include "ksh_mfma.hpp"
#include "ksh_profile.hpp"
#include "ksh_team_order.hpp"

namespace ksh {

namespace {

typedef double ksh_f64x2 __attribute__((ext_vector_type(2)));

constexpr int kB = 64;               // rows per block
constexpr int kTW = 4;               // waves per workgroup (the step is bound by instruction issue: one wave per SIMD)
constexpr int kU = kB / kTW;         // columns of a block per wave
constexpr int kAhead = 4;            // blocks a helper loads ahead
constexpr int kLead = 3;             // blocks the leader loads ahead
constexpr unsigned long long kSentinel = 0x7FF7A5A5A5A5A5A5ull;
constexpr unsigned kPollLimit = 1u << 16;  // polls of one slot (tens of ms), then its reader stops waiting
constexpr unsigned kFormLimit = 64;        // polls of the team's forming (tens of us)

struct TeamDesc {
    const void *fac;
    double *x;                   // right-hand side in, solution out
    int n, bw;
    unsigned *ctl;               // [0] registered workgroups, [1] team size once closed
    // vectors padded to 64: the right-hand side; then the team's slots of the forward solution, the solution,
    // the forward and the backward c_k; then the same four of a leader without helpers
    double *b;
    double *mat;                 // per block four 64 x 64: M_k, M_k^T, Q_k, P_k (see mat_at)
};
constexpr int kM = 0, kMt = 1, kMq = 2, kMp = 3;
// entry (row, col) of such a matrix: pairs of columns interleaved, so that a lane (= row) loads 16 bytes
__host__ __device__ constexpr int mat_at(int row, int col) { return (col >> 1) * 128 + 2 * row + (col & 1); }

// The team's kernel takes its pointers as what they are, global memory: through generic ones every access would
// be a flat one, which drains every load in flight at each wait.
typedef __attribute__((address_space(1))) double gdouble;
typedef __attribute__((address_space(1))) const double cgdouble;
typedef __attribute__((address_space(1))) unsigned long long gu64;
typedef __attribute__((address_space(1))) const unsigned long long cgu64;
typedef __attribute__((address_space(1))) unsigned gu32;
typedef __attribute__((address_space(1))) const ksh_f64x2 cgf64x2;

constexpr int kSlotVecs = 8;
__host__ __device__ constexpr size_t pad_rows(int n) { return ((size_t)n + kB - 1) / kB * kB; }

struct TeamMem {
    gdouble *x, *b, *y, *xo, *cf, *cb, *mat;
    __device__ TeamMem(const TeamDesc &d, bool alone) : x((gdouble *)d.x), b((gdouble *)d.b), mat((gdouble *)d.mat)
    {
        const size_t np = pad_rows(d.n);
        y = b + np * (alone ? 5 : 1);
        xo = y + np;
        cf = xo + np;
        cb = cf + np;
    }
};

__device__ __forceinline__ double slot_load(cgdouble *p)
{
    return __builtin_bit_cast(double, __hip_atomic_load((cgu64 *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ bool slot_empty(double v) { return __builtin_bit_cast(unsigned long long, v) == kSentinel; }
__device__ __forceinline__ void slot_store(gdouble *p, double v)
{
    unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    if (b == kSentinel) b = 0x7FF8000000000000ull;
    __hip_atomic_store((gu64 *)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A wave's waits: `gone`, once a slot did not come within `limit` polls, ends all later ones after one poll.
struct Poll {
    unsigned limit;
    bool gone;
};
// v, a value of *p read before, once it is there (whole wave), else NaN.  The
// first look is outside the polling loop: inside it every wait is for the loop's own load, which would
// drain the band entries loaded ahead.
__device__ __forceinline__ double slot_spin(cgdouble *p, Poll &poll)
{
    double v;
    unsigned it = 0;
    do {
        v = slot_load(p);
        poll.gone = poll.gone || ++it > poll.limit;
    } while (__any(slot_empty(v)) && !poll.gone);
    return slot_empty(v) ? __builtin_nan("") : v;
}
__device__ __forceinline__ double slot_wait(cgdouble *p, double v, Poll &poll)
{
    if (__any(slot_empty(v))) v = slot_spin(p, poll);
    return v;
}

// sum over the four lanes l % 16 + 16 g, in all of them
__device__ __forceinline__ double sum_groups(double v)
{
    v = swap_add16(v, v);
    return swap_add32(v, v);
}
// acc + sum_u v(lane u of each 16-lane row) l[u]: the broadcast is part of the multiply-add (DPP).  The wait
// at the head covers the write of v (two wait states before a DPP read).
__device__ __forceinline__ double dot_bcast(double acc, double v, const double (&l)[kU])
{
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l0] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l1] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l2] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l3] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l4] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l5] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l6] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l7] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l8] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l9] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l10] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l11] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l12] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l13] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l14] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %[a], %[v], %[l15] row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
        : [a] "+v"(acc)
        : [v] "v"(v), [l0] "v"(l[0]), [l1] "v"(l[1]), [l2] "v"(l[2]), [l3] "v"(l[3]), [l4] "v"(l[4]), [l5] "v"(l[5]), [l6] "v"(l[6]), [l7] "v"(l[7]), [l8] "v"(l[8]), [l9] "v"(l[9]), [l10] "v"(l[10]), [l11] "v"(l[11]), [l12] "v"(l[12]), [l13] "v"(l[13]), [l14] "v"(l[14]), [l15] "v"(l[15]));
    return acc;
}
__device__ __forceinline__ double dot_bcast(double acc, double v, const float (&l)[kU])
{
    double w[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) w[u] = (double)l[u];
    return dot_bcast(acc, v, w);
}

// ---- M_k, Q_k, P_k of every block, and the slots of a solve ------------------------------------------
// One workgroup of four waves per block.  Wave c inverts the unit lower 16 x 16 block c by rows (lane =
// row, 120 multiply-adds with the block's entries broadcast from LDS); then wave w solves L X = I for
// columns 16 w .. 16 w + 15 by 16-row blocks on MFMA, substitution between them.  Q_k and P_k^T = L_{k+1,k}
// M_k are products on MFMA.  FP64 for both factor precisions.
template <typename T>
__global__ __launch_bounds__(256) void k_team_prep(TeamDesc d)
{
    using M = Mfma16<double>;
    constexpr int Q = 16;
    __shared__ double ls[kB][kB + 1];  // L[r0 + i][r0 + j], zero on and above the diagonal; then L_{k+1,k}
    __shared__ double ns[kB][kB + 1];  // L_{k,k-1}
    __shared__ double ms[kB][kB + 1];  // M_k
    __shared__ double op[4][4 * 64];   // inverse of 16 x 16 block c as an MFMA operand
    const int n = d.n, bw = d.bw;
    const int k = (int)blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r0 = k * kB;
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(d.fac, (unsigned)((size_t)n * ldu * es));
    // lane = row: a block's column is contiguous
    T v[kB / 4], v1[kB / 4], v2[kB / 4];
#pragma unroll
    for (int q = 0; q < kB / 4; ++q) {
        const int j = 4 * q + wv, i = lane;
        v[q] = load_if<T>(i > j && r0 + i < n && i - j <= bw, rs, ((unsigned)(r0 + j) * ldu + (unsigned)(i - j)) * es);
        const int o = kB + i - j;  // row minus column one block off
        v1[q] = load_if<T>(k > 0 && r0 + i < n && o <= bw, rs, ((unsigned)(r0 - kB + j) * ldu + (unsigned)o) * es);
        v2[q] = load_if<T>(r0 + kB + i < n && o <= bw, rs, ((unsigned)(r0 + j) * ldu + (unsigned)o) * es);
    }
    if (tid < kB) {
        const double empty = __builtin_bit_cast(double, kSentinel);
        double *p = d.b + r0 + tid;
        *p = r0 + tid < n ? d.x[r0 + tid] : 0.0;
#pragma unroll
        for (int q = 0; q < kSlotVecs; ++q) *(p += pad_rows(n)) = empty;
        if (k == 0 && tid < 2) d.ctl[tid] = 0;
    }
#pragma unroll
    for (int q = 0; q < kB / 4; ++q) {
        ls[lane][4 * q + wv] = (double)v[q];
        ns[lane][4 * q + wv] = (double)v1[q];
    }
    __syncthreads();
    {
        // row li of the inverse: w[c] = [c = li] - sum_{q > c} w[q] L[q][c]
        double w[Q];
#pragma unroll
        for (int c = Q - 1; c >= 0; --c) {
            double s = c == li ? 1.0 : 0.0;
#pragma unroll
            for (int q = Q - 1; q > c; --q) s -= w[q] * ls[Q * wv + q][Q * wv + c];
            w[c] = s;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {  // column krow(l, s) = l / 16 + 4 s
            const double lo = lk == 0 ? w[4 * s] : w[4 * s + 1], hi = lk == 2 ? w[4 * s + 2] : w[4 * s + 3];
            op[wv][s * 64 + lane] = lk < 2 ? lo : hi;
        }
    }
    __syncthreads();
    double *out = d.mat + (size_t)k * 4 * kB * kB;
    const int col = Q * wv + li;  // this lane's column of the results
    M::acc_t x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        M::acc_t t = {0.0, 0.0, 0.0, 0.0};
        if (c == wv) {
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = M::row(lane, e) == li ? 1.0 : 0.0;
        }
#pragma unroll
        for (int e = 0; e < c; ++e)
#pragma unroll
            for (int s = 0; s < 4; ++s) t = M::run(-ls[Q * c + li][Q * e + M::row(lane, s)], x[e][s], t);
        const M::acc_t zero = {0.0, 0.0, 0.0, 0.0};
        x[c] = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) x[c] = M::run(op[c][s * 64 + lane], t[s], x[c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = Q * c + M::row(lane, e);
            ms[row][col] = x[c][e];
            out[kM * kB * kB + mat_at(row, col)] = x[c][e];
            out[kMt * kB * kB + mat_at(col, row)] = x[c][e];
        }
    }
    __syncthreads();  // ms complete, ls free
#pragma unroll
    for (int q = 0; q < kB / 4; ++q) ls[lane][4 * q + wv] = (double)v2[q];
    auto product = [&](const double (&a)[kB][kB + 1], const double (&b)[kB][kB + 1], M::acc_t (&r)[4]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = M::acc_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int kk = Q * e + M::row(lane, s);
                const double bv = b[kk][col];
#pragma unroll
                for (int c = 0; c < 4; ++c) r[c] = M::run(a[Q * c + li][kk], bv, r[c]);
            }
    };
    product(ms, ns, x);  // Q_k
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) out[kMq * kB * kB + mat_at(Q * c + M::row(lane, e), col)] = x[c][e];
    __syncthreads();  // L_{k+1,k} staged
    product(ls, ms, x);  // P_k^T
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) out[kMp * kB * kB + mat_at(col, Q * c + M::row(lane, e))] = x[c][e];
}

// ---- the team ---------------------------------------------------------------------------------------
template <typename T>
struct Band {
    __amdgpu_buffer_rsrc_t rs;
    int n, bw, nblk, lane, wv;
};

// entries L[64 ib + lane][64 jb + 16 wv + u] of the band, u < 16 (zero outside it, and everywhere if !on).
// Straight-line: a uniform branch around the masks makes the compiler copy the loaded registers, which waits
// for the loads at once.
template <typename T>
__device__ __forceinline__ void load_cols(const Band<T> &B, int ib, int jb, bool on, T (&dst)[kU])
{
    constexpr unsigned es = sizeof(T);
    const int i0 = kB * ib, j0 = kB * jb + kU * B.wv;
    unsigned so = ((unsigned)j0 * (unsigned)B.bw + (unsigned)i0) * es;  // element (i, j) is j bw + i
    const unsigned ds = (unsigned)B.bw * es, vo = (unsigned)B.lane * es;
    const int rows = on ? B.n - 1 - i0 : -1;  // column u: lanes up to min(rows, in + u)
    int in = B.bw + j0 - i0;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
        dst[u] = load_vs<T>(B.rs, B.lane <= min(rows, in) ? vo : kMaskedOff, so);
        so += ds;
        ++in;
    }
}

struct TeamLds {
    double far[kTW][kB];   // partial sums of the helper's exchanges
    double part[kTW][kB];
    double lead[kLeadBuffers][kTW][kB];  // of the leader's, by lead_buffer (one barrier a step, in and between the sweeps)
    double vec[kTW][kU];
    unsigned team, rank, nan;
};

// sixteen columns of one of block k's matrices: entries [lane][16 wv + u]
__device__ __forceinline__ void load_mat(const TeamMem &d, int k, int which, int wv, int lane, double (&dst)[kU])
{
    cgf64x2 *m = (cgf64x2 *)(d.mat + ((size_t)k * 4 + which) * (kB * kB) + (size_t)(kU * wv) * kB);
#pragma unroll
    for (int u = 0; u < kU; u += 2) {
        const ksh_f64x2 v = m[(unsigned)(u / 2 * kB + lane)];
        dst[u] = v.x;
        dst[u + 1] = v.y;
    }
}

// c_k of the forward sweep for blocks k0, k0 + step, ... < k1
template <typename T>
__device__ __forceinline__ void help_forward(const Band<T> &B, const TeamMem &d, TeamLds &sh, int k0, int step, int k1, Poll &poll)
{
    const int lane = B.lane, wv = B.wv, jl = kU * wv + (lane & 15);
    double m[kU], rhs = 0.0;
    auto begin = [&](int k) {  // what the block needs at its end
        load_mat(d, k, kM, wv, lane, m);
        rhs = d.b[kB * k + jl];
    };
    auto finish = [&](int k, double acc) {
        sh.far[wv][lane] = acc;
        lds_barrier();
        const double t = rhs - sum_groups(sh.far[lane >> 4][jl]);
        sh.part[wv][lane] = dot_bcast(0.0, t, m);
        lds_barrier();
        if (wv == 0)
            slot_store(d.cf + kB * k + lane, (sh.part[0][lane] + sh.part[1][lane]) + (sh.part[2][lane] + sh.part[3][lane]));
    };
    int k = k0;
    for (; k < k1 && (k < 2 || B.bw <= kB); k += step) {  // blocks without far entries
        begin(k);
        finish(k, 0.0);
    }
    if (k >= k1) return;
    auto first = [&](int q) { return max(0, kB * q - B.bw) / kB; };
    T l[kAhead][kU];
    double yv[kAhead];
    int kl = k, jb = first(k);  // next block to load
    auto fill = [&](int p) {
        const bool on = kl < k1;
        load_cols<T>(B, on ? kl : 0, on ? jb : 0, on, l[p]);
        yv[p] = slot_load(d.y + (on ? kB * jb : 0) + jl);
        if (on && ++jb > kl - 2) {
            kl += step;
            jb = kl < k1 ? first(kl) : 0;
        }
    };
#pragma unroll
    for (int p = 0; p < kAhead; ++p) fill(p);
    begin(k);
    int j = first(k);
    double acc = 0.0;
    for (;;) {
#pragma unroll
        for (int p = 0; p < kAhead; ++p) {
            acc = dot_bcast(acc, slot_wait(d.y + kB * j + jl, yv[p], poll), l[p]);
            if (++j > k - 2) {
                finish(k, acc);
                acc = 0.0;
                k += step;
                if (k >= k1) return;
                j = first(k);
                begin(k);
            }
            fill(p);
        }
    }
}

// c_k of the backward sweep for blocks k0, k0 - step, ... >= k1
template <typename T>
__device__ __forceinline__ void help_backward(const Band<T> &B, const TeamMem &d, TeamLds &sh, int k0, int step, int k1, Poll &poll)
{
    const int lane = B.lane, wv = B.wv, jl = kU * wv + (lane >> 2);
    double m[kU], y = 0.0;
    T piv = T(1);
    auto begin = [&](int k) {
        load_mat(d, k, kMt, wv, lane, m);
        const int j = kB * k + jl;
        y = slot_load(d.y + j);
        piv = load_if<T>(j < B.n, B.rs, (unsigned)j * ((unsigned)B.bw + 1) * (unsigned)sizeof(T));
    };
    auto finish = [&](int k, const double (&acc)[kU]) {
        const int j = kB * k + jl;
        const double z = slot_wait(d.y + j, y, poll) / (double)piv;
        const double t = (j < B.n ? z : 0.0) - sum_lanes(acc, lane);
        // the wave's 16 entries: from one per four lanes to one per lane of each 16-lane row
        if ((lane & 3) == 0) sh.vec[wv][lane >> 2] = t;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        const double part = dot_bcast(0.0, sh.vec[wv][lane & 15], m);
        lds_barrier();  // the last block's partial sums are read
        sh.part[wv][lane] = part;
        lds_barrier();
        if (wv == 0)
            slot_store(d.cb + kB * k + lane, (sh.part[0][lane] + sh.part[1][lane]) + (sh.part[2][lane] + sh.part[3][lane]));
    };
    double acc[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) acc[u] = 0.0;
    int k = k0;
    for (; k >= k1 && (k + 2 >= B.nblk || B.bw <= kB); k -= step) {
        begin(k);
        finish(k, acc);
    }
    if (k < k1) return;
    auto last = [&](int q) { return min(B.nblk - 1, (kB * q + kB - 1 + B.bw) / kB); };
    T l[kAhead][kU];
    double xv[kAhead];
    int kl = k, il = last(k);
    auto fill = [&](int p) {
        const bool on = kl >= k1;
        load_cols<T>(B, on ? il : 0, on ? kl : 0, on, l[p]);
        xv[p] = slot_load(d.xo + (on ? kB * il : 0) + lane);
        if (on && --il < kl + 2) {
            kl -= step;
            il = kl >= k1 ? last(kl) : 0;
        }
    };
#pragma unroll
    for (int p = 0; p < kAhead; ++p) fill(p);
    begin(k);
    int i = last(k);
    for (;;) {
#pragma unroll
        for (int p = 0; p < kAhead; ++p) {
            const double x = slot_wait(d.xo + kB * i + lane, xv[p], poll);
#pragma unroll
            for (int u = 0; u < kU; ++u) acc[u] += (double)l[p][u] * x;
            if (--i < k + 2) {
                finish(k, acc);
#pragma unroll
                for (int u = 0; u < kU; ++u) acc[u] = 0.0;
                k -= step;
                if (k < k1) return;
                i = last(k);
                begin(k);
            }
            fill(p);
        }
    }
}

// The chain of one sweep: v_k = c_k - W_k v_prev with W = Q (forward, v = y) or P (backward, v = x).
template <typename T, bool kFwd, bool kAlone>
__device__ __forceinline__ void lead(const Band<T> &B, const TeamMem &d, TeamLds &sh, Poll &poll)
{
    const int lane = B.lane, wv = B.wv, jl = kU * wv + (lane & 15);
    cgdouble *cs = kFwd ? d.cf : d.cb;
    gdouble *vs = kFwd ? d.y : d.xo;
    struct Regs {
        double w[kU], c;
    } r[kLead];
    auto block = [&](int s) { return kFwd ? s : B.nblk - 1 - s; };
    auto load = [&](Regs &q, int s) {
        const int k = block(min(s, B.nblk - 1));
        q.c = slot_load(cs + kB * k + jl);
        load_mat(d, k, kFwd ? kMq : kMp, wv, lane, q.w);
    };
    double v = 0.0;  // solution of the block before, entry 16 wv + lane % 16
    auto step = [&](Regs &q, int s) {
        const int k = block(s), buf = lead_buffer(lead_step(kFwd, B.nblk, s));
        const double c = q.c;
        sh.lead[buf][wv][lane] = dot_bcast(0.0, v, q.w);
        if constexpr (kAlone) {
            if (kFwd)
                help_forward<T>(B, d, sh, k, 1, k + 1, poll);
            else
                help_backward<T>(B, d, sh, k, 1, k, poll);
        }
        lds_barrier();
        const double sum = sum_groups(sh.lead[buf][lane >> 4][jl]);
        v = slot_wait(cs + kB * k + jl, c, poll) - sum;
        if (lane < kU) {
            slot_store(vs + kB * k + jl, v);
            if (!kFwd && kB * k + jl < B.n) d.x[kB * k + jl] = v;
        }
        load(q, s + kLead);
    };
#pragma unroll
    for (int p = 0; p < kLead; ++p) load(r[p], p);
    // (the loops below leave by return from the middle: a skip to the loop's end would be a path on which
    // the loads in flight are others, and the compiler would wait for all of them)
    for (int s = 0;; s += kLead) {
#pragma unroll
        for (int p = 0; p < kLead; ++p) {
            if (s + p >= B.nblk) return;
            step(r[p], s + p);
        }
    }
}

// A team of up to `size` workgroups: every eighth one of the grid (workgroups go to the XCDs round robin, so
// they share one), the others leave
template <typename T>
__global__ __launch_bounds__(64 * kTW) void k_team_solve(TeamDesc desc, int size, unsigned polls)
{
    __shared__ TeamLds sh;
    if (blockIdx.x % 8 != 0) return;
    // (as values of this kernel; as its arguments the compiler places the helpers' loads worse: 1.5% of a solve)
    desc.fac = uniform_ptr(desc.fac);
    desc.x = uniform_ptr(desc.x);
    desc.b = uniform_ptr(desc.b);
    desc.mat = uniform_ptr(desc.mat);
    if (threadIdx.x == 0) {
        gu32 *ctl = (gu32 *)desc.ctl;
        const unsigned rank = __hip_atomic_fetch_add(&ctl[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned team = 0, it = 0;
        if (rank == 0) {
            do {
                team = __hip_atomic_load(&ctl[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } while (team < (unsigned)size && ++it < kFormLimit);
            __hip_atomic_store(&ctl[1], team, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            while (!(team = __hip_atomic_load(&ctl[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) && ++it < polls) {}
        }
        sh.team = team;
        sh.rank = rank;
        sh.nan = 0;
    }
    __syncthreads();
    const int team = __builtin_amdgcn_readfirstlane((int)sh.team), rank = __builtin_amdgcn_readfirstlane((int)sh.rank);
    if (rank >= team) return;
    Band<T> B;
    B.n = desc.n;
    B.bw = desc.bw;
    B.nblk = (desc.n + kB - 1) / kB;
    B.lane = threadIdx.x & 63;
    B.wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    B.rs = band_rsrc(desc.fac, (unsigned)((size_t)desc.n * ((unsigned)desc.bw + 1) * sizeof(T)));
    Poll poll{polls, false};
    if (rank > 0) {
        const TeamMem d(desc, false);
        const int h = rank - 1, H = team - 1;
        help_forward<T>(B, d, sh, h, H, B.nblk, poll);
        help_backward<T>(B, d, sh, B.nblk - 1 - h, H, 0, poll);
        return;
    }
    if (team > 1) {
        const TeamMem d(desc, false);
        lead<T, true, false>(B, d, sh, poll);
        lead<T, false, false>(B, d, sh, poll);
        // the chain's last block, read back: kept from the loop, it costs the steps 4% (other waits there)
        Poll own{kPollLimit, false};
        cgdouble *last = d.xo + kU * B.wv + (B.lane & 15);
        const double v = slot_wait(last, slot_load(last), own);
        if (__any(v != v)) __hip_atomic_store(&sh.nan, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane((int)sh.nan) == 0) return;
    }
    const TeamMem d(desc, true);
    Poll own{kPollLimit, false};
    lead<T, true, true>(B, d, sh, own);
    lead<T, false, true>(B, d, sh, own);
}

}  // namespace

// workspace: counters, right-hand side and slot vectors, the blocks' matrices
size_t team_solve_bytes(int n) { return 256 + pad_rows(n) * (1 + kSlotVecs + 4 * kB) * sizeof(double); }

// Workgroups per team: the leader, two helpers, and one more per 28 KB of what a block's c_k reads.  Measured
// (cycles a block, forward): half-width 326 in FP64 10,007 with one helper, 2,772 with 5, 2,340 with 7 and
// 2,285 with 19; half-width 1166 in FP64 3,515 with 15, 3,228 with 19; half-width 240 in FP32 2,491 with
// 3, 2,205 with 5: past these the round trip through memory from a solution block to the c_k two blocks
// on bounds the step (about 4,600 cycles for two blocks).  KSH_TEAM=k forces teams of k.
static int team_size(int n, int bw, int prec)
{
    if (const char *e = std::getenv("KSH_TEAM"))
        if (const int v = std::atoi(e); v > 0) return std::min(v, 32);
    const int far = std::max(0, std::min(bw, n) - kB);
    const double bytes = (double)far * kB * (prec == KSH_FP64 ? 8.0 : 4.0) + 8.0 * kB * kB;
    return 3 + std::min(18, (int)(bytes / 28672.0));
}

// KSH_TEAM_POLLS=k: waits of at most k polls (any k gives the same bits)
static unsigned poll_limit()
{
    const char *e = std::getenv("KSH_TEAM_POLLS");
    return e && *e ? (unsigned)std::max(0, std::atoi(e)) : kPollLimit;
}

// The team is for calls with one band, whose time is the chain's: a block and sweep takes about 1 us
// against 5 us in the one-workgroup kernel (roof 32 x 32: 562 -> 120 us a solve, of which 11 us form the
// matrices) and 7 us in the stepped one (128 x 128 plate: 11.2 -> 2.3 ms).  Up to two blocks the
// one-workgroup kernel is as fast.  With all the chip's CUs on bands of their own (batches), that kernel's
// traffic, the band alone, is the lower one.
bool team_solve_takes(int n, int bw, int prec)
{
    const size_t es = prec == KSH_FP64 ? sizeof(double) : sizeof(float);
    return n > 2 * kB && (size_t)n * (size_t)(bw + 1) * es < 0x7F000000ull;
}

int team_solve(hipStream_t s, const void *fac, int n, int bw, double *x, int prec, void *work)
{
    TeamDesc d;
    d.fac = fac;
    d.x = x;
    d.n = n;
    d.bw = bw;
    d.ctl = (unsigned *)work;
    d.b = (double *)((unsigned char *)work + 256);
    d.mat = d.b + pad_rows(n) * (1 + kSlotVecs);
    const int size = team_size(n, bw, prec);
    const unsigned polls = poll_limit();
    const dim3 gp((unsigned)(pad_rows(n) / kB)), gs((unsigned)(8 * size));
    if (prec == KSH_FP64) {
        hipLaunchKernelGGL(k_team_prep<double>, gp, dim3(256), 0, s, d);
        hipLaunchKernelGGL(k_team_solve<double>, gs, dim3(64 * kTW), 0, s, d, size, polls);
    } else {
        hipLaunchKernelGGL(k_team_prep<float>, gp, dim3(256), 0, s, d);
        hipLaunchKernelGGL(k_team_solve<float>, gs, dim3(64 * kTW), 0, s, d, size, polls);
    }
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

}  // namespace ksh
