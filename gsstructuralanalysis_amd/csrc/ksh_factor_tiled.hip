// ksh_factor_tiled.hip -- banded LDL^T factorization of a batch of bands spread over the whole
// GPU: every panel step is a pair of launches covering all bands still being factored, so a
// single large band (the 128 x 128 plate: n 49k, bw 1166) and a batch of uneven ones (the
// imperfection sweep: bw 182..470) both keep all CUs busy, and no panel has to fit LDS.
//
// Replaces SimplicialLDLT::compute on the arc-length, Newton and eigen paths
// (src/gsALMSolvers/gsALMBase.hpp:186-211, src/gsStaticSolvers/gsStaticNewton.hpp:215-240,
// src/gsEigenSolvers/gsBucklingSolver.h:131-133).  No pivoting, as there; by Sylvester's law of
// inertia the number of negative pivots does not depend on the ordering, so the band ordering
// reproduces the count gsALMBase::_computeStability takes (src/gsALMSolvers/gsALMHelper.h:30-42).
//
// Layout: lower band, column major, fac[j*ld + (i-j)], ld = bw+1, factored in place into unit L
// and D.  Right-looking in panels of NB = 64 columns.  Panel step at c0:
//   1. rows (k_band_rows, one wave per one or two 16-row tiles): L = A L_dd^-T D^-1 against the factored
//      64 x 64 diagonal block, on MFMA, spread over as many workgroups as the band has rows for;
//   2. trailing update (k_band_trailing): the lower triangle of the bw x bw trailing window is cut into
//      32 x 32 blocks, one wave each, 2 x 2 MFMA tiles (v_mfma_f64_16x16x4f64 /
//      v_mfma_f32_16x16x4f32) over the NB panel columns; panel operands -d_k L[j][k] and L[i][k]
//      come from L2, the block is read, updated and written once.  The launch's first workgroups
//      (one per band, four waves) update and factor the next diagonal block, 16 columns at a time.
// The chain from one diagonal block to the next (rows of the next 64 columns, update, 64 pivots) is what
// bounds a single band and small batches; the panel of one workgroup per band that these kernels
// replace (diagonal blocks of 32 by v_readlane, rows by substitution) took 38 us a step in FP64 at
// bw 326 and 107 us at bw 1166, against 16 + 6 us in two launches and 14 us in one (fused schedule), most
// of it the diagonal block's 12 us: factors of a 32 x 32 roof 2.5 -> 1.3 -> 0.8 ms, of the 128 x 128 plate
// 89 -> 17 -> 11.8 ms.
// Plain schedule: rows, then every block, per step.  Lookahead schedule: the blocks of the next panel's
// columns first (k_band_trailing), then k_band_step, whose first workgroups solve the next panel's
// rows while the others apply the remaining blocks.  Fused schedule: one launch a step, whose workgroups
// solve the rows they need themselves (k_band_fused).
// Bands are sorted by order, largest first, so a step's grids cover exactly the bands that are
// still active.  Work per band: about n bw^2 multiply-adds; HBM traffic about 2 n bw^2 / NB
// entries (the trailing window of a step, read and written).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "ksh_devutil.hpp"
#include "ksh_elim_steps.hpp"
#include "ksh_factor_order.hpp"
#include "ksh_internal.hpp"
#include "ksh_mfma.hpp"
#include "ksh_profile.hpp"
#include "ksh_tune.hpp"

namespace ksh {

namespace {

constexpr int kQ = 16;        // tile edge
constexpr int kNB = 64;       // panel width (rank of one trailing update)
constexpr int kPT = 512;      // lookahead step kernel threads
constexpr int kUW = 4;        // waves per trailing-update / row-solve workgroup; the diagonal block's strips

// ---- tiles ------------------------------------------------------------------------------------
// A 16 x 16 tile of rows R and columns K of the band lives in a wave "transposed": lane l, register
// v hold A[R + l % 16][K + krow(l, v)], krow = Mfma16<C>::row.  In this form a product of MFMAs is at
// once the next one's operand: with the k index of step s taken as krow(l, s) on both sides (the sum
// over k is in another order, nothing else), the result registers of D = A B are the B operand of the
// next product, and the same registers of another tile (L[j][k], lane = j) are an A operand.  No
// lane exchange sits between dependent products.

// -1 / d from the hardware estimate r and Newton steps (rounding of the last place; the quotient's full
// division sequence is about twice as long and sits on the chain of the 64 pivots)
__device__ __forceinline__ double neg_recip(double d, double r)
{
    r = __builtin_fma(__builtin_fma(d, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(d, r, 1.0), r, r);
}
__device__ __forceinline__ float neg_recip(float d, float r) { return __builtin_fmaf(__builtin_fmaf(d, r, 1.0f), r, r); }
__device__ __forceinline__ double rcp_estimate(double d) { return __builtin_amdgcn_rcp(d); }
__device__ __forceinline__ float rcp_estimate(float d) { return __builtin_amdgcn_rcpf(d); }

// Elimination of a 16 x 16 block from step J on, lane = row r: e[k] = A[r][k], w[q] = columns krow(l, q)
// of the unit matrix, nr = -1 / d_J.  Afterwards e[k] = L[r][k] d_k for k < r and d_r for k = r, w holds
// the inverse of the unit lower factor, and dsel[v] = 1 / d_k of k = krow(l, v).  A step is a
// reciprocal, a multiply and 19 - J multiply-adds.  Rows up to J take the update of e too (their entries
// right of the diagonal are not read again), but not that of w.
template <int J, typename C>
__device__ __forceinline__ void eliminate(C (&e)[kQ], C (&w)[4], C (&dsel)[4], int r, int lk, C nr)
{
    constexpr int v = sizeof(C) == 8 ? J / 4 : J % 4, grp = sizeof(C) == 8 ? J % 4 : J / 4;  // krow(l, v) = J
    if constexpr (J + 1 < kQ) {
        const C m = e[J] * nr;
        const C mw = r > J ? m : C(0);
        C est;
        const C d = elim_step<J>(e, w, m, mw, est);
        const C next = neg_recip(d, est);
        dsel[v] = lk == grp ? -nr : dsel[v];
        eliminate<J + 1, C>(e, w, dsel, r, lk, next);
    } else {
        dsel[v] = lk == grp ? -nr : dsel[v];
    }
}

// What the row solves of a panel need beside its factored block, per band: the operands of the four
// 16 x 16 inverses (step s of sub-block c at [(4 c + s) * 64 + lane]), then 1 / d of the 64 columns.
constexpr int kWorkInv = 4 * 4 * 64;
constexpr size_t kWorkSlot = (kWorkInv + kNB) * sizeof(double);
template <typename C>
__device__ __forceinline__ C *panel_work(void *work, int band, int c0)
{
    return (C *)((unsigned char *)work + (size_t)band * kBandWorkBytes + (size_t)panel_slot(c0) * kWorkSlot);
}
static_assert(kPanelSlots * kWorkSlot <= kBandWorkBytes && kNB == 64, "factor workspace");

// Row tiles of the panel at c0 (tile t: rows c0 + 64 + 16 t .. + 15, its 64 columns) against the factored
// diagonal block, one wave: X = A L^-T by blocks of 16 columns (substitution between them, the 16 x 16
// inverse within), L = X D^-1.  40 MFMAs in one chain; the operands of the diagonal block are read
// from L2 by every wave, which spreads a band's rows over as many CUs as there are.  Tiles t0, t0 +
// stride, ...: out(t, column, value) takes lane li's entry of row li of the tile.  Rows past the panel
// are zero.
template <typename T, typename C, typename F>
__device__ __forceinline__ void solve_tiles(const BandDesc &d, int c0, int t0, int stride, int ntile, const C *work, F &&out)
{
    using M = Mfma16<C>;
    using acc_t = typename M::acc_t;
    const int n = d.n, bw = d.bw;
    const int nr = min(n - c0, kNB + bw);  // panel rows (relative to c0); the panel is full: n > c0 + 64
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(d.fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x & 63, li = lane & 15;
    C inv[4][4], dinv[4][4], l[4][4][4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            inv[c][s] = work[(4 * c + s) * 64 + lane];
            dinv[c][s] = work[kWorkInv + kQ * c + M::row(lane, s)];
#pragma unroll
            for (int e = 0; e < c; ++e) {  // L[16 c + li][16 e + krow]
                const int row = kQ * c + li, col = kQ * e + M::row(lane, s);
                l[c][e][s] = -(C)load_if<T>(row - col <= bw, rs, ((unsigned)(c0 + col) * ldu + (unsigned)(row - col)) * es);
            }
        }
    for (int q = 0; q < ntile; ++q) {
        const int t = t0 + q * stride, r = kNB + kQ * t + li;
        acc_t a[4], x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int col = kQ * c + M::row(lane, v);
                a[c][v] = (C)load_if<T>(r < nr && r - col <= bw, rs, ((unsigned)(c0 + col) * ldu + (unsigned)(r - col)) * es);
            }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int e = 0; e < c; ++e)
#pragma unroll
                for (int s = 0; s < 4; ++s) a[c] = M::run(l[c][e][s], x[e][s], a[c]);
            const acc_t zero = {C(0), C(0), C(0), C(0)};
            x[c] = zero;
#pragma unroll
            for (int s = 0; s < 4; ++s) x[c] = M::run(inv[c][s], a[c][s], x[c]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) out(t, kQ * c + M::row(lane, v), (T)(x[c][v] * dinv[c][v]));
    }
}

// tiles t0 .. t0 + ntile - 1 of the panel at c0, back to the band
template <typename T, typename C>
__device__ __forceinline__ void solve_rows(const BandDesc &d, int c0, int t0, int ntile, const C *work)
{
    const int n = d.n, bw = d.bw, nr = min(n - c0, kNB + bw);
    if (n <= c0 + kNB || kNB + kQ * t0 >= nr) return;
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(d.fac, (unsigned)((size_t)n * ldu * es));
    const int li = threadIdx.x & 15;
    const int left = (nr - kNB - kQ * t0 + kQ - 1) / kQ;
    solve_tiles<T, C>(d, c0, t0, 1, min(ntile, left), work, [&](int t, int col, T v) {
        const int r = kNB + kQ * t + li;
        store_if<T>(r < nr && r - col <= bw, rs, ((unsigned)(c0 + col) * ldu + (unsigned)(r - col)) * es, v);
    });
}

// place of entry (row, k) of a 64 x 64 operand block in LDS: the 16 rows and 4 columns an MFMA operand
// reads at once fall into different banks
__device__ __forceinline__ int panel_at(int k, int row) { return k * kNB + (row ^ ((k & 3) << 4)); }

// Diagonal block of the panel at c0 (64 columns, unit pivots past n): four waves, wave w owning the
// 16-row strip w (tiles (w, 0..w)).  With kUpdate, the block first takes the rank-64 update of the
// panel at c0 - 64, whose 64 x 64 operand block goes through LDS (one memory latency for the whole
// block); with kSolve its rows there are still unsolved, and the workgroup solves these 64 first (`prev`:
// that panel's workspace).  Then for c = 0..3: wave c factors tile (c, c) by rows; the strips below solve their tile
// (i, c) against it (one product with the 16 x 16 inverse) and update their remaining tiles.  The
// inverses are of 16 x 16 unit lower blocks only: between sub-blocks the solve is a substitution.
// Bound by its chain: 64 pivots of about 100 cycles each (reciprocal and broadcasts), four LDS round
// trips and product chains between the sub-blocks.
template <typename C>
struct DiagLds {
    C panel[kNB * kNB];   // L[c0 + row][c0 - 64 + k] at panel_at(k, row)
    C nd[kNB];            // -d of the previous panel
    C tr[kQ * (kQ + 1)];  // a diagonal tile on its way to lane = row
    C inv[4 * 64];        // sub-block c: operands of the inverse
    C dinv[4 * 64];       // and 1 / d, by (register, lane)
    C dk[kNB];            // 1 / d of the block
    C l[4][4 * 64];       // the strips' L[i][c]: operands of the other strips' updates
    int bad;
};

enum DiagMode { kFirst, kUpdate, kSolve };
template <typename T, typename C, int kMode>
__device__ __forceinline__ void diag_panel(const BandDesc &d, int c0, C *work, const C *prev, DiagLds<C> &sh)
{
    using M = Mfma16<C>;
    using acc_t = typename M::acc_t;
    const int n = d.n, bw = d.bw;
    if (c0 >= n) return;
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(d.fac, (unsigned)((size_t)n * ldu * es));
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int w = min(kNB, n - c0);
    if (tid == 0) sh.bad = 0;
    const int i = kQ * wv + li;  // this lane's row
    constexpr int kP = kNB * kNB / (64 * kUW);
    T pv[kP], dv = T(0);
    const int cp = c0 - kNB;
    if constexpr (kMode != kFirst) dv = load_if<T>(tid < kNB, rs, (unsigned)(cp + lane) * ldu * es);
    if constexpr (kMode == kUpdate) {  // panel operands: lanes along a column's rows
#pragma unroll
        for (int q = 0; q < kP; ++q) {
            const int k = kUW * q + wv;
            pv[q] = load_if<T>(lane < w && lane + kNB - k <= bw, rs, ((unsigned)(cp + k) * ldu + (unsigned)(lane + kNB - k)) * es);
        }
    }
    acc_t acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j > wv) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int col = kQ * j + M::row(lane, v);
            const int hi = max(i, col), lo = min(i, col);  // the upper half of a diagonal tile mirrors the lower
            const bool ok = hi < w && hi - lo <= bw;
            const C x = (C)load_if<T>(ok, rs, ((unsigned)(c0 + lo) * ldu + (unsigned)(hi - lo)) * es);
            acc[j][v] = (hi >= w && hi == lo) ? C(1) : x;
        }
    }
    if constexpr (kMode != kFirst) {
        if constexpr (kMode == kUpdate) {
#pragma unroll
            for (int q = 0; q < kP; ++q) sh.panel[panel_at(kUW * q + wv, lane)] = (C)pv[q];
        } else {
            solve_tiles<T, C>(d, cp, wv, 1, 1, prev, [&](int t, int k, T v) { sh.panel[panel_at(k, kQ * t + li)] = (C)v; });
        }
        if (tid < kNB) sh.nd[tid] = -(C)dv;
        lds_barrier();
        C own[kNB / 4], nd[kNB / 4];
#pragma unroll
        for (int s = 0; s < kNB / 4; ++s) {
            nd[s] = sh.nd[4 * s + lk];
            own[s] = sh.panel[panel_at(4 * s + lk, i)];
        }
        // wave 0 has the least of it and goes on to its diagonal tile while the others finish
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j > wv) continue;
#pragma unroll
            for (int s = 0; s < kNB / 4; ++s)
                acc[j] = M::run(nd[s] * sh.panel[panel_at(4 * s + lk, kQ * j + li)], own[s], acc[j]);
        }
    }
    C lkeep[4] = {C(0), C(0), C(0), C(0)};
    auto store_l = [&](int c, const C (&l)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int col = kQ * c + M::row(lane, v);
            store_if<T>(i < w && i - col <= bw, rs, ((unsigned)(c0 + col) * ldu + (unsigned)(i - col)) * es, (T)l[v]);
        }
    };
    // acc[0] is the strip's tile in column c, acc[j] the one in column c + j: shifted down after every
    // sub-block, so that the loop stays rolled (its code is fetched once, not four times)
#pragma unroll 1
    for (int c = 0; c < 4; ++c) {
        C e[kQ], inv[4], dinv[4];
        if (wv == c) {
#pragma unroll
            for (int v = 0; v < 4; ++v) sh.tr[M::row(lane, v) * (kQ + 1) + li] = acc[0][v];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
            for (int k = 0; k < kQ; ++k) e[k] = sh.tr[k * (kQ + 1) + li];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                inv[q] = M::row(lane, q) == li ? C(1) : C(0);
                dinv[q] = C(0);
            }
            const C d0 = row_bcast<0>(e[0]);
            eliminate<0, C>(e, inv, dinv, li, lk, neg_recip(d0, rcp_estimate(-d0)));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                sh.inv[q * 64 + lane] = inv[q];
                sh.dinv[q * 64 + lane] = dinv[q];
                if (li == 0) sh.dk[kQ * c + M::row(lane, q)] = dinv[q];
            }
        }
        lds_barrier();
        acc_t x = {C(0), C(0), C(0), C(0)};
        C lv[4];
        if (wv > c) {
#pragma unroll
            for (int s = 0; s < 4; ++s) x = M::run(sh.inv[s * 64 + lane], acc[0][s], x);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                lv[v] = x[v] * sh.dinv[v * 64 + lane];
                sh.l[wv][v * 64 + lane] = lv[v];
            }
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (c + j == wv) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[j] = M::run(-lv[s], x[s], acc[j]);
                }
        }
        lds_barrier();
        if (wv > c) {
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (c + j < wv) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[j] = M::run(-sh.l[c + j][s * 64 + lane], x[s], acc[j]);
                }
#pragma unroll
            for (int j = 0; j < 3; ++j) acc[j] = acc[j + 1];
            if (wv > c + 1) {
                store_l(c, lv);
            } else {  // its own sub-block is next: the stores follow it
#pragma unroll
                for (int v = 0; v < 4; ++v) lkeep[v] = lv[v];
            }
        } else if (wv == c) {
            if (c > 0) store_l(c - 1, lkeep);
            // off the chain: the factored tile and the row solves' operands to memory, the pivots' check; lane
            // (li, lk) stores columns 4 lk .. 4 lk + 3 of its row
            C sel[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const C lo = lk == 0 ? e[q] : e[4 + q], hi = lk == 2 ? e[8 + q] : e[12 + q];
                sel[q] = lk < 2 ? lo : hi;
            }
            const int k0 = 4 * lk;
            unsigned off = ((unsigned)(c0 + kQ * c + k0) * ldu + (unsigned)(li - k0)) * es;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = k0 + q;
                const C val = k == li ? sel[q] : sel[q] * sh.dk[kQ * c + k];
                store_if<T>(k <= li && i < w && li - k <= bw, rs, off, (T)val);
                off += (ldu - 1) * es;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) work[(4 * c + q) * 64 + lane] = inv[q];
            if (lane < kQ) work[kWorkInv + kQ * c + lane] = sh.dk[kQ * c + lane];
            const C d01 = (li & 1) ? sel[1] : sel[0], d23 = (li & 1) ? sel[3] : sel[2];
            const C dr = (li & 2) ? d23 : d01;  // the pivot of row li, in the lanes lk = li / 4
            const bool bad = lk == (li >> 2) && i < w && (dr == C(0) || !isfinite(dr) || !isfinite((double)(T)dr));
            const unsigned long long bm = __ballot(bad);
            // (these lanes are in the order of their rows)
            if (lane == 0 && bm != 0 && sh.bad == 0) sh.bad = c0 + kQ * c + ((__ffsll((long long)bm) - 1) & (kQ - 1)) + 1;
        }
    }
    lds_barrier();  // sh.bad of every sub-block
    if (tid == 0 && d.info) {
        if (c0 == 0)
            *d.info = sh.bad;
        else if (sh.bad != 0 && *d.info == 0)
            *d.info = sh.bad;
    }
}

// Blocks p[0] < p[1] < ... of the given part (wave-uniform), computed together (independent
// accumulators, the loads of all of them in flight at once): A[i][j] -= sum_k L[i][k] d_k L[j][k]
// over the window rows/columns [w, nr) of the frame at c0.  Indices past the part's block count
// are computed on block p[0]'s operands with their stores masked off.  Each block's MFMA sequence
// (k ascending) is the same for every NBLK, so the result does not depend on it.
template <typename T, int NBLK>
__device__ __forceinline__ void trailing_blocks(const BandDesc &d, int c0, int part, const int (&p)[NBLK])
{
    using M = Mfma16<T>;
    using acc_t = typename M::acc_t;
    const int n = d.n, bw = d.bw;
    if (c0 >= n) return;
    const int w = min(kNB, n - c0), nr = min(n - c0, w + bw);
    const int nbk = (nr - w + 31) / 32;
    const int nblock = trail_blocks(nbk, part);
    if (p[0] >= nblock) return;
    T *fac = (T *)d.fac;
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(fac, (unsigned)((size_t)n * ldu * es));
    const int lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    bool valid[NBLK], diag[NBLK];
    int ri0[NBLK], rj0[NBLK];
    // accumulator rows = j (A's column), columns = i (A's row): lanes run along a column
    acc_t cur[NBLK][2][2];
    unsigned off[NBLK][2][2][4];
#pragma unroll
    for (int s = 0; s < NBLK; ++s) {
        valid[s] = p[s] < nblock;
        const int q = valid[s] ? p[s] : p[0];
        int bi, bj;
        trail_decode(q, nbk, part, bi, bj);
        diag[s] = bi == bj;
        ri0[s] = w + 32 * bi + li;
        rj0[s] = w + 32 * bj + li;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = w + 32 * bi + 16 * a + li, j = w + 32 * bj + 16 * b + M::row(lane, v);
                    const bool ok = valid[s] && i < nr && i >= j;
                    off[s][a][b][v] = ok ? ((unsigned)c0 * ldu + (unsigned)j * (ldu - 1) + (unsigned)i) * es : kMaskedOff;
                    cur[s][a][b][v] = load_vs<T>(rs, off[s][a][b][v], 0);
                }
    }
    // panel operands: rows rj (block column bj) and ri (block row bi), k = 4 s + lk, in chunks
    constexpr int kCh = 8 / NBLK;
#pragma unroll
    for (int c = 0; c < kNB / 4 / kCh; ++c) {
        T A0[NBLK][kCh], A1[NBLK][kCh], B0[NBLK][kCh], B1[NBLK][kCh];
#pragma unroll
        for (int u = 0; u < kCh; ++u) {
            const int k = 4 * (kCh * c + u) + lk;
            const unsigned col = ((unsigned)c0 * ldu + (unsigned)k * (ldu - 1)) * es;  // + row * es
            const T nd = -load_if<T>(k < w, rs, (unsigned)(c0 + k) * ldu * es);
#pragma unroll
            for (int s = 0; s < NBLK; ++s) {
                const int rj = rj0[s], ri = ri0[s];
                A0[s][u] = nd * load_if<T>(k < w && rj < nr && rj - k <= bw, rs, col + (unsigned)rj * es);
                A1[s][u] = nd * load_if<T>(k < w && rj + 16 < nr && rj + 16 - k <= bw, rs, col + (unsigned)(rj + 16) * es);
                B0[s][u] = load_if<T>(k < w && ri < nr && ri - k <= bw, rs, col + (unsigned)ri * es);
                B1[s][u] = load_if<T>(k < w && ri + 16 < nr && ri + 16 - k <= bw, rs, col + (unsigned)(ri + 16) * es);
            }
        }
#pragma unroll
        for (int u = 0; u < kCh; ++u)
#pragma unroll
            for (int s = 0; s < NBLK; ++s) {
                cur[s][0][0] = M::run(A0[s][u], B0[s][u], cur[s][0][0]);
                cur[s][1][0] = M::run(A0[s][u], B1[s][u], cur[s][1][0]);
                cur[s][1][1] = M::run(A1[s][u], B1[s][u], cur[s][1][1]);
                if (!diag[s]) cur[s][0][1] = M::run(A1[s][u], B0[s][u], cur[s][0][1]);
            }
    }
#pragma unroll
    for (int s = 0; s < NBLK; ++s)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) store_vs<T>(rs, off[s][a][b][v], 0, cur[s][a][b][v]);
}

// Descriptor of a workgroup's band in scalar registers.  The compiler takes a descriptor read behind a
// division or a store for possibly divergent, and would then turn every buffer access through it into a loop
// over the lanes' (equal) descriptors.
__device__ __forceinline__ BandDesc uniform_desc(const BandDesc *descs, int band)
{
    const BandDesc &s = descs[__builtin_amdgcn_readfirstlane(band)];
    BandDesc d;
    d.fac = uniform_ptr(s.fac);
    d.n = __builtin_amdgcn_readfirstlane(s.n);
    d.bw = __builtin_amdgcn_readfirstlane(s.bw);
    d.info = uniform_ptr(s.info);
    d.stats = nullptr;
    d.x = nullptr;
    d.active = 1;
    return d;
}

// Diagonal block at column 0 of every band (the later ones are factored by the trailing launches).
template <typename T, typename C>
__global__ __launch_bounds__(64 * kUW) void k_band_diag(const BandDesc *descs, void *work)
{
    __shared__ DiagLds<C> sh;
    const BandDesc d = uniform_desc(descs, (int)blockIdx.x);
    diag_panel<T, C, kFirst>(d, 0, panel_work<C>(work, (int)blockIdx.x, 0), nullptr, sh);
}

// a launch's workgroup h as (band, index within the band); false for a padding one
__device__ __forceinline__ bool band_of_workgroup(int h, int active, int wg, int &band, int &local)
{
    workgroup_decode(h, active, wg, band, local);
    // the divisions run on the vector unit: back to scalars
    band = __builtin_amdgcn_readfirstlane(band);
    local = __builtin_amdgcn_readfirstlane(local);
    return band < active;
}
// Rows of the panel at c0, kUW waves per workgroup and `tiles` 16-row tiles per wave
template <typename T, typename C>
__global__ __launch_bounds__(64 * kUW) void k_band_rows(const BandDesc *descs, void *work, int c0, int wg_per_band, int tiles,
                                                        int active)
{
    int band, local;
    if (!band_of_workgroup((int)blockIdx.x, active, wg_per_band, band, local)) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const BandDesc d = uniform_desc(descs, band);
    solve_rows<T, C>(d, c0, (local * kUW + wave) * tiles, tiles, panel_work<C>(work, band, c0));
}

// One part of the trailing update at c0, kUW blocks (one per wave) per workgroup; workgroups
// [0, ndiag) update and factor the next diagonal block of their band.  They hold the step's longest
// chain, so they are dispatched first.  (The update part starts at workgroup `pad`, ndiag rounded up to
// a multiple of the XCD count, so that its XCD-aware mapping lines up with the first part's.)
template <typename T, typename C>
__global__ __launch_bounds__(64 * kUW) void k_band_trailing(const BandDesc *descs, void *work, int c0, int ndiag, int pad,
                                                            int wg_per_band, int part, int active)
{
    const int b = (int)blockIdx.x;
    if (b < ndiag) {
        __shared__ DiagLds<C> sh;
        const BandDesc d = uniform_desc(descs, b);
        diag_panel<T, C, kUpdate>(d, c0 + kNB, panel_work<C>(work, b, c0 + kNB), nullptr, sh);
        return;
    }
    if (b < pad) return;
    int band, local;
    if (!band_of_workgroup(b - pad, active, wg_per_band, band, local)) return;
    const int p[1] = {__builtin_amdgcn_readfirstlane((int)(local * kUW + (threadIdx.x >> 6)))};
    const BandDesc d = uniform_desc(descs, band);
    trailing_blocks<T, 1>(d, c0, part, p);
}

// Lookahead step: the first workgroups (nrow per band, padded to `pad`) solve the rows of the panel at
// c0 + NB while the others apply the rest of the trailing update at c0 (block columns 2 and up), NBLK
// blocks per wave.  The two parts touch disjoint columns: the rows read and write columns
// [c0 + NB, c0 + 2 NB), already updated by the kNext part; the rest of the update reads the panel at
// c0 and writes columns from c0 + 2 NB on.
template <typename T, typename C, int NBLK>
__global__ __launch_bounds__(kPT) void k_band_step(const BandDesc *descs, void *work, int c0, int nrow, int tiles, int np, int pad,
                                                   int wg_per_band, int active)
{
    const int b = (int)blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    constexpr int kW = kPT / 64;
    int band, local;
    if (b < pad) {
        if (!band_of_workgroup(b, np, nrow, band, local)) return;
        const BandDesc d = uniform_desc(descs, band);
        solve_rows<T, C>(d, c0 + kNB, (local * kW + wave) * tiles, tiles, panel_work<C>(work, band, c0 + kNB));
        return;
    }
    if (!band_of_workgroup(b - pad, active, wg_per_band, band, local)) return;
    int p[NBLK];
#pragma unroll
    for (int s = 0; s < NBLK; ++s) p[s] = (local * NBLK + s) * kW + wave;
    const BandDesc d = uniform_desc(descs, band);
    trailing_blocks<T, NBLK>(d, c0, kRest, p);
}

// 64 x 64 tile (I, J), J <= I, of the trailing window at c0 with the panel's rows still unsolved: the four
// waves solve the 64 rows of I and of J into LDS, then take one 32 x 32 block each of the tile's update
// (the same MFMA sequence per block as trailing_blocks).
template <typename T>
struct TileLds {
    T pi[kNB * kNB], pj[kNB * kNB];  // L[window row][k] at panel_at(k, row)
    T nd[kNB];
};
template <typename T, typename C>
__device__ __forceinline__ void fused_tile(const BandDesc &d, int c0, int I, int J, const C *work, TileLds<T> &sh)
{
    using M = Mfma16<T>;
    using acc_t = typename M::acc_t;
    const int n = d.n, bw = d.bw;
    const int nr = min(n - c0, kNB + bw);
    const unsigned ldu = (unsigned)bw + 1;
    constexpr unsigned es = sizeof(T);
    const __amdgpu_buffer_rsrc_t rs = band_rsrc(d.fac, (unsigned)((size_t)n * ldu * es));
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ri = 32 * (wv >> 1), rj = 32 * (wv & 1);  // the wave's block in the tile
    const bool mine = I != J || ri >= rj, diag = I == J && ri == rj;
    const T dv = load_if<T>(tid < kNB, rs, (unsigned)(c0 + lane) * ldu * es);
    acc_t cur[2][2];
    unsigned off[2][2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = kNB + kNB * I + ri + 16 * a + li, j = kNB + kNB * J + rj + 16 * b + M::row(lane, v);
                const bool ok = mine && i < nr && i >= j;
                off[a][b][v] = ok ? ((unsigned)c0 * ldu + (unsigned)j * (ldu - 1) + (unsigned)i) * es : kMaskedOff;
                cur[a][b][v] = load_vs<T>(rs, off[a][b][v], 0);
            }
    solve_tiles<T, C>(d, c0, 4 * I + wv, 4 * (J - I), I == J ? 1 : 2, work, [&](int t, int k, T v) {
        (t == 4 * I + wv ? sh.pi : sh.pj)[panel_at(k, kQ * wv + li)] = v;
    });
    if (tid < kNB) sh.nd[tid] = -dv;
    lds_barrier();
    if (!mine) return;
    const T *pj = I == J ? sh.pi : sh.pj;
#pragma unroll
    for (int s = 0; s < kNB / 4; ++s) {
        const int k = 4 * s + lk;
        const T nd = sh.nd[k];
        const T A0 = nd * pj[panel_at(k, rj + li)], A1 = nd * pj[panel_at(k, rj + 16 + li)];
        const T B0 = sh.pi[panel_at(k, ri + li)], B1 = sh.pi[panel_at(k, ri + 16 + li)];
        cur[0][0] = M::run(A0, B0, cur[0][0]);
        cur[1][0] = M::run(A0, B1, cur[1][0]);
        cur[1][1] = M::run(A1, B1, cur[1][1]);
        if (!diag) cur[0][1] = M::run(A1, B0, cur[0][1]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) store_vs<T>(rs, off[a][b][v], 0, cur[a][b][v]);
}

// Fused step at c0, one launch a step: workgroup 0 of a band solves the next 64 rows, updates and factors
// the next diagonal block; `ntile` workgroups apply the rest of the update, solving the rows they need
// themselves (the panel at c0 is only read, so no workgroup waits for another); the last ones write the
// solved rows of the panel before, which nothing in this launch reads.  Three times the update's
// multiply-adds and one launch on the chain instead of two: for few bands.
template <typename T, typename C>
__global__ __launch_bounds__(64 * kUW) void k_band_fused(const BandDesc *descs, void *work, int c0, int ntile, int nrow)
{
    __shared__ union {
        DiagLds<C> diag;
        TileLds<T> tile;
    } sh;
    const int per = 1 + ntile + nrow;
    const int band = __builtin_amdgcn_readfirstlane((int)blockIdx.x / per), g = (int)blockIdx.x - band * per;
    const BandDesc d = uniform_desc(descs, band);
    if (g > ntile) {
        if (c0 == 0) return;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        solve_rows<T, C>(d, c0 - kNB, (g - 1 - ntile) * kUW + wave, 1, panel_work<C>(work, band, c0 - kNB));
        return;
    }
    if (d.n <= c0 + kNB) return;
    const C *here = panel_work<C>(work, band, c0);
    if (g == 0) {
        diag_panel<T, C, kSolve>(d, c0 + kNB, panel_work<C>(work, band, c0 + kNB), here, sh.diag);
        return;
    }
    int I, J;
    tri_decode(g, I, J);  // tile 0, the next diagonal block, is workgroup 0's
    if (kNB + kNB * I >= min(d.n - c0, kNB + d.bw)) return;
    fused_tile<T, C>(d, c0, I, J, here, sh.tile);
}

// negatives, min d, max |d|, min |d| of each factored diagonal (one workgroup of 1024 threads per band)
template <typename T>
__global__ __launch_bounds__(1024) void k_pivot_stats(const BandDesc *descs)
{
    __shared__ double part[16][4];
    const BandDesc &dd = descs[blockIdx.x];
    if (!dd.stats) return;
    const T *fac = (const T *)dd.fac;
    const size_t ld = (size_t)dd.bw + 1;
    double c = 0.0, mn = INFINITY, mxa = 0.0, mna = INFINITY;
    for (int i = threadIdx.x; i < dd.n; i += 1024) {
        const double d = (double)fac[(size_t)i * ld];
        c += d < 0.0 ? 1.0 : 0.0;
        mn = fmin(mn, d);
        mxa = fmax(mxa, fabs(d));
        mna = fmin(mna, fabs(d));
    }
    for (int o = 32; o > 0; o >>= 1) {
        c += __shfl_xor(c, o);
        mn = fmin(mn, __shfl_xor(mn, o));
        mxa = fmax(mxa, __shfl_xor(mxa, o));
        mna = fmin(mna, __shfl_xor(mna, o));
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        part[wave][0] = c;
        part[wave][1] = mn;
        part[wave][2] = mxa;
        part[wave][3] = mna;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 16; ++q) {
            c += part[q][0];
            mn = fmin(mn, part[q][1]);
            mxa = fmax(mxa, part[q][2]);
            mna = fmin(mna, part[q][3]);
        }
        dd.stats[0] = c;
        dd.stats[1] = mn;
        dd.stats[2] = mxa;
        dd.stats[3] = mna;
    }
}

// Factor schedules (every one gives the same result bit for bit):
//   0 plain: per step the panel's rows, then the whole trailing update, whose first workgroups update
//   and factor the next diagonal block;
//   1 lookahead: per step the next panel's columns (kNext, with the next diagonal block), then the
//   next panel's rows together with the rest of the update (k_band_step);
//   2 fused (k_band_fused), one launch a step, for up to kFusedBands bands; for more, lookahead with two
//   blocks per wave.
// Plain has the rest of the update beside the diagonal block's chain, lookahead beside the rows, fused the
// shortest chain and the most arithmetic; which one is fastest depends on the number and shape of the
// bands, so the autotuner picks per shape bucket (KSH_LOOKAHEAD=k forces k).
// Fused up to kFusedBands bands: a band's workgroups (22 at bw 326, 192 at bw 1166) then stay around the
// chip's 256 CUs; with more, the threefold arithmetic is what bounds the step.
constexpr int kSchedules = 3;

int schedule_forced()
{
    const char *e = std::getenv("KSH_LOOKAHEAD");
    if (!e || !*e) return -1;
    const int v = std::atoi(e);
    return v >= 0 && v < kSchedules ? v : -1;
}

// bands (orders descending) with a column c
inline int active_at(const std::vector<int> &ns, int c)
{
    int a = (int)ns.size();
    while (a > 0 && ns[a - 1] <= c) --a;
    return a;
}

// 16-row tiles per wave of the row solves: one while the tiles leave the chip room (the solve is one
// chain of 40 MFMAs per tile), two when there are enough bands to fill it (the operands of the diagonal
// block, 20 KB in FP64, are then read once for two tiles of 8 KB)
inline int row_tiles(int active) { return active >= 32 ? 2 : 1; }

template <typename T, typename C, int NBLK>
void run_lookahead(hipStream_t s, const BandDesc *d_descs, void *work, const std::vector<int> &ns, int maxbw)
{
    constexpr int kW = kPT / 64;
    const int nbk = (maxbw + 31) / 32, ntile = (maxbw + kQ - 1) / kQ;
    const int wg1 = (trail_blocks(nbk, kNext) + kUW - 1) / kUW;
    const int wg2 = (trail_blocks(nbk, kRest) + kW * NBLK - 1) / (kW * NBLK);
    int np = active_at(ns, kNB);  // bands with rows below the current panel
    if (np == 0) return;
    {
        const int tiles = row_tiles(np), wg = (ntile + kUW * tiles - 1) / (kUW * tiles);
        if (wg > 0)
            hipLaunchKernelGGL((k_band_rows<T, C>), dim3(band_grid(np, wg)), dim3(64 * kUW), 0, s, d_descs, work, 0, wg, tiles, np);
    }
    for (int c0 = 0; np > 0; c0 += kNB) {
        const int pad1 = np >= kXcds ? (np + kXcds - 1) / kXcds * kXcds : np;
        hipLaunchKernelGGL((k_band_trailing<T, C>), dim3((unsigned)pad1 + (wg1 > 0 ? band_grid(np, wg1) : 0u)), dim3(64 * kUW), 0, s,
                           d_descs, work, c0, np, pad1, wg1, (int)kNext, np);
        const int np1 = active_at(ns, c0 + 2 * kNB);
        const int tiles = row_tiles(np1), nrow = (ntile + kW * tiles - 1) / (kW * tiles);
        int pad = np1 > 0 && nrow > 0 ? (int)band_grid(np1, nrow) : 0;
        if (np >= kXcds) pad = (pad + kXcds - 1) / kXcds * kXcds;
        const unsigned grid = (unsigned)pad + (wg2 > 0 ? band_grid(np, wg2) : 0u);
        if (grid > 0)
            hipLaunchKernelGGL((k_band_step<T, C, NBLK>), dim3(grid), dim3(kPT), 0, s, d_descs, work, c0, nrow, tiles, np1, pad, wg2,
                               np);
        np = np1;
    }
}

template <typename T, typename C>
void run_tiled_sched(hipStream_t s, const BandDesc *d_descs, void *work, const std::vector<int> &ns, int maxbw, int sched)
{
    // ns: orders of the bands, descending (the device array is in the same order)
    const int nbands = (int)ns.size();
    hipLaunchKernelGGL((k_band_diag<T, C>), dim3((unsigned)nbands), dim3(64 * kUW), 0, s, d_descs, work);
    if (sched == 0) {
        const int nbk = (maxbw + 31) / 32, ntile = (maxbw + kQ - 1) / kQ;
        const int wg = (trail_blocks(nbk, kAll) + kUW - 1) / kUW;
        int np;
        for (int c0 = 0; (np = active_at(ns, c0 + kNB)) > 0; c0 += kNB) {
            const int tiles = row_tiles(np), wgr = (ntile + kUW * tiles - 1) / (kUW * tiles);
            if (wgr > 0)
                hipLaunchKernelGGL((k_band_rows<T, C>), dim3(band_grid(np, wgr)), dim3(64 * kUW), 0, s, d_descs, work, c0, wgr, tiles, np);
            const int pad = np >= kXcds ? (np + kXcds - 1) / kXcds * kXcds : np;
            hipLaunchKernelGGL((k_band_trailing<T, C>), dim3((unsigned)pad + (wg > 0 ? band_grid(np, wg) : 0u)), dim3(64 * kUW), 0, s,
                               d_descs, work, c0, np, pad, wg, (int)kAll, np);
        }
    } else if (sched == 1) {
        run_lookahead<T, C, 1>(s, d_descs, work, ns, maxbw);
    } else if (nbands <= kFusedBands) {
        const int nt = (maxbw + kNB - 1) / kNB, ntile = std::max(0, nt * (nt + 1) / 2 - 1);
        const int nrow = ((maxbw + kQ - 1) / kQ + kUW - 1) / kUW;
        int c0 = 0;
        for (;; c0 += kNB) {  // the step past a band's last panel still writes that panel's rows
            const int np = active_at(ns, c0);
            if (np == 0) break;
            hipLaunchKernelGGL((k_band_fused<T, C>), dim3((unsigned)(np * (1 + ntile + nrow))), dim3(64 * kUW), 0, s, d_descs, work, c0,
                               ntile, nrow);
        }
    } else {
        run_lookahead<T, C, 2>(s, d_descs, work, ns, maxbw);
    }
    hipLaunchKernelGGL(k_pivot_stats<T>, dim3((unsigned)nbands), dim3(1024), 0, s, d_descs);
}

// Arithmetic of the panel (diagonal block and rows): the storage precision up to half-width kPanelBw; an
// FP32 factor of a wider band has its panel in FP64 (longer sums per entry).
constexpr int kPanelBw = 480;
template <typename T>
void run_tiled(hipStream_t s, const BandDesc *d_descs, const std::vector<int> &ns, int maxbw, int sched)
{
    void *work = (unsigned char *)const_cast<BandDesc *>(d_descs) + factor_desc_offset(ns.size());
    if (maxbw <= kPanelBw)
        run_tiled_sched<T, T>(s, d_descs, work, ns, maxbw, sched);
    else
        run_tiled_sched<T, double>(s, d_descs, work, ns, maxbw, sched);
}

// Captured launch sequences of factor calls (opt-in: KSH_GRAPHS=1).  A call's sequence (about
// 2 n / 64 launches) depends only on the precision, the device descriptor array, the largest band
// width and the orders of the bands; it is captured into a hipGraph the second time that key is
// seen and replayed from then on (the descriptors themselves are uploaded by an ordinary copy
// before each replay).  At most kGraphs sequences are kept; later keys run eagerly.  Off by
// default: replaying changed the batched arc-length throughput by less than 1% (the launches are
// queued asynchronously well ahead of the GPU), and eager launches are what the kernel profiles
// record.
struct GraphKey {
    int prec;
    int sched;
    const void *descs;
    int maxbw;
    std::vector<int> ns;
    bool operator<(const GraphKey &o) const
    {
        if (prec != o.prec) return prec < o.prec;
        if (sched != o.sched) return sched < o.sched;
        if (descs != o.descs) return descs < o.descs;
        if (maxbw != o.maxbw) return maxbw < o.maxbw;
        return ns < o.ns;
    }
};
struct GraphEntry {
    hipGraphExec_t exec = nullptr;
    int seen = 0;
};
constexpr size_t kGraphs = 64;
std::mutex g_graph_mu;
std::map<GraphKey, GraphEntry> g_graphs;
size_t g_captured = 0;

bool graphs_enabled()
{
    const char *e = std::getenv("KSH_GRAPHS");
    return e && std::strcmp(e, "1") == 0;
}

template <typename T>
int run_tiled_graph(hipStream_t s, const BandDesc *d_descs, const std::vector<int> &ns, int maxbw, int prec, int la)
{
    if (!graphs_enabled() || tune_measuring()) {
        run_tiled<T>(s, d_descs, ns, maxbw, la);
        return KSH_SUCCESS;
    }
    std::lock_guard<std::mutex> lk(g_graph_mu);
    GraphKey key{prec, la, d_descs, maxbw, ns};
    auto it = g_graphs.find(key);
    if (it == g_graphs.end()) {
        if (g_graphs.size() < 4 * kGraphs) g_graphs.emplace(key, GraphEntry{nullptr, 1});
        run_tiled<T>(s, d_descs, ns, maxbw, la);
        return KSH_SUCCESS;
    }
    GraphEntry &en = it->second;
    if (!en.exec && ++en.seen >= 2 && g_captured < kGraphs) {
        hipGraph_t g = nullptr;
        KSH_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        run_tiled<T>(s, d_descs, ns, maxbw, la);
        KSH_HIP(hipStreamEndCapture(s, &g));
        const hipError_t e = hipGraphInstantiate(&en.exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) return fail(KSH_OTHER_ERROR, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        ++g_captured;
    }
    if (en.exec) {
        KSH_HIP(hipGraphLaunch(en.exec, s));
    } else {
        run_tiled<T>(s, d_descs, ns, maxbw, la);
    }
    return KSH_SUCCESS;
}

// Schedule: forced by KSH_LOOKAHEAD, else the autotuner's choice for the bucket of (precision,
// largest band width, number of bands, largest order); its timing calls are whole factor calls.
template <typename T>
int run_factor(hipStream_t s, const BandDesc *d_descs, const std::vector<int> &ns, int maxbw, int prec)
{
    const int forced = schedule_forced();
    if (forced >= 0) return run_tiled_graph<T>(s, d_descs, ns, maxbw, prec, forced);
    const long long bucket =
        ((((long long)prec * 64 + tune_bucket(maxbw)) * 64 + count_bucket((int)ns.size())) * 64) + tune_bucket(ns[0]);
    int rc = KSH_SUCCESS;
    tune_launch("band_factor", bucket, kSchedules, 0, s,
                [&](int v) { rc = run_tiled_graph<T>(s, d_descs, ns, maxbw, prec, v); });
    return rc;
}

}  // namespace

int band_factor_tiled_batch(hipStream_t s, void *d_descs, const std::vector<BandDescHost> &h, int prec)
{
    const size_t es = prec == KSH_FP64 ? sizeof(double) : sizeof(float);
    std::vector<BandDesc> dd;
    for (const auto &x : h) {
        if (!x.active) continue;
        if (x.n < 1) return fail(KSH_SOLVER_ERROR, "empty band");
        if ((size_t)x.n * (size_t)(x.bw + 1) * es >= 0x80000000ull)
            return fail(KSH_SOLVER_ERROR, "band of 2 GiB or more: beyond the band kernels' 32-bit offsets");
        dd.push_back(BandDesc{x.fac, x.n, x.bw, x.info, x.stats, x.x, 1, 0});
    }
    if (dd.empty()) return KSH_SUCCESS;
    std::stable_sort(dd.begin(), dd.end(), [](const BandDesc &a, const BandDesc &b) { return a.n > b.n; });
    std::vector<int> ns(dd.size());
    int maxbw = 0;
    for (size_t i = 0; i < dd.size(); ++i) {
        ns[i] = dd[i].n;
        maxbw = std::max(maxbw, dd[i].bw);
    }
    KSH_HIP(hipMemcpyAsync(d_descs, dd.data(), sizeof(BandDesc) * dd.size(), hipMemcpyHostToDevice, s));
    int rc = prec == KSH_FP64 ? run_factor<double>(s, (const BandDesc *)d_descs, ns, maxbw, prec)
                              : run_factor<float>(s, (const BandDesc *)d_descs, ns, maxbw, prec);
    if (rc) return rc;
    KSH_HIP(hipGetLastError());
    return KSH_SUCCESS;
}

}  // namespace ksh
