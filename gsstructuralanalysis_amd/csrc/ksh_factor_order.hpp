// ksh_factor_order.hpp -- which part of a panel step of the band factor (ksh_factor_tiled.hip) a workgroup or
// wave takes: index arithmetic only, so that the host can check it (tests/test_factor_schedule.py compiles
// this file alone).
#pragma once

#ifdef __HIPCC__
#define KSH_INDEX __host__ __device__ __forceinline__
#else
#define KSH_INDEX inline
#endif

namespace ksh {

// lower-triangle block index p -> (bi, bj), bj <= bi
KSH_INDEX void tri_decode(int p, int &bi, int &bj)
{
    int b = (int)((__builtin_sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
    if ((b + 1) * (b + 2) / 2 <= p) ++b;
    if (b * (b + 1) / 2 > p) --b;
    bi = b;
    bj = p - b * (b + 1) / 2;
}

// Parts of a step's trailing update (32 x 32 blocks (bi, bj), bj <= bi, of the window):
// kAll every block; kNext block columns 0 and 1 (the next panel's columns); kRest the others.  The
// three blocks of the next diagonal block, (0,0), (1,0) and (1,1), are left out of kAll and kNext:
// the workgroup that factors it updates it (diag_panel).
enum TrailPart { kAll = 0, kNext = 1, kRest = 2 };
KSH_INDEX int trail_blocks(int nbk, int part)
{
    const int tail = nbk > 2 ? nbk - 2 : 0;  // block rows below the diagonal block
    return part == kRest ? tail * (tail + 1) / 2 : part == kNext ? 2 * tail : tail * (tail + 1) / 2 + 2 * tail;
}
// block q < trail_blocks(nbk, part) of a part
KSH_INDEX void trail_decode(int q, int nbk, int part, int &bi, int &bj)
{
    if (part == kNext) {
        bj = q < nbk - 2 ? 0 : 1;
        bi = 2 + (bj == 0 ? q : q - (nbk - 2));
    } else {
        tri_decode(part == kAll ? q + 3 : q, bi, bj);
        if (part == kRest) {
            bi += 2;
            bj += 2;
        }
    }
}

// Most bands of a call that schedule 2 serves by fused steps (one launch a step); more take the lookahead
// schedule with two blocks per wave.
constexpr int kFusedBands = 8;
// The autotuner's bucket for the number of bands, ceil(log2): its edges lie where a schedule changes, so no
// choice timed on fused steps serves calls that cannot have them (9 to 15 bands of 32 x 32 roofs took
// 17% to 21% longer with schedule 2 than with the best, which 8 bands have as their best).
KSH_INDEX int count_bucket(int bands)
{
    int b = 0;
    while (1 << b < bands) ++b;
    return b;
}

// Panel workspaces of a band: three, by panel, since a launch of the fused schedule writes the next panel's
// while it still reads this one's and the last one's.
constexpr int kPanelSlots = 3;
KSH_INDEX int panel_slot(int c0) { return c0 / 64 % kPanelSlots; }

// XCD-aware assignment of a launch's workgroups to (band, index within the band).  Workgroups are
// dispatched to the 8 XCDs round robin (id mod 8), each XCD with its own L2.  Every trailing block
// of a band reads that band's panel, so with 8 or more bands the workgroups of band b take the ids
// h = b (mod 8): all of them run on one XCD and its L2 serves the panel, which otherwise every
// XCD would fetch once per band.  The diagonal blocks' workgroups already put band b on workgroup b, the
// same XCD.  With fewer bands than XCDs the plain mapping keeps every XCD busy.  A band past the active
// ones marks a padding workgroup of the XCD-aware grid (8 ceil(active / 8) wg of them).
constexpr int kXcds = 8;
KSH_INDEX void workgroup_decode(int h, int active, int wg, int &band, int &local)
{
    if (active < kXcds) {
        band = h / wg;
        local = h % wg;
    } else {
        const int s = h / kXcds;
        band = h % kXcds + kXcds * (s / wg);
        local = s % wg;
    }
}
inline unsigned band_grid(int active, int wg)
{
    return (unsigned)(active < kXcds ? active * wg : ((active + kXcds - 1) / kXcds) * kXcds * wg);
}

}  // namespace ksh
