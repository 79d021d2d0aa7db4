// ksh_elim_steps.hpp -- elimination steps of a 16 x 16 symmetric block held one row per lane (the
// diagonal blocks of the band factor, ksh_factor_tiled.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace ksh {

// Broadcast of lane J of each 16-lane row to the row's lanes (DPP row_newbcast).  A DPP read must not
// follow the write of its source within two wait states, which the compiler does not see through
// inline assembly: the blocks below hold their own waits.
template <int J>
__device__ __forceinline__ double row_bcast(double v)
{
    double r;
    asm("s_nop 1\n\tv_mov_b64_dpp %[r], %[v] row_newbcast:%[jj] row_mask:0xf bank_mask:0xf" : [r] "=v"(r) : [v] "v"(v), [jj] "n"(J));
    return r;
}
template <int J>
__device__ __forceinline__ float row_bcast(float v)
{
    float r;
    asm("s_nop 1\n\tv_mov_b32_dpp %[r], %[v] row_newbcast:%[jj] row_mask:0xf bank_mask:0xf" : [r] "=v"(r) : [v] "v"(v), [jj] "n"(J));
    return r;
}

// Elimination step J of a 16 x 16 block, lane = row r (the four lane rows hold the same rows): e[k] +=
// m row_J(e[k]) for k > J, w[q] += mw row_J(w[q]), where row_J is lane J's value (DPP inside the
// multiply-add, so no LDS round trip and no scalar registers); returns the next pivot, broadcast, and
// its reciprocal's estimate (of -d) in nr, both begun while the rest of the step issues.  Each block is one
// piece of assembly: a wait before its first DPP read covers whatever wrote the operands, inside it
// every DPP read is at least two instructions behind its source's write, and the last instructions
// keep the estimate's first use a wait state away.
template <int J>
__device__ __forceinline__ double elim_step(double (&e)[16], double (&w)[4], double m, double mw, double &nr)
{
    double d;
    if constexpr (J == 0)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e1], %[e1], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e2], %[e2], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e3], %[e3], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e1] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e4], %[e4], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e5], %[e5], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e1] "+v"(e[1]), [e2] "+v"(e[2]), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 1)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e2], %[e2], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e3], %[e3], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e4], %[e4], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e2] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e5], %[e5], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e2] "+v"(e[2]), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 2)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e3], %[e3], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e4], %[e4], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e5], %[e5], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e3] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 3)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e4], %[e4], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e5], %[e5], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e4] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 4)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e5], %[e5], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e5] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 5)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e6], %[e6], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e6] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 6)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e7], %[e7], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e7] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 7)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e8], %[e8], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e8] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 8)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e9], %[e9], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e9] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 9)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e10], %[e10], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e10] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 10)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e11], %[e11], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e11] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 11)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e12], %[e12], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e12] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 12)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e13], %[e13], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e13] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 13)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e14], %[e14], %[m] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e14] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 14)
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %[e15], %[e15], %[m] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w0], %[w0], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w1], %[w1], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b64_dpp %[d], %[e15] row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w2], %[w2], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %[w3], %[w3], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f64 %[r], -%[d]\n\t"
            "s_nop 1\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    return d;
}
template <int J>
__device__ __forceinline__ float elim_step(float (&e)[16], float (&w)[4], float m, float mw, float &nr)
{
    float d;
    if constexpr (J == 0)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e1], %[e1], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e2], %[e2], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e3], %[e3], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e1] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e4], %[e4], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e5], %[e5], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e1] "+v"(e[1]), [e2] "+v"(e[2]), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 1)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e2], %[e2], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e3], %[e3], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e4], %[e4], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e2] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e5], %[e5], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e2] "+v"(e[2]), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 2)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e3], %[e3], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e4], %[e4], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e5], %[e5], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e3] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e3] "+v"(e[3]), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 3)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e4], %[e4], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e5], %[e5], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e4] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e4] "+v"(e[4]), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 4)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e5], %[e5], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e5] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e5] "+v"(e[5]), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 5)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e6], %[e6], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e6] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e6] "+v"(e[6]), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 6)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e7], %[e7], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e7] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e7] "+v"(e[7]), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 7)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e8], %[e8], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e8] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e8] "+v"(e[8]), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 8)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e9], %[e9], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e9] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e9] "+v"(e[9]), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 9)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e10], %[e10], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e10] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e10] "+v"(e[10]), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 10)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e11], %[e11], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e11] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e11] "+v"(e[11]), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 11)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e12], %[e12], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e12] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e12] "+v"(e[12]), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 12)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e13], %[e13], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e13] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e13] "+v"(e[13]), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 13)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e14], %[e14], %[m] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e14] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e14] "+v"(e[14]), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    if constexpr (J == 14)
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %[e15], %[e15], %[m] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w0], %[w0], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w1], %[w1], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_mov_b32_dpp %[d], %[e15] row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w2], %[w2], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %[w3], %[w3], %[mw] row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
            "v_rcp_f32 %[r], -%[d]\n\t"
            "s_nop 1\n\t"
            : [d] "=&v"(d), [r] "=&v"(nr), [e15] "+v"(e[15]), [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3])
            : [m] "v"(m), [mw] "v"(mw));
    return d;
}

}  // namespace ksh
