// ksh_team_order.hpp -- order of the leader's steps in a team solve (ksh_solve_team.hip), as far as the
// host can check it (tests/test_team_order.py compiles this file alone).
#pragma once

namespace ksh {

// Step s of a sweep over nblk blocks, counted over the whole solve: the backward sweep follows the forward one
constexpr int lead_step(bool forward, int nblk, int s) { return forward ? s : nblk + s; }

// LDS buffer of a step's exchange.  A step is: write the wave's partial sums, barrier, read the other waves'.
// With one barrier a step, a wave may write for the next step while another still reads for this one,
// so steps that follow each other use different buffers, also from the last step of the forward sweep
// (of an odd or even number) to the first of the backward sweep.
constexpr int kLeadBuffers = 2;
constexpr int lead_buffer(int step) { return step % kLeadBuffers; }

}  // namespace ksh
