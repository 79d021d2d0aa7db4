"""Order of the team solve's leader steps (gsstructuralanalysis_amd/csrc/ksh_team_order.hpp, the file the
kernel itself includes), compiled for the CPU.

A leader step is, for each of the four waves: write the wave's partial sums to the step's LDS buffer,
barrier, read all waves' sums from it.  Between two barriers a wave may so still read for step t
while another already writes for step t + 1.  The test takes the steps of a whole solve, forward and
backward, for 3 to 70 blocks of 64 rows (a team takes three or more) and checks that no buffer is written
in an interval between barriers in which it is read."""
import subprocess

import pytest

CSRC = __file__.rsplit("/tests/", 1)[0] + "/gsstructuralanalysis_amd/csrc"

PROGRAM = """
#include <cstdio>
#include "ksh_team_order.hpp"
int main()
{
    for (int nblk = 3; nblk <= 70; ++nblk) {
        for (int sweep = 0; sweep < 2; ++sweep)
            for (int s = 0; s < nblk; ++s) std::printf("%d ", ksh::lead_buffer(ksh::lead_step(sweep == 0, nblk, s)));
        std::printf("\\n");
    }
    return 0;
}
"""


def conflicts(buffers):
    """Steps t whose buffer is written for step t + 1 while it may still be read for step t."""
    reads, writes = {}, {}  # interval (number of barriers passed) -> buffers
    for t, b in enumerate(buffers):
        writes.setdefault(t, set()).add(b)      # before the step's barrier
        reads.setdefault(t + 1, set()).add(b)   # after it
    return [t for t in reads if reads[t] & writes.get(t, set())]


@pytest.fixture(scope="module")
def buffers(tmp_path_factory):
    d = tmp_path_factory.mktemp("team_order")
    src, exe = d / "order.cpp", d / "order"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)])
    out = subprocess.check_output([str(exe)], text=True).splitlines()
    return {len(line.split()) // 2: [int(v) for v in line.split()] for line in out}


def test_no_buffer_is_written_while_it_is_read(buffers):
    assert sorted(buffers) == list(range(3, 71))
    for nblk, seq in buffers.items():
        assert len(seq) == 2 * nblk
        assert conflicts(seq) == [], nblk


def test_the_check_sees_a_sweep_that_starts_anew():
    """Buffers that start at 0 again with the backward sweep meet where the number of blocks is odd."""
    for nblk in range(3, 12):
        anew = [s % 2 for s in range(nblk)] * 2
        assert conflicts(anew) == ([nblk] if nblk % 2 else [])
