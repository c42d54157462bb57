"""The moving-frame scan's groups of slices (cltem_amd/csrc/frame_plan.hpp): no GPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cltem_amd", "csrc")

COMMON = r"""
#include <cstdio>
#include <cstdlib>
#include "frame_plan.hpp"
using namespace mse_rt;
#define CHECK(c) do { if (!(c)) { std::printf("ns %d most %d: %s\n", ns, most, #c); std::exit(1); } } while (0)
"""

# the groups hold every slice once and none beyond the specimen; no more groups than needed, none
# deeper than asked for
GROUPS = r"""
int main() {
    for (int ns = 1; ns <= 300; ++ns)
        for (int most = 0; most <= 320; ++most) {
            const int cs = frame_slices(ns, most), room = most < 1 ? 1 : most;
            CHECK(cs >= 1 && cs <= room && cs <= ns);
            int built = 0, groups = 0;
            for (int s = 0; s < ns; ++s)
                if (s % cs == 0) {
                    const int here = frame_group(ns, cs, s);
                    CHECK(here >= 1 && here <= cs && s + here <= ns);
                    CHECK(s + here == ns ? here == (ns - 1) % cs + 1 : here == cs);
                    built += here;
                    ++groups;
                }
            CHECK(built == ns);
            CHECK(groups == (ns + room - 1) / room);
        }
}
"""

# memory that runs out: fewer slices at a time, down to one; never more than there is room for, and
# no smaller groups than halving finds
NO_MEMORY = r"""
int main() {
    for (int ns = 1; ns <= 200; ++ns)
        for (int most = 0; most <= 70; ++most)
            for (int room = 0; room <= 70; ++room) {
                int tried = 0, last = 1 << 30;
                const int cs = frame_slices_that_fit(ns, most, [&](int slices) {
                    CHECK(slices >= 1 && slices < last);
                    last = slices;
                    ++tried;
                    return slices <= room;
                });
                if (room == 0) {
                    CHECK(cs == 0 && last == 1);
                } else {
                    CHECK(cs >= 1 && cs <= room && cs == last);
                    if (frame_slices(ns, most) <= room) CHECK(tried == 1);
                }
            }
}
"""


@pytest.mark.parametrize("body", [GROUPS, NO_MEMORY], ids=["groups", "no_memory"])
def test_frame_plan(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text(COMMON + body)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + CSRC, "-o", exe, str(src)], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
