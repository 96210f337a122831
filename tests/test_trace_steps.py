"""Cycles of the flow tracing's border tables, on the CPU: entries round a
ring hop in place, as the device's threads do, until none is an exit any more.

Steps round a ring at least double with each round of hops, so they pass any
bound below 2^30 within 31 rounds; the counts of an entry saturate at
2^30 - 1, and rasters may have more cells than that.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "trace_steps.hpp"
using namespace cageo;
int main(int argc, char** argv) {
    const uint32_t cells = (uint32_t)strtoull(argv[1], nullptr, 10);
    const int slots = atoi(argv[2]), steps = atoi(argv[3]);
    std::vector<uint64_t> t(slots + 3);
    for (int i = 0; i < slots; ++i) t[i] = pack(K_EXIT, steps, (i + 1) % slots);
    t[slots] = pack(K_EXIT, 7, 0);                // leads into the ring
    t[slots + 1] = pack(K_EXIT, 5, slots + 2);    // leads to an end
    t[slots + 2] = pack(K_RESOLVED, 3, -42);
    int rounds = 0;
    for (bool pending = true; pending && rounds < 100;) {
        ++rounds;
        pending = false;
        for (uint64_t& e : t) {
            if (kind_of(e) != K_EXIT) continue;
            uint64_t n = hop(e, t[value_of(e)]);
            if (kind_of(n) == K_EXIT) {
                if (is_cycle(steps_of(n), cells)) n = pack(K_STUCK, 0, 0);
                else pending = true;
            }
            e = n;
        }
    }
    bool ok = rounds <= 31 && t[slots + 1] == pack(K_RESOLVED, 8, -42);
    for (int i = 0; i <= slots; ++i) ok = ok && kind_of(t[i]) == K_STUCK;
    printf("%d rounds\n", rounds);
    return ok ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("steps")
    (d / "steps.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cageo_amd", "csrc"),
                    str(d / "steps.cpp"), "-o", str(d / "steps")], check=True)
    return str(d / "steps")


@pytest.mark.parametrize("cells", [64 * 64, 4096 * 4096, 2 ** 30 - 2, 2 ** 30 - 1, 2 ** 30, 2 ** 31 - 1])
@pytest.mark.parametrize("slots,steps", [(1, 1), (2, 64), (7, 1), (256, 3)])
def test_a_cycle_through_tiles_ends(program, cells, slots, steps):
    done = subprocess.run([program, str(cells), str(slots), str(steps)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
