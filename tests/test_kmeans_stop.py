"""The stop flag of the merge's Lloyd passes (csrc/kmeans_stop.hpp), checked by
the compiler: whatever moment a wave of pass `it` reads the flag at, before or
after its own launch's store, it goes on; every later pass stops.  A flag that
only says "stop" lets the waves of one block disagree, and those that stay
then wait at barriers for, and read LDS of, those that left."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(__file__), "..", "tensor-adapt_amd", "csrc")

SRC = """
#include "kmeans_stop.hpp"
using namespace ta;
constexpr bool holds(int passes) {
    for (int it = 0; it < passes; it++) {
        if (kmeans_stopped(kKmeansRunning, it)) return false;
        const int32_t stored = kmeans_stop_after(it);
        if (stored == kKmeansRunning) return false;
        if (kmeans_stopped(stored, it) != kmeans_stopped(kKmeansRunning, it)) return false;
        for (int later = it + 1; later < passes; later++)
            if (!kmeans_stopped(stored, later)) return false;
    }
    return true;
}
static_assert(holds(300), "every wave of a launch agrees; later launches stop");
"""


def test_waves_of_a_launch_agree(tmp_path):
    f = tmp_path / "stop.cpp"
    f.write_text(SRC)
    subprocess.check_call(["g++", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(f)])
