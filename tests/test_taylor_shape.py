"""The launch shapes of the series over dense rows, compiled for the host: every launch fits the room for its norms -- series
of at most a batch of terms with norms, squarings of any number of terms without -- and every row and column has a lane."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "taylor_shape.hpp"
using namespace dq;
int main() {
    int seen = 0;
    for (int64_t N = 1; N <= TAYLOR_MAX_N; ++N) {
        const int i = taylor_shape(N);
        const TaylorShape s = TAYLOR_SHAPES[i];
        seen |= 1 << i;
        const int64_t room = taylor_parts_room(N);
        if (int64_t(s.threads) * s.cols < N || taylor_grid(N) * s.rows < N) return std::printf("%ld: rows\n", long(N)), 1;
        for (int terms = 1; terms <= TAYLOR_BATCH; ++terms)
            for (int64_t block = 0, last = taylor_grid(N) - 1; block <= last; block += last ? last : 1)
                if ((terms - 1) * taylor_grid(N) + block >= room) return std::printf("%ld: %d terms\n", long(N), terms), 1;
        if (taylor_parts(N, TAYLOR_BATCH, true) > room) return std::printf("%ld: batch\n", long(N)), 1;
        if (taylor_parts(N, TAYLOR_BATCH + 1, true) <= room) return std::printf("%ld: unchecked\n", long(N)), 1;
        if (taylor_parts(N, 100, false) != 0) return std::printf("%ld: squaring\n", long(N)), 1;
    }
    return seen == 63 ? 0 : 2;  // all six shapes
}
"""


def test_launches_fit_their_workspace(tmp_path):
    src, exe = tmp_path / "shape.cpp", tmp_path / "shape"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "diaq_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
