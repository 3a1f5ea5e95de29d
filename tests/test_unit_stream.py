"""The cursors of a K-side workgroup (sa2_units.h), walked on the host as split_kv_lone_kernel walks them, with the compiler's check for
signed overflow: every unit of the stream comes once and the walk ends."""
import subprocess

from simplical_attn_amd import build

PROGRAM = r"""
#include "sa2_units.h"
#include <cstdio>
#include <initializer_list>
using namespace sa2;
int main() {
    for (int w2 : {0, 1, 2, 7, 40}) for (int blocks : {1, 2, 5}) for (int first : {0, 3}) for (int cut : {0, 1}) {
        auto last_of = [&](int ib) { int d = 32 * ib + 31 < w2 ? 32 * ib + 31 : w2; return cut && ib == blocks - 1 && d > 1 ? d - 1 : d; };
        auto stop_of = [&](int ib) { return ib < blocks ? last_of(ib) : NEVER; };
        const int d0 = first <= last_of(0) ? first : 0;
        int f_ib = 0, f_delta = d0, f_stop = stop_of(0), l_ib = 0, l_delta = d0, l_stop = f_stop, ib = 0, delta = d0, stop = f_stop;
        auto request_turn = [&] { if (l_delta > l_stop) { ++l_ib; l_delta = 0; l_stop = stop_of(l_ib); } };
        auto form_turn = [&](int n) { f_delta += n; if (f_delta > f_stop) { ++f_ib; f_delta = 0; f_stop = stop_of(f_ib); } };
        ++l_delta; request_turn();
        for (int x = 0; x < 2; ++x) { form_turn(1); ++l_delta; request_turn(); }
        long done = 0, all = -d0, steps = 0;
        for (int x = 0; x < blocks; ++x) all += last_of(x) + 1;
        while (ib < blocks) {
            int n = units_left(units_left(stop - delta + 1, f_delta, f_stop), l_delta, l_stop);
            if (stop > ib * 32) { const int whole = ib * 32 - delta + 1; if (whole < n) n = whole > 1 ? whole : 1; }
            if (n < 1 || ++steps > all) return std::printf("w2 %d blocks %d: %d units at (%d, %d)\n", w2, blocks, n, ib, delta), 1;
            done += n;
            l_delta += n;
            request_turn();
            form_turn(n);
            delta += n;
            if (delta > stop) { ++ib; delta = 0; if (ib < blocks) stop = last_of(ib); }
        }
        if (done != all) return std::printf("w2 %d blocks %d: %ld of %ld units\n", w2, blocks, done, all), 1;
    }
    static_assert(units_left(5, 0, NEVER) == 5 && units_left(5, 3, 7) == 5 && units_left(5, 4, 7) == 4 && units_left(5, 7, 7) == 1, "");
}
"""


def test_the_cursors_of_a_stream(tmp_path):
    src, exe = str(tmp_path / "walk.cpp"), str(tmp_path / "walk")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O0", "-fsanitize=signed-integer-overflow", "-fno-sanitize-recover=all", "-I", build.CSRC, src, "-o", exe], check=True)
    got = subprocess.run([exe], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout + got.stderr
