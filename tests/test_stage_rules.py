"""The index rules of the persistent sweep's exchange (csrc/stages.h), compiled
by the host compiler: the rows that its strip loads address, and the strip
buffers that successive stages use."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "immerseflow_amd", "csrc")


def _run(tmp_path, body):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include "stages.h"\n#include <cstdio>\n#include <initializer_list>\nusing namespace iff;\nint main() {\n' + body + "\nreturn 0;\n}\n")
    subprocess.run([cxx, "-std=c++20", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_strip_rows_lie_in_the_field(tmp_path):
    """Every row of every tile, for tile heights and halos around those in use
    and grids from three rows up, addresses a row of the field, and a row of
    the field addresses itself."""
    _run(tmp_path, """
    for (int ny = 3; ny < 700; ny++)
        for (int ty : {16, 32, 48, 64, 80, 96})
            for (int h : {8, 16, 24, 32})
                for (int t = 0; t * ty < ny - 2; t++)
                    for (int k = 0; k < ty + 2 * h; k++) {
                        const int j = 1 + t * ty - h + k, row = strip_row(j, ny);
                        if (row < 0 || row >= ny || (j >= 0 && j < ny && row != j)) {
                            std::printf("ny %d row %d -> %d\\n", ny, j, row);
                            return 1;
                        }
                    }""")


def test_stages_in_a_row_never_share_a_strip_buffer(tmp_path):
    """Steps of random length over many times 2^32 stages, counted in 32 bits as
    the tiles' counters are: three stages in a row use three buffers, and only
    zeroed counters go back."""
    _run(tmp_path, """
    unsigned long long seed = 12345;
    int zeroed = 0;
    for (unsigned long long most : {1ull, 1000ull, 400000ull, 2147483647ull}) {
        StageCount c;
        unsigned counter = most < 1000000 ? 0xffffffffu - 100000u : 0;  // the tiles' counters
        c.used = counter;
        for (int step = 0; step < 200000; step++) {
            seed = seed * 6364136223846793005ull + 1442695040888963407ull;
            const unsigned n = (unsigned)(most - (seed >> 33) % (most / 8 + 1));  // this step's stages
            if (c.wraps(most)) {
                counter = 0;
                zeroed++;
            }
            for (unsigned l = 0; l < (n < 64 ? n : 64); l++)
                for (unsigned g : {counter + l, counter + n - 2 - l}) {
                    const unsigned a = strip_of(g), b = strip_of(g + 1u), d = strip_of(g + 2u);
                    if (n > l + 2 && (a == b || b == d || a == d)) {
                        std::printf("stage %u: buffers %u %u %u\\n", g, a, b, d);
                        return 1;
                    }
                }
            counter += n;
            if (counter > c.used) {
                std::printf("%u stages, at most %llu expected\\n", counter, c.used);
                return 1;
            }
        }
    }
    if (zeroed < 4) return 1;""")
