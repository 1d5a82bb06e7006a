"""touch_pages (csrc/pages.h) faults a buffer's pages in and leaves what they
hold, at any alignment: a fetch that fails behind it has not changed the
caller's buffer."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "immerseflow_amd", "csrc")


def test_touch_pages_keeps_contents(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("""
#include "pages.h"
#include <vector>
int main() {
    for (size_t off : {0, 1, 8, 4095})
        for (size_t n : {0, 1, 8, 4095, 4096, 4097, 70001}) {
            std::vector<unsigned char> v(off + n + 1);
            for (size_t k = 0; k < v.size(); k++) v[k] = (unsigned char)(k * 7 + 1);
            iff::touch_pages(v.data() + off, n);
            for (size_t k = 0; k < v.size(); k++)
                if (v[k] != (unsigned char)(k * 7 + 1)) return 1;
        }
    return 0;
}
""")
    subprocess.run([cxx, "-std=c++20", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
