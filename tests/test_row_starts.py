"""The sub-tile range of a row (csrc/row_starts.hpp) in a host build: inside the
array of first rows for every 64-bit row pointer, also one that is no row
pointer, and exact for one that is."""

import os
import shutil
import subprocess

import pytest

import flagsparse_amd

CSRC = os.path.join(os.path.dirname(flagsparse_amd.__file__), "csrc")
ITEMS = 768
TOP = 2**63 - 1
PROGRAM = """
#include "row_starts.hpp"
#include <cstdio>
int main() {
  long long e, items, n_sub;
  while (std::scanf("%lld %lld %lld", &e, &items, &n_sub) == 3)
    std::printf("%lld\\n", (long long)fs::row_sub_tile(e, items, n_sub));
}
"""


def test_sub_tiles_stay_in_range(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", exe, str(tmp_path / "main.cpp")], check=True)
    entries = [-TOP - 1, -1, 0, 1, 767, 768, 769, 1536, 10**6, 2**31, 2**32, TOP - 768, TOP - 767, TOP - 766, TOP]
    cases = [(e, ITEMS, n) for e in entries for n in (1, 2, 3, 1303, 2**32 // ITEMS)]
    text = "\n".join(" ".join(map(str, c)) for c in cases)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
    for (e, items, n), got in zip(cases, map(int, out.split())):
        assert 0 <= got <= n
        assert got == min(n, max(0, -(-e // items))), (e, n)
