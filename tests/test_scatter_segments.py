"""The segment arithmetic of the scattered-product SpMV
(csrc/scatter_segments.hpp) in a host build: every entry of a bucket lies in
exactly one segment, up to the largest entry count the calls take."""

import os
import shutil
import subprocess

import pytest

import flagsparse_amd

CSRC = os.path.join(os.path.dirname(flagsparse_amd.__file__), "csrc")
MAX_NNZ = 0xFFFFFFFF - 6144 - 1  # entry counts below 2^32 - 1 less a tile of 6144 are taken
PROGRAM = """
#include "scatter_segments.hpp"
#include <cstdio>
int main() {
  long long nnz, used, c;
  while (std::scanf("%lld %lld %lld", &nnz, &used, &c) == 3) {
    const uint32_t items = fs::scatter_segment_items(nnz, used);
    std::printf("%u %u\\n", items, fs::scatter_bucket_segments((uint32_t)c, items));
  }
}
"""


@pytest.fixture(scope="module")
def segments(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("segments")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(d / "main"), str(d / "main.cpp")], check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return run


def test_segments_cover_a_bucket_once(segments):
    cases = []
    for nnz in (1, 2047, 2048, 2049, 10**6, 2**31, 4_290_800_000, 4_293_000_000, MAX_NNZ - 1, MAX_NNZ):
        for used in (1, 2, 1024, 2048):
            for c in sorted({0, 1, min(nnz, 2048), min(nnz, 2049), nnz // used, nnz - nnz // 5, nnz - 1, nnz}):
                cases.append((nnz, used, c))
    for (nnz, used, c), (items, count) in zip(cases, segments(cases)):
        assert 2048 <= items < 2**32
        assert count == max(1, -(-c // items)), (nnz, used, c)
        # the largest offset a segment forms: its end, rounded up to 256 entries
        assert nnz + 256 < 2**32
