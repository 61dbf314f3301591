"""Launch sizes of batches with several lanes per query, on the host: every slice stays within HIP's 2^32
work-items a dimension, and the slices cover each query once, up to the sizes that one lane per query serves."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "gwn_slices.hpp"
int main(int, char **argv) {
    std::printf("%zu\n", gwn::k_quad_slice);
    gwn::for_each_slice(std::strtoull(argv[1], nullptr, 0), gwn::k_quad_slice,
                        [](std::size_t first, std::size_t count) { std::printf("%zu %zu\n", first, count); });
}
"""


@pytest.mark.parametrize("n", [1, (1 << 28) - 1, 1 << 28, (1 << 28) + 1, 1 << 30, (1 << 32) - 256])
def test_quad_slices(tmp_path, n):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "slices.cpp", tmp_path / "slices"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++20", "-I", os.path.join(ROOT, "smallgwn_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    lines = subprocess.run([str(exe), str(n)], check=True, capture_output=True, text=True).stdout.split("\n")[:-1]
    at = 0
    for first, count in (map(int, line.split()) for line in lines[1:]):
        assert first == at and 0 < count <= int(lines[0])
        assert -(-4 * count // 256) * 256 < 1 << 32
        at += count
    assert at == n
