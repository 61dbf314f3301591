"""Launch shapes, on the host.  Batches with several lanes per query: every slice stays within HIP's 2^32
work-items a dimension, and the slices cover each query once, up to the sizes that one lane per query serves.
The batched mode's tuner: no two of its first candidates run the same launch."""

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


SHAPES = r"""
#include <cstdio>
#include "gwn_tune.hpp"
int main(int, char **) {
    for (auto const &s : gwn::batch_shapes())
        std::printf("%d %d %d %d\n", s.block, s.chunk, s.blocks_per_cu, s.traversal);
}
"""


def _output(tmp_path, program, *args):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "host.cpp", tmp_path / "host"
    src.write_text(program)
    subprocess.run([cxx, "-std=c++20", "-I", os.path.join(ROOT, "smallgwn_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe), *args], check=True, capture_output=True, text=True).stdout.split("\n")[:-1]


def test_tuner_shapes_are_distinct_launches(tmp_path):
    shapes = [tuple(map(int, line.split())) for line in _output(tmp_path, SHAPES)]
    launches = [(block, bpc, traversal, chunk if traversal else 0) for block, chunk, bpc, traversal in shapes]
    assert len(set(launches)) == len(launches)
    assert {s[3] for s in shapes} == {0, 1} and all(chunk % block == 0 for block, chunk, _, _ in shapes)


@pytest.mark.parametrize("n", [1, (1 << 28) - 1, 1 << 28, (1 << 28) + 1, 1 << 30, (1 << 32) - 256])
def test_quad_slices(tmp_path, n):
    lines = _output(tmp_path, PROGRAM, str(n))
    at = 0
    for first, count in (map(int, line.split()) for line in lines[1:]):
        assert first == at and 0 < count <= int(lines[0])
        assert -(-4 * count // 256) * 256 < 1 << 32
        at += count
    assert at == n
