"""Optional device scratch (device_buffer::try_allocate, which the exact batches' shares of the triangles use): a
request that cannot be met is reported, not thrown, and leaves no HIP error for the next launch check."""

import os
import subprocess

import pytest

from smallgwn_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "gwn_core.hpp"
int main() {
    gwn::device_buffer<double> b;
    bool const got = b.try_allocate(std::size_t(1) << 47, nullptr);  // 1 PiB, or no device at all
    std::printf("%d %d %zu %d\n", int(got), int(b.ptr != nullptr), b.count, int(hipPeekAtLastError()));
}
"""


def test_unmet_request_is_reported_and_leaves_no_error(tmp_path):
    if not os.path.exists(build.LIB_PATH):
        pytest.skip("library not built")
    src, exe = tmp_path / "scratch.hip", tmp_path / "scratch"
    src.write_text(PROGRAM)
    subprocess.run([build.hipcc(), "--cuda-host-only", *build.COMMON_FLAGS, "-w", "-I", os.path.join(ROOT, "smallgwn_amd", "csrc"),
                    str(src), "-o", str(exe), "-L", os.path.dirname(build.LIB_PATH), "-l:" + os.path.basename(build.LIB_PATH),
                    "-Wl,-rpath," + os.path.dirname(build.LIB_PATH)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert out[:3] == ["0", "0", "0"]
    assert out[3] in ("0", "100")  # hipErrorNoDevice: without a device every HIP call reports it anew
