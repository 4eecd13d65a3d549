"""Launch shapes at the largest hierarchy a handle takes, by the compiler's constants (a
launch has fewer than 2^32 threads in a dimension); no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "bin", "hipcc")

CHECK = """
#include "heom_device.hpp"
using namespace heom_hip;
static_assert(matrix_blocks(1) == 1 && matrix_blocks(65) == 65);
static_assert((int64_t)matrix_blocks(kMaxAdos) * kMatrixThreads < (int64_t)1 << 32);
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_matrix_copies_of_the_largest_hierarchy(tmp_path):
    src = tmp_path / "check.hip"
    src.write_text(CHECK)
    r = subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only",
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "dm-heom_amd", "csrc"), str(src)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
