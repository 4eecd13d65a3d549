"""Launch shapes at the largest hierarchy a handle takes, by the compiler's constants (a
launch has fewer than 2^32 threads in a dimension); no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "bin", "hipcc")

def compiles(tmp_path, code):
    src = tmp_path / "check.hip"
    src.write_text(code)
    csrc = os.path.join(ROOT, "dm-heom_amd", "csrc")
    r = subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only",
                        "-fconstexpr-steps=200000000",
                        "-I" + os.path.join(ROOT, "include"), "-I" + csrc, str(src)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_matrix_copies_of_the_largest_hierarchy(tmp_path):
    compiles(tmp_path, """
#include "heom_device.hpp"
using namespace heom_hip;
static_assert(matrix_blocks(1) == 1 && matrix_blocks(65) == 65);
static_assert((int64_t)matrix_blocks(kMaxAdos) * kMatrixThreads < (int64_t)1 << 32);
""")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_wide_workgroups_fit_and_the_default_may_be_chosen(tmp_path):
    """For every N, mode list and hierarchy size: the default number of wavefronts per workgroup
    is one that a caller may set and the autotuner times, and whatever may be set fits the LDS."""
    compiles(tmp_path, """
#include "stage_wide.hip"
using namespace heom_hip;
template <typename R, int SZ>
constexpr bool fits(int from, int to)
{
    const int cb = (int)sizeof(c2<R>);
    for (int N = from; N <= to; ++N)
        for (int real = 0; real < 2; ++real)
            for (int W : {1, N, 2 * N, 65, 71, 400})
                for (int len : {1, 2 * N - 1, N * N}) {
                    const int most = wide_most_waves(N, cb, real, W, len);
                    for (int ntiles : {1, 5, 9, 103, 5000})
                        for (int ados : {0, 1, 2, 4, 8}) {
                            const WideShape s = wide_shape<R, SZ>(N, real, W, len, ntiles, ados);
                            if (s.T > most || (ados > 0 && ados <= most && s.T != ados) ||
                                wide_lds(N, cb, real, kWideGamLds<R, SZ>, s.T, wide_where_bytes(W, len)).total > 163840)
                                return false;
                        }
                }
    return true;
}
static_assert(fits<double, 16>(9, 16) && fits<double, 24>(17, 24) && fits<double, 32>(25, 32));
static_assert(fits<float, 16>(9, 16) && fits<float, 24>(17, 24) && fits<float, 32>(25, 32));
""")
