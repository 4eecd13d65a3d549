"""Launch shapes at the largest hierarchy a handle takes, by the compiler's constants (a
launch has fewer than 2^32 threads in a dimension); no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "bin", "hipcc")
MODES = """
#include <cstdio>
#include "handle.hpp"
using namespace heom_hip;
int main()
{
    constexpr int N = @N@, W = N + 1, CLASSES = @CLASSES@;
    std::vector<std::vector<Term>> per(CLASSES * N * N);
    for (int cl = 0; cl < CLASSES; ++cl)
        for (int i = 0; i < N; ++i)
            for (int j = 0; j < N; ++j)
                for (int m = 0; m < W; ++m)
                    if (m == i || m == j || (m == N && cl == 1)) {
                        Term t{};
                        t.mode = m;
                        t.plus_c = 1000 * cl + m;
                        per[(cl * N + i) * N + j].push_back(t);
                    }
    const heom_rt::WideModes t = heom_rt::wide_modes(per, CLASSES, N, W);
    if ((t.stride == 0) != (CLASSES == 2) || t.terms.size() != CLASSES * t.words || t.where.size() != t.terms.size())
        return 1;
    for (int cl = 0; cl < CLASSES; ++cl) {
        int rounds = 0;
        for (int m = 0; m < W; ++m) {
            const int count = m < N ? 2 * N - 1 : cl ? N * N : 0;
            const uint32_t* where = &t.where[cl * t.words];
            const int from = t.stride ? m * t.stride : where[m] & 0xffff, n = t.stride ? t.stride : where[m] >> 16;
            if (from < 0 || from >= t.words || from + n > t.words)
                return 2;
            rounds += n > 64 ? (n + 63) / 64 : 1;
            int last = -1, seen = 0;
            for (int k = from; k < from + n; ++k) {
                const Term& e = t.terms[cl * t.words + k];
                if (where[k] >> 16 == 0xffff)
                    continue;
                const int i = e.mode / N, j = e.mode % N;
                if ((m < N && i != m && j != m) || e.mode <= last || e.plus_c != 1000 * cl + m ||
                    where[k] != (uint32_t)(wide_pos(N, i, j) | (i * wide_pitch(N) + j) << 16))
                    return 3;
                last = e.mode;
                ++seen;
            }
            if (seen != count)
                return 4;
        }
        if (rounds != W + cl * ((N * N + 63) / 64 - 1))
            return 5;
    }
    return 0;
}
"""


def compiles(tmp_path, code, *how):
    src = tmp_path / "check.hip"
    src.write_text(code)
    csrc = os.path.join(ROOT, "dm-heom_amd", "csrc")
    r = subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "--cuda-host-only", *(how or ["-fsyntax-only"]),
                        "-fconstexpr-steps=200000000", "-I" + os.path.join(ROOT, "include"), "-I" + csrc, str(src)],
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
            for (int words : {1, N, N * (2 * N - 1), 2900, 4095, 4096, 4097, 8 * N * N}) {
                const int most = wide_most_waves(N, cb, real, words);
                for (int ntiles : {1, 5, 9, 103, 5000})
                    for (int ados : {0, 1, 2, 4, 8}) {
                        const WideShape s = wide_shape<R, SZ>(N, real, words, ntiles, ados);
                        if (s.T > most || (ados > 0 && ados <= most && s.T != ados) ||
                            wide_lds(N, cb, real, kWideGamLds<R, SZ>, s.T, wide_where_bytes(words)).total > 163840)
                            return false;
                    }
            }
    return true;
}
static_assert(fits<double, 16>(9, 16) && fits<double, 24>(17, 24) && fits<double, 32>(25, 32));
static_assert(fits<float, 16>(9, 16) && fits<float, 24>(17, 24) && fits<float, 32>(25, 32));
""")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("N,classes", [(9, 1), (9, 2), (16, 2), (24, 2), (32, 1), (32, 2)])
def test_modes_take_the_rounds_of_their_own_lists(tmp_path, N, classes):
    """A bath per site and, in a second class, one more that couples to all sites: every mode's
    list holds its elements in their order, and an ADO with an edge in every mode makes one
    round of 64 elements per site and ceil(N N / 64) for the shared bath."""
    compiles(tmp_path, MODES.replace("@N@", str(N)).replace("@CLASSES@", str(classes)), "-o", str(tmp_path / "check"))
    assert subprocess.run([str(tmp_path / "check")], timeout=60).returncode == 0
