"""Index rules of the kernels (csrc/access_rules.hpp), checked exhaustively over
small shapes on the CPU: every load that a rule allows lies inside its operand."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nalgebra_amd", "csrc")


def _run(tmp_path, body):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include "access_rules.hpp"\n#include <algorithm>\n#include <cstdio>\n'
                   "using namespace nrocm_rules;\nint main()\n{\n" + body + "\n    return 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_gemm_wide_slices_stay_inside(tmp_path):
    """Column strides of either sign, smaller and larger than the column."""
    _run(tmp_path, r"""
    const long tile = 8, bk = 4;
    long wide = 0;
    for (long m = 1; m <= 20; ++m)
        for (long k = 1; k <= 10; ++k)
            for (long lda = -24; lda <= 24; ++lda) {
                const long first = std::min(0L, (k - 1) * lda), end = std::max(0L, (k - 1) * lda) + m;
                for (long bm = 0; bm < m; bm += tile)
                    for (long k0 = 0; k0 < k; k0 += bk) {
                        if (!gemm_wide_slice(m, k, lda, bm, tile, k0, bk)) continue;
                        ++wide;
                        for (long c = k0; c < k0 + bk; ++c)
                            for (long r = bm; r < bm + tile; ++r)
                                if (c >= k || c * lda + r < first || c * lda + r >= end) {
                                    std::printf("m %ld k %ld lda %ld: row %ld column %ld\n", m, k, lda, r, c);
                                    return 1;
                                }
                    }
            }
    if (wide == 0) return 2;""")


def test_dot_phases_read_rows_of_x(tmp_path):
    """Every element of every phase, the rounds that end past the last row too."""
    _run(tmp_path, r"""
    for (int n = 1; n <= 70; ++n)
        for (int p = 0; p <= dot_last_phase(n); ++p)
            for (int e = 0; e < 200; ++e) {
                const int row = dot_first_row(n, p) + std::min(e, dot_last_element(n, p));
                if (row < 0 || row >= n || (e < p && p < n && row != n - p + e)) {
                    std::printf("n %d phase %d element %d: row %d\n", n, p, e, row);
                    return 1;
                }
            }""")
