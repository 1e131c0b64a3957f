"""Size rules of the launch header that buffers rely on, evaluated by the host compiler (no device)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "tpsc_launch.hpp"
using namespace tpsc;
constexpr int kN[] = {4, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256};
constexpr long points(int N) { return (long)(N / 2 + 1) * (N / 2 - 1); }
// the rows that a context of lattice N holds suffice on every sub-lattice, and every point has a workgroup
constexpr bool rows_suffice()
{
    for (int N : kN)
        for (int n : kN)
            if (n <= N && (jj_blocks(points(n)) > jj_blocks_max(points(N)) ||
                           jj_blocks(points(n)) * jj_points(points(n)) < points(n)))
                return false;
    return true;
}
static_assert(rows_suffice(), "Lambda rows of a sub-lattice");
"""


def test_lambda_rows_of_sub_lattices(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src = tmp_path / "rules.hip"
    src.write_text(SRC)
    r = subprocess.run([hipcc, "-std=c++17", "--cuda-host-only", "-fsyntax-only", "-I",
                        os.path.join(ROOT, "tpsc_conductivity_amd", "csrc"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
