"""expm_col0 (reapers/expm.h), the first column of the exponential of a
Krylov driver's Hessenberg matrix, against the first column of expm in the
same header, by a small program (tests/expm_check.cc): skew-Hermitian
tridiagonal, Hessenberg and full matrices of 1 to 60 rows at norms that take
every Pade degree, scaling, and the squaring path.

Tolerance: both evaluate the same Pade approximants of A / 2^s; applying r
2^s times or squaring it s times each lets a relative rounding of a few
eps64 grow by up to 2^s = ||A|| / 5.4: 1e-15 (1 + ||A||)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def output(tmp_path_factory):
    cxx = shutil.which(os.environ.get("CXX", "g++"))
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path_factory.mktemp("expm") / "expm_check")
    r = subprocess.run([cxx, "-O2", "-std=c++20", "-ffp-contract=off",
                        "-I" + os.path.join(ROOT, "reapers_amd", "include", "reapers"),
                        os.path.join(ROOT, "tests", "expm_check.cc"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return subprocess.run([exe], capture_output=True, text=True, check=True).stdout


def test_first_column_matches_expm(output):
    rows = re.findall(r"norm (\S+) skew (\S+) hess (\S+) full (\S+)", output)
    assert len(rows) == 8
    for row in rows:
        nrm, *errs = map(float, row)
        assert max(errs) <= 1e-15 * (1 + nrm), row


def test_special_matrices(output):
    assert re.search(r"^zero 0\.000e\+00$", output, re.M)
    assert float(re.search(r"nilpotent (\S+)", output).group(1)) <= 2e-16
    assert "empty 0 nan 1" in output
