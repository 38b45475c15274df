"""The whole-number limits that k-fault sampling compares its draws with
(clifft_amd/csrc/svm_tree_plan.h) decide as the comparison of the numbers does,
also for probabilities that are not numbers: the quotient of two sums over
millions of sites that overflowed is one, and no draw is below it."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
E = 2.0 ** -53

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def limit(tmp_path_factory):
    so = tmp_path_factory.mktemp("limit") / "liblimit.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "clifft_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "draw_limit_check.cpp"),
                    "-o", str(so)], check=True, timeout=120)
    f = ctypes.CDLL(str(so)).limit
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_double]
    return f


@pytest.mark.parametrize("p", [0.0, -1.0, 5e-324, E / 2, E, 1.5 * E, 2 * E, 1e-3, 1 / 3, 0.5, 1 - E, 1 - E / 2, 1.0, 1.5, np.inf,
                               -np.inf, np.nan])
def test_draws_below(limit, p):
    n = limit(p)
    assert 0 <= n <= 1 << 53
    for x in {0, 1, 2, (1 << 52), (1 << 53) - 1} | {x for x in (n - 2, n - 1, n, n + 1) if 0 <= x < 1 << 53}:
        assert (x < n) == (x * E < p), x
