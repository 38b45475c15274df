"""The pool of pinned blocks (clifft_amd/csrc/svm_block_pool.h): whatever
sizes came before, calls that repeat stop allocating, and the idle blocks stay
within the bound."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
K, M = 1 << 10, 1 << 20
BOUND = 128 * M

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("pool") / "libpool.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "clifft_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "block_pool_check.cpp"), "-o", str(so)], check=True, timeout=120)
    L = ctypes.CDLL(str(so))
    L.pool_new.argtypes = [ctypes.c_uint64]
    for f in (L.pool_allocs, L.pool_live, L.pool_kept):
        f.restype = ctypes.c_uint64
    L.pool_calls.restype = ctypes.c_int64
    L.pool_calls.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32]
    return L


def calls(lib, sizes, back=None):
    sizes = np.asarray(sizes, np.uint64)
    back = np.asarray(range(len(sizes)) if back is None else back, np.uint32)
    assert lib.pool_calls(sizes.ctypes.data, back.ctypes.data, len(sizes)) >= 0
    assert lib.pool_kept() <= BOUND


@pytest.mark.parametrize("before", [[64 * M], [64 * M, 64 * M], [32 * M] * 5, [64 * K], [2 * M, 16 * M, 64 * M]])
@pytest.mark.parametrize("steady", [[[64 * K]], [[64 * M], [64 * K]], [[256 * K], [8 * M], [64 * M]],
                                    [[64 * K, 64 * K]], [[64 * M], [64 * K, 64 * K, 64 * K]]])
def test_repeated_calls_stop_allocating(lib, before, steady):
    """`steady`: rounds of calls in turn, those of an inner list at once."""
    lib.pool_new(BOUND)
    calls(lib, before)
    for _ in range(8):
        for s in steady:
            calls(lib, s)
    n = lib.pool_allocs()
    for i in range(50):
        for s in steady:
            calls(lib, s, list(range(len(s)))[:: -1 if i % 2 else 1])
    assert lib.pool_allocs() == n


def test_random_calls_stay_within_the_bound(lib):
    lib.pool_new(BOUND)
    rng = np.random.default_rng(1)
    for _ in range(500):
        n = int(rng.integers(1, 9))
        calls(lib, [64 * K << int(e) for e in rng.integers(0, 12, n)], rng.permutation(n))
    assert lib.pool_live() * 64 * K <= BOUND
    calls(lib, [256 * M])  # one above the bound is not kept
    assert lib.pool_kept() <= BOUND
