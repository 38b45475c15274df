"""The shared-state executor's rules of dispatch (svm_tree_shape.h) on the CPU:
programs for which the choice was measured to matter, and the limits that
every shape has to keep."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from randprog import random_program
from test_tree_plan import ranks

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("shape") / "libshape.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "clifft_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "tree_shape_check.cpp"),
                    "-o", str(so)], check=True, timeout=120)
    L = ctypes.CDLL(str(so))
    L.shape.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_int,
                        ctypes.c_uint32, ctypes.c_void_p]
    return L


def shape(lib, p, shots, faults=0, mode=1, copies=0):
    """(threads, shots a team, entries, LDS bytes, in memory), or None on the
    per-shot executors"""
    out, kh, v = np.zeros(5, np.uint64), ranks(p), p.view()
    n = lib.shape(ctypes.addressof(v), kh.ctypes.data, shots, faults, CUS, mode, copies, out.ctypes.data)
    return tuple(int(x) for x in out) if n == 1 else None


def parting(peak, length, u_nodes=True):
    return random_program(190 + peak, num_qubits=peak + 10, peak=peak, length=length, u_nodes=u_nodes, exp_vals=False)


def with_resets(t, every, n=24, layers=40):
    """Random Clifford layers with t T gates; every few layers four qubits are
    measured and reset."""
    rng = np.random.default_rng(t)
    at = set(np.linspace(0, layers - 1, t).astype(int).tolist())
    out = [f"H {' '.join(map(str, range(n)))}"]
    for layer in range(layers):
        q = rng.permutation(n)
        out += [f"{('H', 'S', 'S_DAG')[rng.integers(3)]} {i}" for i in range(n)]
        out += [f"CX {q[i]} {q[i + 1]}" for i in range(0, n - 1, 2)]
        if layer in at:
            out.append(f"T {rng.integers(n)}")
        if (layer + 1) % every == 0:
            out.append("MR " + " ".join(map(str, rng.choice(n, 4, replace=False))))
    out.append("M " + " ".join(map(str, range(n))))
    return "\n".join(out)


@pytest.mark.parametrize("peak,length,u_nodes,shots", [
    (12, 400, False, 3000), (13, 400, True, 3000), (14, 400, True, 3000), (14, 400, True, 10000), (16, 400, True, 1000),
    (18, 400, True, 1000)])
def test_small_teams_are_not_filled_where_shots_part(lib, peak, length, u_nodes, shots):
    """64 threads with the most shots that fit were 1.6 to 2.8 times as slow as
    the best shape of these, and 1.07 to 1.7 times as slow as one shot a team."""
    threads, chunk = shape(lib, parting(peak, length, u_nodes), shots)[:2]
    assert threads >= 128 or chunk == 1 or chunk <= 4 and shots == 10000


@pytest.mark.parametrize("peak,length,few,many", [(9, 150, 100, 10000), (9, 400, 100, 10000), (10, 400, 300, 1000)])
def test_few_shots_of_many_passes(lib, peak, length, few, many):
    """A pass for every few instructions at peak 9 and 10: 0.81 to 0.95 times
    the per-shot executors' speed at a few hundred shots, 1.3 to 2.5 at more."""
    p = parting(peak, length)
    assert shape(lib, p, few) is None and shape(lib, p, few, mode=2) is not None
    assert shape(lib, p, many) is not None


@pytest.mark.parametrize("peak,length,u_nodes", [(8, 400, True), (9, 400, False), (10, 150, True), (11, 400, True)])
def test_few_shots_of_fewer_passes(lib, peak, length, u_nodes):
    assert all(shape(lib, parting(peak, length, u_nodes), s) is not None for s in (1, 100, 1000))


@pytest.mark.parametrize("t,layers", [(8, 40), (12, 40), (16, 40)])
def test_noiseless_programs_share(lib, t, layers):
    from clifft_amd import workloads as W
    from clifft_amd.compiler import compile as ccompile
    p = ccompile(W.random_clifford_t(n=24, layers=layers, t_count=t, seed=42))
    for shots in (1, 2000, 100000):
        assert shape(lib, p, shots) is not None


@pytest.mark.parametrize("t,resets,shots", [(11, 7, 5500), (14, 7, 3400), (14, 10, 11000), (17, 10, 1100)])
def test_resets_leave_no_compute_unit_idle(lib, t, resets, shots):
    """The memory's time is the same for many shapes: 64 shots a team (173
    teams) took 1.22 times the time of 4 a team for such a program."""
    from clifft_amd.compiler import compile as ccompile
    p = ccompile(with_resets(t, resets))
    assert p.peak_rank >= 8
    threads, chunk = shape(lib, p, shots)[:2]
    assert -(-shots // chunk) >= 256, (threads, chunk)


@pytest.mark.parametrize("peak", [1, 2, 3, 4, 5])
def test_many_shots_of_many_passes_run_on_lanes(lib, peak):
    """300 instructions, a pass for every six: 1.35 to 3.1 times as slow at
    300000 shots, as fast or faster at a few."""
    p = random_program(40 + peak, num_qubits=peak + 10, peak=peak, length=300, u_nodes=False, exp_vals=False)
    assert shape(lib, p, 300000) is None and shape(lib, p, 300000, mode=2) is not None
    assert shape(lib, p, 1) is not None


@pytest.mark.parametrize("distance,rounds", [(3, 3), (5, 5), (5, 25)])
def test_many_shots_of_memories_share(lib, distance, rounds):
    from clifft_amd.compiler import compile as ccompile
    from memory_circuit import memory_text
    p = ccompile(memory_text(distance, rounds, 0.002))
    assert all(shape(lib, p, s) is not None for s in (1, 5000, 200000))


@pytest.mark.parametrize("peak,shots", [(7, 1000), (8, 1000), (9, 1000), (10, 1000)])
def test_small_batches_use_the_whole_device(lib, peak, shots):
    """8 programs in one team each left 248 of 256 compute units idle: 1.4 to
    3.3 times as slow as the per-shot executors."""
    threads, chunk = shape(lib, parting(peak, 300), shots, copies=8)[:2]
    assert 8 * -(-shots // chunk) >= CUS
    assert shape(lib, parting(peak, 300), shots, copies=512)[1] > chunk


@pytest.mark.parametrize("peak,shots,copies,shared", [
    (3, 1000, 256, False), (3, 8000, 64, False),  # up to 1.8 times as slow
    (3, 100, 8, True), (6, 100, 8, True), (6, 8000, 64, True)])  # 1.3 to 4 times as fast
def test_low_ranks_in_batches(lib, peak, shots, copies, shared):
    p = parting(peak, 300, u_nodes=False)
    assert (shape(lib, p, shots, copies=copies) is not None) == shared
    assert shape(lib, p, shots, mode=2, copies=copies) is not None and shape(lib, p, shots, mode=0, copies=copies) is None


@pytest.mark.parametrize("distance", [3, 5])
def test_memories_share_in_batches(lib, distance):
    from clifft_amd.compiler import compile as ccompile
    from memory_circuit import memory_text
    p = ccompile(memory_text(distance, distance, 0.002))
    assert all(shape(lib, p, s, copies=n) is not None for s in (100, 10000, 1000000) for n in (1, 16, 512))


@pytest.mark.parametrize("seed", range(24))
def test_every_shape_keeps_the_limits(lib, seed):
    p = random_program(5000 + seed, num_qubits=(9, 20, 33, 90)[seed % 4], peak=(1, 6, 9, 14)[seed % 4],
                       length=(40, 200, 400)[seed % 3], u_nodes=seed % 2 == 0)
    for shots in (1, 3, 64, 1000, 1 << 20):
        for faults, copies in ((0, 0), (8, 0), (64, 0), (0, 1), (0, 500)):
            s = shape(lib, p, shots, faults, mode=2, copies=copies)
            if s is None:
                assert faults  # (the fault lists leave no room)
                continue
            threads, chunk, elems, lds, memory = s
            assert threads in (64, 128, 256, 512, 1024) and 1 <= chunk <= threads and lds <= 158 * 1024
            assert memory == (elems > 2048) and (chunk == 1 or elems <= max(1 << 18, 1 << p.peak_rank))
