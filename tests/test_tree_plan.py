"""The planner of the shared-state executor (clifft_amd/csrc/svm_tree_plan.h)
on the CPU: its tables, run one shot at a time by plain scalar code that
follows their documented meaning (tests/cpp/tree_plan_check.cpp), give the
oracle's records and expectation values shot for shot.  The programs cover
every opcode the planner accepts: random ones (noise, resets, U2/U4 nodes,
H, all measurement kinds, expectation values, frames that part the shots) and
compiled Clifford+T circuits with and without mid-circuit resets."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from clifft_amd.program import Op
from randprog import fanout_program, random_program

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXPANDS = (Op.EXPAND, Op.EXPAND_T, Op.EXPAND_T_DAG, Op.EXPAND_ROT)
MEASURES = (Op.MEAS_ACTIVE_DIAGONAL, Op.MEAS_ACTIVE_INTERFERE, Op.SWAP_MEAS_INTERFERE)

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("tree") / "libtree_plan.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "clifft_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "tree_plan_check.cpp"),
                    "-o", str(so)], check=True, timeout=120)
    L = ctypes.CDLL(str(so))
    L.tree_sample.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint64] + [ctypes.c_void_p] * 4
    return L


def ranks(p):
    k, out = 0, []
    for op in p.bytecode["opcode"]:
        out.append(k)
        k += int(op in EXPANDS) - int(op in MEASURES)
    return np.array(out, np.int32)


def check(lib, orc, p, shots, seed):
    kh, v = ranks(p), p.view()
    m, d, o, e = (np.zeros((shots, n), t) for n, t in ((p.num_measurements, np.uint8), (p.num_detectors, np.uint8),
                                                       (p.num_observables, np.uint8), (p.num_exp_vals, np.float64)))
    n = lib.tree_sample(ctypes.addressof(v), kh.ctypes.data, shots, seed, *(a.ctypes.data for a in (m, d, o, e)))
    if n < 0:
        return n
    rm, rd, ro, re, gone = orc.sample(p, shots, seed=seed, per_shot=True)
    m, d, o, e, rm, rd, ro, re = (a[gone == 0] for a in (m, d, o, e, rm, rd, ro, re))
    assert len(m) and np.array_equal(m, rm) and np.array_equal(d, rd) and np.array_equal(o, ro)
    np.testing.assert_allclose(e, re, atol=1e-12, rtol=0)
    return n


@pytest.mark.parametrize("seed", range(40))
def test_random_programs(lib, orc, seed):
    p = random_program(9000 + seed, num_qubits=(6, 9, 14, 70, 150)[seed % 5], peak=(1, 3, 5, 6, 9)[seed % 5],
                       length=(60, 160, 300)[seed % 3], noise=seed % 4 != 0, u_nodes=seed % 2 == 0)
    assert check(lib, orc, p, 24, seed) >= 0


@pytest.mark.parametrize("distance,rounds", [(3, 3), (5, 2), (7, 2)])
def test_memories(lib, orc, distance, rounds):
    """Noisy surface-code memories (17, 49 and 97 qubits), also post-selected
    on the first round's detectors (the surviving shots' rows)."""
    from clifft_amd.compiler import compile as ccompile
    from memory_circuit import memory_text
    p = ccompile(memory_text(distance, rounds, 0.004))
    assert check(lib, orc, p, 60, distance) >= 0
    first = np.flatnonzero(p.bytecode["opcode"] == Op.DETECTOR)[: (distance ** 2 - 1) // 2]
    p.bytecode["opcode"][first] = Op.POSTSELECT
    p.has_postselection = True
    assert check(lib, orc, p, 60, distance) >= 0


@pytest.mark.parametrize("peak", [1, 2, 5, 6, 7, 11])
def test_fanout_programs(lib, orc, peak):
    assert check(lib, orc, fanout_program(300 + peak, max(peak, 2), frames=True), 16, peak) > 0


@pytest.mark.parametrize("t,resets", [(3, 0), (6, 0), (9, 5), (12, 0), (12, 7)])
def test_clifford_t(lib, orc, t, resets):
    from clifft_amd import workloads as W
    from clifft_amd.compiler import compile as ccompile
    p = ccompile(W.random_clifford_t(n=16 + t, layers=24, t_count=t, seed=t, mr_every=resets, mr_count=3))
    assert check(lib, orc, p, 12, 77 + t) > 0


def test_refusals(lib, orc):
    """Rotation weights off the unit circle and records written twice go to
    the other executors."""
    from clifft_amd.program import build_program, make_array_rot, make_expand, make_meas
    twice = [make_meas(Op.MEAS_DORMANT_RANDOM, 0, 0), make_meas(Op.MEAS_DORMANT_STATIC, 0, 0)]
    assert check(lib, orc, build_program(twice, peak_rank=0, num_qubits=1, num_measurements=1), 2, 1) == -1
    p = build_program([make_expand(0), make_array_rot(0, 0.9, 0.1), make_meas(Op.MEAS_ACTIVE_DIAGONAL, 0, 0)],
                      peak_rank=1, num_qubits=1, num_measurements=1)
    assert check(lib, orc, p, 2, 1) == -1
