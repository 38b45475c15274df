"""Expectation values as sums of products (clifft_amd/csrc/svm_terms.h) on the
CPU against the oracle's state, over every operation the planner accepts, in
random order; its derivatives against central differences of the same sums;
its refusals."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from clifft_amd import program as P
from clifft_amd.program import Op
from gradprog import oracle_exp_vals, rz_circuit

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXPANDS = (Op.EXPAND, Op.EXPAND_T, Op.EXPAND_T_DAG, Op.EXPAND_ROT)

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("terms") / "libterms.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "clifft_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "terms_check.cpp"),
                    "-o", str(so)], check=True, timeout=120)
    L = ctypes.CDLL(str(so))
    L.terms_eval.restype = ctypes.c_int64
    L.terms_eval.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_uint32, ctypes.c_uint64] + [ctypes.c_void_p] * 3
    return L


def run(lib, p, slots, angles, limit=1 << 20):
    rank = np.concatenate([[0], np.cumsum([int(o in EXPANDS) for o in p.bytecode["opcode"]])]).astype(np.int32)
    slot_of = np.full(len(p.bytecode), -1, np.int32)
    slot_of[list(slots)] = np.arange(len(slots))
    v, np_ = p.view(), len(slots)
    angles = np.ascontiguousarray(angles, np.float64)
    ev, grad = np.zeros(p.num_exp_vals), np.zeros((p.num_exp_vals, max(np_, 1)))
    n = lib.terms_eval(ctypes.addressof(v), rank.ctypes.data, slot_of.ctypes.data, np_, limit, angles.ctypes.data,
                       ev.ctypes.data, grad.ctypes.data)
    return n, ev, grad


def rotating_program(seed, peak, length):
    """Random expansions, Clifford operations and phases (some of them
    parameters), probes in between and at the end; (program, slots, angles)."""
    rng = np.random.default_rng(seed)
    n, k, bc, slots, angles, masks = peak + 2, 0, [], [], [], []

    def rot(make):
        a = rng.uniform(-4, 4)
        if rng.random() < 0.7:
            slots.append(len(bc))
            angles.append(a)
        return make(k if make is P.make_expand_rot else int(rng.integers(0, k)), np.cos(a), np.sin(a))

    def probe(low):
        x, z = (int(rng.integers(0, 1 << (k if low else n))) if k or not low else 0 for _ in range(2))
        masks.append((x, z, int(rng.integers(0, 2))))
        return P.make_exp_val(len(masks) - 1, len(masks) - 1)

    while len(bc) < length:
        r = rng.integers(0, 16)
        if k < peak and (k < 2 or r == 0):
            e = rng.integers(0, 6)
            bc.append((P.make_expand, P.make_expand_t, P.make_expand_t_dag)[e](k) if e < 3 else rot(P.make_expand_rot))
            k += 1
            continue
        a, b = (int(q) for q in rng.choice(k, 2, replace=False)) if k > 1 else (0, 0)
        m = int(rng.integers(0, 1 << k))
        one = {1: P.make_array_h, 2: P.make_array_s, 3: P.make_array_s_dag, 9: P.make_frame_h, 10: P.make_array_h}
        two = {4: P.make_array_cnot, 5: P.make_array_cz, 6: P.make_array_swap}
        if r in one:
            bc.append(one[r](a))
        elif r in two and k > 1:
            bc.append(two[r](a, b))
        elif r == 7:
            bc.append(P.make_array_multi_cnot(a, m & ~(1 << a)))
        elif r == 8:
            bc.append(P.make_array_multi_cz(a, m))
        elif r == 11 and rng.random() < 0.4:
            bc.append((P.make_array_t, P.make_array_t_dag)[m & 1](a))
        elif r == 12 and rng.random() < 0.6:
            bc.append(rot(P.make_array_rot))
        elif r == 13:
            bc.append(probe(rng.random() < 0.8))
    for _ in range(6):
        bc.append(probe(True))
    p = P.build_program(bc, peak_rank=peak, num_qubits=n, num_exp_vals=len(masks), exp_val_masks=masks)
    return p, slots, np.array(angles)


@pytest.mark.parametrize("seed", range(30))
def test_against_the_state(lib, orc, seed):
    """1e-12: the tolerance of the other expectation-value tests (rounding
    only); central differences of a trigonometric polynomial of degree 1 in
    each angle, h = 1e-5: h^2 / 6 + eps / h < 1e-9."""
    p, slots, angles = rotating_program(seed, 1 + seed % 7, 30 + 2 * seed)
    n, ev, grad = run(lib, p, slots, angles)
    assert n >= 0
    np.testing.assert_allclose(ev, orc.sample(p, 1, seed=0)[3][0], atol=1e-12, rtol=0)
    for i in range(len(slots)):
        h = np.zeros(len(slots))
        h[i] = 1e-5
        d = (run(lib, p, slots, angles + h)[1] - run(lib, p, slots, angles - h)[1]) / 2e-5
        np.testing.assert_allclose(grad[:, i], d, atol=1e-9, rtol=0)


def test_compiled_circuit(lib, orc):
    from clifft_amd.compiler import compile as ccompile
    build, _ = rz_circuit(n=9, layers=4, n_params=9, seed=6, repeat_qubits=False)
    th = np.random.default_rng(1).uniform(0, 6, 9)
    p = ccompile(build(th), keep_rotations=True, fusion=False)
    n, ev, _ = run(lib, p, p.param_instr, np.asarray(p.param_sign) * th)
    assert n > 0
    np.testing.assert_allclose(ev, oracle_exp_vals(orc, p, th), atol=1e-12, rtol=0)


def test_refusals(lib):
    z = [(1, 0, 0)]
    ok = [P.make_expand(0), P.make_array_t(0), P.make_exp_val(0, 0)]
    make = lambda bc, n=1: P.build_program(bc, peak_rank=1, num_qubits=1, num_exp_vals=n, exp_val_masks=z)  # noqa: E731
    assert run(lib, make(ok), [], [])[0] == 1
    assert run(lib, make(ok), [], [], limit=0)[0] == -1
    assert run(lib, make(ok, 2), [], [])[0] == -1  # an output never written
    assert run(lib, make(ok + [P.make_exp_val(0, 0)]), [], [])[0] == -1  # one written twice
    assert run(lib, make([P.make_expand(0), P.make_array_rot(0, 0.9, 0.1)] + ok[2:]), [], [])[0] == -1
    many = [P.make_expand(0)] + [P.make_array_rot(0, 1.0, 0.0)] * 65 + ok[2:]
    assert run(lib, make(many), range(1, 66), np.zeros(65))[0] == -1
