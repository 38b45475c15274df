"""The executors behind the shared-state one and behind the sums of products.

Every program here is one that the newer planner refuses, by a change that
leaves its results as they are: its first detector written twice, or a U2 node
on an axis that is not active.  So the calls run one shot per lane, wavefront
team or workgroup team (LDS and global amplitudes, frames of one and of more
words, forced records, forced faults, post-selection), and the adjoint sweeps
over LDS and global states; records are compared with the oracle's bit for
bit, expectation values to 1e-12, log-probabilities and gradients to 1e-10, as
in the tests of the same calls."""

from __future__ import annotations

import ctypes
import shutil

import numpy as np
import pytest

from clifft_amd.compiler import compile as ccompile
from clifft_amd.program import U2_DTYPE, Op, make_array_rot, make_array_u2
from gradprog import oracle_exp_vals, oracle_param_shift, rz_circuit
from memory_circuit import memory_text
from randprog import random_measure_only_program, random_program
from test_terms import lib as terms_lib, run as terms_run  # noqa: F401
from test_tree_plan import lib as plan_lib, ranks  # noqa: F401

needs_compiler = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


def refused(p):
    """`p` with its first detector written twice; where it has none, with a
    weight off the unit circle on its first axis."""
    q = p.copy()
    at = np.flatnonzero(q.bytecode["opcode"] == Op.DETECTOR)
    if len(at):
        q.bytecode = np.insert(q.bytecode, at[0] + 1, q.bytecode[at[0]])
    else:
        first = np.flatnonzero(np.isin(q.bytecode["opcode"], (Op.EXPAND, Op.EXPAND_T, Op.EXPAND_T_DAG, Op.EXPAND_ROT)))[0]
        q.bytecode = np.insert(q.bytecode, first + 1, np.array([make_array_rot(0, 0.8, 0.3)], q.bytecode.dtype))
    return q


def idle_node(p):
    """`p` with a U2 node on an axis that is never active, first of all."""
    assert p.num_qubits > p.peak_rank and not len(p.u2_nodes)
    q = p.copy()
    q.u2_nodes = np.zeros(1, U2_DTYPE)
    q.u2_nodes["matrices"] = [1, 0, 0, 1]
    q.u2_nodes["gamma"] = 1.0
    q.bytecode = np.insert(q.bytecode, 0, np.array([make_array_u2(p.num_qubits - 1, 0)], q.bytecode.dtype))
    q.param_instr = np.asarray(p.param_instr) + 1
    return q


def sampled(nq, peak, **kw):
    return random_program(2600 + peak + nq, num_qubits=nq, peak=peak, length=150 + 10 * peak, **kw)


def memory(distance, post=False):
    p = ccompile(memory_text(distance, 3, 0.01))
    if post:
        first = np.flatnonzero(p.bytecode["opcode"] == Op.DETECTOR)[: (distance ** 2 - 1) // 2]
        p.bytecode["opcode"][first] = Op.POSTSELECT
        p.has_postselection = True
    return p


# lanes, wavefront teams (LDS), workgroup teams (LDS), global amplitudes; wide frames
SAMPLED = [(10, 2, 300), (40, 6, 300), (16, 8, 300), (20, 10, 700), (24, 12, 150), (24, 13, 100), (24, 14, 1100),
           (30, 15, 600), (24, 16, 64), (26, 18, 8), (100, 3, 300), (130, 9, 200), (100, 14, 60)]
FORCED = [(12, 7), (16, 10), (18, 12), (20, 14), (80, 8)]


@needs_compiler
@pytest.mark.parametrize("make", [lambda: sampled(20, 10), lambda: sampled(100, 3), lambda: memory(3), lambda: memory(7, True),
                                  lambda: random_measure_only_program(7, num_qubits=12, peak=7, length=120)])
def test_no_shared_plan(plan_lib, make):  # noqa: F811
    for p, planned in ((make(), True), (refused(make()), False)):
        out, v, kh = [np.zeros(1 << 16, np.uint8) for _ in range(4)], p.view(), ranks(p)
        n = plan_lib.tree_sample(ctypes.addressof(v), kh.ctypes.data, 1, 1, *(a.ctypes.data for a in out))
        assert (n >= 0) == planned


def gradient_program(n, params, seed):
    build, coeffs = rz_circuit(n=n, layers=4, n_params=params, seed=seed, repeat_qubits=False)
    th = np.random.default_rng(seed).uniform(0, 2 * np.pi, (2, params))
    return idle_node(ccompile(build(th[0]), keep_rotations=True, fusion=False)), coeffs, th


@needs_compiler
def test_no_sums(terms_lib):  # noqa: F811
    p, _, th = gradient_program(8, 6, 2)
    assert terms_run(terms_lib, p, p.param_instr, np.asarray(p.param_sign) * th[0])[0] == -1


@pytest.fixture(scope="module")
def svm():
    import clifft_amd.svm as svm
    from clifft_amd import _lib
    assert _lib.backend() == "hip:gfx950", _lib.backend()
    return svm


def same(res, ref):
    for got, want in zip((res.measurements, res.detectors, res.observables), ref):
        assert np.array_equal(got, want)
    np.testing.assert_allclose(res.exp_vals, ref[3], atol=1e-12, rtol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,peak,shots", SAMPLED)
def test_sampling(svm, orc, nq, peak, shots):
    print("CASE fallback", nq, peak, shots, flush=True)
    p = refused(sampled(nq, peak))
    ref = orc.sample(p, shots, seed=peak, per_shot=True)
    same(svm.sample(p, shots, seed=peak), ref)
    packed = svm.sample(p, shots, seed=peak, packed=True)
    assert np.array_equal(packed.measurements, np.packbits(ref[0], axis=1, bitorder="little"))


@pytest.mark.gpu
@pytest.mark.parametrize("nq,peak", FORCED)
def test_forced_records(svm, orc, nq, peak):
    print("CASE fallback forced", nq, peak, flush=True)
    p = refused(random_measure_only_program(peak, num_qubits=nq, peak=peak, length=120))
    recs, *_ = orc.sample(p, 40, seed=3)
    flipped = recs.copy()
    flipped[::3, np.random.default_rng(peak).integers(0, p.num_measurements)] ^= 1
    recs = np.concatenate([recs, flipped])
    got, ref = svm.record_probabilities(p, recs), orc.record_log_probs(p.forced(), recs)
    assert np.array_equal(got < -1e300, ref < -1e300)
    np.testing.assert_allclose(got[ref > -1e300], ref[ref > -1e300], atol=1e-10, rtol=1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("make,k", [(lambda: memory(3), 2), (lambda: memory(5), 4), (lambda: memory(7), 4),
                                    (lambda: sampled(16, 9, readout=True), 3), (lambda: sampled(20, 14, readout=True), 1)])
def test_forced_faults(svm, orc, make, k):
    p = refused(make())
    print("CASE fallback faults", p.num_qubits, p.peak_rank, k, flush=True)
    same(svm.sample_k(p, 64, k, seed=17), orc.sample_k(p, 64, k, seed=17))


@pytest.mark.gpu
@pytest.mark.parametrize("distance", [3, 7])
def test_survivors(svm, orc, distance):
    print("CASE fallback survivors", distance, flush=True)
    p = refused(memory(distance, post=True))
    _, _, o, _, gone = orc.sample(p, 300, seed=9, per_shot=True)
    r = svm.sample_survivors(p, 300, seed=9)
    o = o[gone == 0]
    assert 0 < r.passed_shots == len(o) < 300 and r.logical_errors == int(o.any(1).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("n,params,seed", [(8, 6, 2), (10, 8, 4), (12, 12, 7), (15, 14, 9)])
def test_adjoint_sweeps(orc, n, params, seed):
    """Peak 2 to 9, LDS states."""
    from clifft_amd import grad
    p, coeffs, th = gradient_program(n, params, seed)
    print("CASE fallback sweeps", n, params, p.peak_rank, flush=True)
    ev, g = grad.Adjoint(p).run(th, coeffs)
    for b in range(len(th)):
        np.testing.assert_allclose(ev[b], oracle_exp_vals(orc, p, th[b]), atol=1e-12, rtol=0)
        np.testing.assert_allclose(g[b], oracle_param_shift(orc, p, th[b], coeffs), atol=1e-10, rtol=0)
    assert np.abs(g).max() > 1e-3


@pytest.mark.gpu
def test_adjoint_sweeps_in_memory(orc):
    """The 24-qubit, 16-parameter, 32-probe workload, peak 16."""
    from clifft_amd import grad
    from clifft_amd import workloads as W
    print("CASE fallback sweeps 16", flush=True)
    build, coeffs, _ = W.rz_exp_val()
    th = np.random.default_rng(42).uniform(0, 2 * np.pi, (3, 16))
    plain = ccompile(build(th[0]), keep_rotations=True)
    p = idle_node(plain)
    ev, g = grad.Adjoint(p).run(th, coeffs)
    np.testing.assert_allclose(ev[0], oracle_exp_vals(orc, p, th[0]), atol=1e-12, rtol=0)
    np.testing.assert_allclose(g[0], oracle_param_shift(orc, p, th[0], coeffs), atol=1e-10, rtol=0)
    ev2, g2 = grad.Adjoint(plain).run(th, coeffs)  # the sums of products
    np.testing.assert_allclose(ev, ev2, atol=1e-12, rtol=0)
    np.testing.assert_allclose(g, g2, atol=1e-10, rtol=0)


@pytest.mark.gpu
def test_a_probe_that_vanishes(orc):
    """The term planner gives up on it (test_terms_bound.py): the sweeps' values
    and derivatives are 0."""
    from clifft_amd import grad
    from test_terms_bound import vanishing
    p, slots, angles = vanishing(38)
    sign = np.ones(len(slots), np.int8)
    ev, g = grad.Adjoint(p, param_instr=np.array(slots), param_sign=sign).run(np.stack([angles, angles + 0.7]), np.ones(1))
    np.testing.assert_allclose(ev, 0.0, atol=1e-12, rtol=0)
    np.testing.assert_allclose(g, 0.0, atol=1e-10, rtol=0)
