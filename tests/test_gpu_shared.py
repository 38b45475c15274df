"""The shared-state executor against the oracle where its teams, rows and
node tables have edges: one shot, shots around a wavefront and a chunk,
records that end inside a byte, ranks around one wavefront's pairs (6, 7, 8),
frames of more than one word (which always run there), post-selection, fault
lists of no and of many faults, forced records.  Records are compared bit for
bit, expectation values to the 1e-12 of the other executors' tests."""

from __future__ import annotations

import numpy as np
import pytest

from clifft_amd.compiler import compile as ccompile
from clifft_amd.program import Op
from memory_circuit import memory_text
from randprog import random_program

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("peak,shots", [(1, 1), (2, 63), (5, 64), (6, 65), (7, 257), (8, 1000), (11, 130)])
def test_random_programs(svm, orc, peak, shots):
    print("CASE shared", peak, shots, flush=True)
    p = random_program(7100 + peak, num_qubits=70, peak=peak, length=260, u_nodes=peak % 2 == 0, wide_lists=peak > 4)
    ref = orc.sample(p, shots, seed=peak)
    same(svm.sample(p, shots, seed=peak), ref)
    packed = svm.sample(p, shots, seed=peak, packed=True)
    for got, want in zip((packed.measurements, packed.detectors, packed.observables), ref):
        assert np.array_equal(got, np.packbits(want, axis=1, bitorder="little"))


@pytest.mark.parametrize("distance,k", [(3, 0), (3, 20), (5, 4), (7, 64)])
def test_memory_faults(svm, orc, distance, k):
    print("CASE shared faults", distance, k, flush=True)
    p = ccompile(memory_text(distance, 2, 0.002))
    same(svm.sample_k(p, 150, k, seed=5), orc.sample_k(p, 150, k, seed=5))


@pytest.mark.parametrize("distance", [3, 7])
def test_memory_post_selection(svm, orc, distance):
    print("CASE shared post-selection", distance, flush=True)
    p = ccompile(memory_text(distance, 3, 0.01))
    first = np.flatnonzero(p.bytecode["opcode"] == Op.DETECTOR)[: (distance ** 2 - 1) // 2]
    p.bytecode["opcode"][first] = Op.POSTSELECT
    p.has_postselection = True
    m, d, o, _, gone = orc.sample(p, 300, seed=9)
    keep = gone == 0
    res = svm.sample_survivors(p, 300, seed=9, keep_records=True)
    assert res.passed_shots == keep.sum()
    for got, want in zip((res.measurements, res.detectors, res.observables), (m, d, o)):
        assert np.array_equal(got, want[keep])


@pytest.mark.parametrize("n,t", [(66, 1), (70, 7), (70, 10)])
def test_forced_records(svm, orc, n, t):
    """Sampled records and ones with a flipped bit (some unreachable)."""
    from clifft_amd import workloads as W
    print("CASE shared forced", n, t, flush=True)
    p = ccompile(W.random_clifford_t(n=n, layers=12, t_count=t, seed=t))
    rec = svm.sample(p, 40, seed=3).measurements
    flipped = rec.copy()
    flipped[np.arange(40), np.arange(40) % n] ^= 1
    rec = np.concatenate([rec, flipped])
    ref = orc.record_log_probs(p.forced(), rec)
    np.testing.assert_allclose(svm.record_probabilities(p, rec), ref, atol=1e-9, rtol=0)


@pytest.mark.parametrize("n", [8, 9, 63, 64, 65, 128, 130])
def test_row_widths(svm, orc, n):
    """Rows that end at, before and behind the words and bytes they are
    spread by; the last row's end is the array's."""
    print("CASE shared rows", n, flush=True)
    q = " ".join(map(str, range(n)))
    p = ccompile(f"H {q}\nM {q}")
    for shots in (1, 3, 64, 130):
        ref = orc.sample(p, shots, seed=n)[0]
        assert np.array_equal(svm.sample(p, shots, seed=n).measurements, ref)
        packed = svm.sample(p, shots, seed=n, packed=True).measurements
        assert np.array_equal(packed, np.packbits(ref, axis=1, bitorder="little"))
