"""A batch's plan survives its round trips: a tuning set again, read back and
set, chosen by tune() and given to a fresh batch, leaves the programs that
share states in their groups; whether they may is a field that is set and
taken back like the others, through Python and through the C entry points."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from test_gpu_batch import _device_batch, _snapshot, mixed_programs, mods  # noqa: F401

pytestmark = pytest.mark.gpu


def kinds(b):
    return [(g["kind"], g["programs"], g["items"], g["block"], g["lds_bytes"]) for g in b.groups()]


@pytest.fixture()
def batches(mods):  # noqa: F811
    made = []

    def make():
        progs, shots, seeds = mixed_programs(71, 13)
        b, bufs = _device_batch(mods[1], progs, shots)
        made.append((b, bufs))
        return b, bufs, seeds
    yield make
    for b, _ in made:
        b.close()


def records(b, bufs, seeds):
    import torch
    b.run(seeds)
    torch.cuda.synchronize()
    return _snapshot(bufs)


def same(a, b):
    for x, y in zip(a, b):
        assert all(np.array_equal(x[j], y[j]) for j in range(3))
        np.testing.assert_allclose(x[3], y[3], atol=1e-12, rtol=0)


def test_the_same_tuning_again(batches):
    from clifft_amd import _lib
    b, bufs, seeds = batches()
    plan, first = kinds(b), records(b, bufs, seeds)
    assert "shared" in {k[0] for k in plan}
    b.set_tuning(**b.tuning)
    assert kinds(b) == plan
    old = {f: v for f, v in b.tuning.items() if f != "shared"}  # as saved before there was such a field
    b.set_tuning(**old)
    assert kinds(b) == plan
    t = _lib.BatchTuning()
    assert _lib.lib().clifft_svm_batch_get_tuning(b.handle, ctypes.byref(t)) == 0
    assert _lib.lib().clifft_svm_batch_set_tuning(b.handle, ctypes.byref(t)) == 0
    assert kinds(b) == plan
    same(records(b, bufs, seeds), first)


def test_there_and_back(batches):
    b, bufs, seeds = batches()
    plan, first, tuning = kinds(b), records(b, bufs, seeds), b.tuning
    assert tuning["shared"] == 1
    b.set_tuning(lane_chunk=256)
    assert b.tuning == {**tuning, "lane_chunk": 256, "shared": 0} and "shared" not in {k[0] for k in kinds(b)}
    same(records(b, bufs, seeds), first)
    b.set_tuning(lane_chunk=128, shared=1)
    assert "shared" in {k[0] for k in kinds(b)}
    b.set_tuning(**tuning)
    assert kinds(b) == plan and b.tuning == tuning
    b.set_tuning(shared=0)
    assert "shared" not in {k[0] for k in kinds(b)}
    b.set_tuning(shared=1)
    assert kinds(b) == plan
    same(records(b, bufs, seeds), first)


def test_a_tuned_plan_for_a_fresh_batch(batches):
    b, bufs, seeds = batches()
    chosen = b.tune(sample_shots=8)
    assert chosen == b.tuning and chosen["shared"] == 1
    plan, first = kinds(b), records(b, bufs, seeds)
    c, cbufs, _ = batches()
    c.set_tuning(**chosen)
    assert kinds(c) == plan
    same(records(c, cbufs, seeds), first)


def test_refused(batches):
    from clifft_amd import _lib
    from clifft_amd._lib import SvmError
    b, _, _ = batches()
    plan = kinds(b)
    with pytest.raises(SvmError):
        b.set_tuning(shared=2)
    with pytest.raises(SvmError):
        b.set_tuning(global_threads=300, shared=0)
    assert kinds(b) == plan and b.tuning["shared"] == 1
    assert _lib.lib().clifft_svm_batch_get_shared(b.handle, None) != 0
    assert _lib.lib().clifft_svm_batch_set_plan(b.handle, None, 1) != 0
