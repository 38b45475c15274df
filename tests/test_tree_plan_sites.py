"""A program that names a noise site twice is not given a shared-state plan
(clifft_amd/csrc/svm_tree_plan.h): the plan keeps one row of flipped bits a
channel, and which of the two instructions fires the site depends on the shot
where the sites do not come in ascending order."""

from __future__ import annotations

import shutil

import pytest

from clifft_amd.program import (Op, build_program, make_frame_h, make_meas, make_noise, make_noise_block)
from test_tree_plan import check, lib  # noqa: F401  (lib: the compiled planner)

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")

X = [[(1, 0, 0.7)], [(1, 0, 0.6)]]


def program(body):
    return build_program(body + [make_meas(Op.MEAS_DORMANT_STATIC, 0, 0)], peak_rank=0, num_qubits=1, num_measurements=1,
                         noise_sites=X)


@pytest.mark.parametrize("body", [
    [make_noise(1), make_frame_h(0), make_noise(0), make_noise(1)],  # site 1 fires after H only where site 0 did before it
    [make_noise_block(0, 2), make_frame_h(0), make_noise_block(1, 1)],
    [make_noise_block(1, 1), make_frame_h(0), make_noise_block(0, 2)]])
def test_a_site_named_twice(lib, orc, body):  # noqa: F811
    assert check(lib, orc, program(body), 400, 3) == -1


def test_sites_named_once_in_any_order(lib, orc):  # noqa: F811
    assert check(lib, orc, program([make_noise(1), make_frame_h(0), make_noise(0)]), 400, 3) == 0
    assert check(lib, orc, program([make_noise(0), make_frame_h(0), make_noise(1)]), 400, 3) == 0
