"""Gradients as sums of products against the adjoint sweeps over the state,
for the same program and weights that are not finite: the twin holds a U2
node on an axis that is not active, which changes nothing and which only the
sweeps take.  A weight that is not a number, or infinite, leaves no derivative
by an angle that the state already holds at its probe, whether or not the
probe depends on it; a probe that is 0 for its X on an axis that is not
active counts for nothing, and angles that come later keep theirs."""

from __future__ import annotations

import numpy as np
import pytest

from clifft_amd import program as P
from clifft_amd.program import U2_DTYPE

pytestmark = pytest.mark.gpu

# X0; Z0 X1 (0, and so are its derivatives); X3 (not active); X0 after H; Y2
MASKS = [(1, 0, 0), (2, 1, 0), (8, 0, 0), (1, 0, 1), (4, 4, 0)]


def twins():
    """(program, its twin with the U2 node, their parameters' instructions)"""
    rot = (np.cos(0.4), np.sin(0.4))
    bc = [P.make_expand_rot(0, *rot), P.make_exp_val(0, 0), P.make_expand_rot(1, *rot), P.make_array_rot(5, *rot),
          P.make_exp_val(1, 1), P.make_exp_val(2, 2), P.make_array_h(0), P.make_array_rot(0, *rot), P.make_exp_val(3, 3),
          P.make_expand_rot(2, *rot), P.make_exp_val(4, 4)]
    node = np.zeros(1, U2_DTYPE)
    node["matrices"] = [1, 0, 0, 1]
    node["gamma"] = 1.0
    kw = dict(peak_rank=3, num_qubits=6, num_exp_vals=len(MASKS), exp_val_masks=MASKS)
    return (P.build_program(bc, **kw), P.build_program([P.make_array_u2(4, 0)] + bc, u2_nodes=node, **kw),
            np.array([0, 2, 3, 7, 9]))


@pytest.mark.parametrize("probe", range(len(MASKS)))
@pytest.mark.parametrize("weight", [np.nan, np.inf, -np.inf, 0.0])
def test_against_the_sweeps(probe, weight):
    from clifft_amd import grad
    print("CASE weights", probe, weight, flush=True)
    one, other, at = twins()
    sign = np.array([1, -1, 1, 1, -1], np.int8)
    th = np.random.default_rng(3).uniform(-3, 3, (5, 5))
    c = np.array([0.7, -1.2, 0.4, 0.9, 1.5])
    c[probe] = weight
    ev, g = grad.Adjoint(one, param_instr=at, param_sign=sign).run(th, c)
    ev2, g2 = grad.Adjoint(other, param_instr=at + 1, param_sign=sign).run(th, c)
    np.testing.assert_allclose(ev, ev2, atol=1e-12, rtol=0)
    np.testing.assert_allclose(g, g2, atol=1e-12, rtol=0, equal_nan=True)
    if not np.isfinite(weight):
        held = {0: [0], 1: [0, 1], 2: [], 3: [0, 1, 3], 4: [0, 1, 3, 4]}[probe]
        assert np.array_equal(np.isnan(g), np.isin(np.arange(5), held)[None].repeat(5, 0))


@pytest.mark.parametrize("angle", range(5))
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_angles_against_the_sweeps(angle, value):
    from clifft_amd import grad
    print("CASE angles", angle, value, flush=True)
    one, other, at = twins()
    sign = np.array([1, -1, 1, 1, -1], np.int8)
    th = np.random.default_rng(3).uniform(-3, 3, (5, 5))
    th[2, angle] = value
    c = np.array([0.7, -1.2, 0.4, 0.9, 1.5])
    ev, g = grad.Adjoint(one, param_instr=at, param_sign=sign).run(th, c)
    ev2, g2 = grad.Adjoint(other, param_instr=at + 1, param_sign=sign).run(th, c)
    np.testing.assert_allclose(ev, ev2, atol=1e-12, rtol=0)
    np.testing.assert_allclose(g, g2, atol=1e-12, rtol=0, equal_nan=True)
