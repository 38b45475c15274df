"""Expectation values and gradients as sums of products on the device, where
a wavefront's split over parameters and vectors has edges.  Phases on one axis
add up, so products of X and Y probes have closed forms: the tolerances are
those of the adjoint tests (1e-12 for values; 1e-10 for gradients)."""

from __future__ import annotations

import numpy as np
import pytest

from clifft_amd import program as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grad():
    from clifft_amd import _lib, grad
    assert _lib.backend() == "hip:gfx950", _lib.backend()
    return grad


def axes_program(axes, extra):
    """One rotated expansion per axis, `extra` more rotations; probes X_a,
    Y_a of each axis and X on all axes."""
    bc = [P.make_expand_rot(a, 1.0, 0.0) for a in range(axes)]
    bc += [P.make_array_rot(i % axes, 1.0, 0.0) for i in range(extra)]
    masks = [(1 << a, 0, 0) for a in range(axes)] + [(1 << a, 1 << a, 1) for a in range(axes)] + [((1 << axes) - 1, 0, 0)]
    n = len(bc)
    bc += [P.make_exp_val(j, j) for j in range(len(masks))]
    p = P.build_program(bc, peak_rank=axes, num_qubits=axes, num_exp_vals=len(masks), exp_val_masks=masks)
    return p, np.arange(n), np.array([i % axes if i >= axes else i for i in range(n)])


@pytest.mark.parametrize("axes,extra,batch", [(1, 0, 1), (5, 0, 5), (9, 3, 2049), (16, 0, 67), (8, 58, 3), (14, 50, 2)])
def test_closed_form(grad, axes, extra, batch):
    print("CASE terms", axes, extra, batch, flush=True)
    p, instr, axis = axes_program(axes, extra)
    rng = np.random.default_rng(axes)
    sign = rng.choice([-1, 1], size=len(instr)).astype(np.int8)
    adj = grad.Adjoint(p, param_instr=instr, param_sign=sign)
    th, c = rng.uniform(-7, 7, (batch, len(instr))), rng.normal(size=2 * axes + 1)
    ev, g = adj.run(th, c)
    s = np.stack([(th * sign)[:, axis == a].sum(1) for a in range(axes)], 1)
    every = np.prod(np.cos(s), 1)
    np.testing.assert_allclose(ev, np.concatenate([np.cos(s), -np.sin(s), every[:, None]], 1), atol=1e-12, rtol=0)
    others = np.stack([np.prod(np.delete(np.cos(s), a, 1), 1) for a in range(axes)], 1)
    ds = -np.sin(s) * c[:axes] - np.cos(s) * c[axes:-1] - c[-1] * np.sin(s) * others
    np.testing.assert_allclose(g, ds[:, axis] * sign, atol=1e-10, rtol=0)
    only, none = adj.run(th, None, grads=False)
    assert none is None and np.array_equal(only, ev)


def test_angles_that_are_not_finite(grad):
    """The state's norm is then not a number: values 0, gradients nan, for
    that vector alone."""
    p, instr, _ = axes_program(7, 0)
    adj = grad.Adjoint(p, param_instr=instr, param_sign=np.ones(7, np.int8))
    th = np.full((3, 7), 0.3)
    clean = adj.run(th, np.ones(15))
    th[1, 2] = np.nan
    ev, g = adj.run(th, np.ones(15))
    assert np.all(ev[1] == 0) and np.all(np.isnan(g[1]))
    assert np.array_equal(ev[::2], clean[0][::2]) and np.array_equal(g[::2], clean[1][::2])
