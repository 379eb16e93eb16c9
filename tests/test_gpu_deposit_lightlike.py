"""Massless particles along the axis: gamma - pz is exactly 0, and the charge q / 0 is
the infinity that the reference's division gives (lcode.py:651-655), in every form of
the tile kernel (8-, 16- and 24-cell tiles, staged or not, one round and several):
the same cells infinite, with the same sign, and the same cells NaN as the oracle's."""

import types

import numpy as np
import pytest

from gpu_helpers import Workspace, dev, host, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,c", [(65, 2), (217, 2), (217, 1), (433, 3), (433, 2), (721, 3)])
@pytest.mark.parametrize("charge", [-1, 1])
def test_zero_denominator(oracle, N, c, charge):
    say(f"deposit of massless particles N={N} c={c} charge {charge}")
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=c,
        plasma_fineness=2)
    w = Workspace(oracle, cfg)
    rng = np.random.default_rng(N)
    off = [.7 * cfg.grid_step_size * rng.uniform(-1, 1, w.shape) for _ in range(2)]
    w.m.zero_()
    w.q.abs_().mul_(charge)
    zero, pz = np.zeros(w.shape), rng.uniform(.5, 2, w.shape)
    p = [zero, zero, pz]
    with np.errstate(divide="ignore", invalid="ignore"):
        want = oracle.deposit(cfg, w.const.ro_initial, *off, host(w.m), host(w.q), *p, w.vp)
    got = [host(g) for g in w.deposit(*map(dev, off), [dev(a) for a in p])]
    for name, g, o in zip(("ro", "jx", "jy", "jz"), got, want):
        assert np.array_equal(np.isnan(g), np.isnan(o)), name
        inf = np.isinf(o)
        assert np.array_equal(np.isinf(g), inf) and np.array_equal(g[inf], o[inf]), name
    assert np.isinf(want[0]).any() and np.isnan(want[1]).any()
    w.close()
