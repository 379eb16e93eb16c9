"""Fine particles at rest whose grid points lie on the edges of cells (the caller's own
fine grid; make_plasma's points lie inside): a point's cell, found from x / h or from
x (1 / h), may differ by one there, and must not count as a displacement.  Against
the oracle, relative L2 <= 1e-12 as the other depositions (the weights are
continuous across an edge)."""

import types

import numpy as np
import pytest

from gpu_helpers import Workspace, dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [65, 129, 217, 433, 721])
def test_points_on_cell_edges_at_rest(oracle, N):
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=3,
        plasma_fineness=2)
    h = cfg.grid_step_size
    w = Workspace(oracle, cfg)
    nf = len(w.vp.fine_grid)
    w.vp.fine_grid = (np.arange(nf) - nf // 2) / 2 * h
    x = w.vp.fine_grid
    say(f"points on cell edges N={N}",
        int((np.floor(x / h + .5) != np.floor(x * (1 / h) + .5)).sum()), "ambiguous")
    w.keep[2].copy_(dev(x))
    p = [.1 * np.random.default_rng(N).uniform(-1, 1, w.shape) for _ in range(3)]
    zero = np.zeros(w.shape)
    want = oracle.deposit(cfg, w.const.ro_initial, zero, zero, w.const.m, w.const.q, *p, w.vp)
    for noalloc in (False, True):
        got = w.deposit(dev(zero), dev(zero), [dev(a) for a in p], noalloc=noalloc)
        for name, g, o in zip(("ro", "jx", "jy", "jz"), got, want):
            assert rel_l2(host(g), o) < 1e-12, (noalloc, name)
    assert w.faults() == 0
    w.close()
