"""The spill list taken by the tile kernel's last block (a workspace's first depositions,
before spills were seen) and by the kernel after it (the depositions that follow):
displacements whose bound passes the largest halo, with and without particles
that do move so far, in each tile size.  Against the oracle, relative L2 <= 1e-12 as
the other depositions; the four calls in a row take both ways."""

import types

import numpy as np
import pytest

from gpu_helpers import Workspace, dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,c", [(129, 2), (193, 3), (241, 3), (433, 3), (433, 2), (721, 3)])
@pytest.mark.parametrize("cells,one", [(6.3, True), (7.9, True), (7.9, False), (14., False)])
def test_spill_list(oracle, N, c, cells, one):
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=16, plasma_coarseness=c,
        plasma_fineness=2)
    h = cfg.grid_step_size
    w = Workspace(oracle, cfg)
    rng = np.random.default_rng(N)
    off = [h * rng.uniform(-1, 1, w.shape) for _ in range(2)]
    if one:   # one coarse particle beyond, its fine ones partly
        off[0][w.shape[0] // 2, w.shape[1] // 3] = cells * h
    else:
        off = [cells * o for o in off]
    p = [.3 * rng.uniform(-1, 1, w.shape) for _ in range(3)]
    want = oracle.deposit(cfg, w.const.ro_initial, *off, w.const.m, w.const.q, *p, w.vp)
    for call in range(4):
        say(f"spill list N={N} c={c} {cells} cells{' (one)' if one else ''}, call {call}")
        got = w.deposit(*map(dev, off), [dev(a) for a in p])
        for name, g, o in zip(("ro", "jx", "jy", "jz"), got, want):
            assert rel_l2(host(g), o) < 1e-12, (call, name)
    assert w.faults() == 0
    w.close()
