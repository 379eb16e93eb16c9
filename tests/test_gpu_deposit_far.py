"""A coarse particle finite but far beyond the grid, with plasma next to the grid's
edge: the deposition treats what interpolates from it as it treats a non-finite
particle (the same tiles NaN, every other cell the same up to the order of FP64 sums,
relative L2 <= 1e-12; flagged, not counted as a clamped lookup), and does not
clamp it to the edge.  10^9 cells fit an int cell index, 10^12 do not."""

import types

import numpy as np
import pytest

from gpu_helpers import Workspace, dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [65, 217, 433])
@pytest.mark.parametrize("cells", [1e9, 1e12])
@pytest.mark.parametrize("noalloc", [False, True])
def test_far_particle_at_the_edge(oracle, N, cells, noalloc):
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=3, plasma_coarseness=2,
        plasma_fineness=2)
    h = cfg.grid_step_size
    w = Workspace(oracle, cfg)
    nc = w.shape[0]
    rng = np.random.default_rng(N)
    p = [dev(.1 * rng.uniform(-1, 1, w.shape)) for _ in range(3)]
    for sign in (1, -1):
        for axis, (i, j) in ((0, (0, nc // 2)), (0, (nc - 1, nc // 2)), (1, (nc // 2, 0)),
                             (1, (nc // 2, nc - 1))):
            say(f"far particle N={N} {sign * cells:g} cells, axis {axis} at {i}, {j}")
            off = [.3 * h * rng.uniform(-1, 1, w.shape) for _ in range(2)]
            off[axis][i, j] = sign * cells * h
            got = [host(g) for g in w.deposit(*map(dev, off), p, noalloc=noalloc)]
            off[axis][i, j] = np.nan
            want = [host(g) for g in w.deposit(*map(dev, off), p, noalloc=noalloc)]
            for g, o in zip(got, want):
                nan = np.isnan(o)
                assert nan.any() and not nan.all()
                assert np.array_equal(np.isnan(g), nan)
                assert rel_l2(g[~nan], o[~nan]) < 1e-12
    if not noalloc:
        assert w.nonfinite() == 1 and w.faults() == 0
    w.close()
