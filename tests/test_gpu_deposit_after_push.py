"""lcode_deposit in a workspace whose pushes met other states, through the C ABI: a
push of a state with a NaN must not reach the deposition of a finite one (which
is the oracle's, relative L2 <= 1e-12), and deposited itself it spoils the tiles
around its particle alone.  Both orders of the workspace's slots."""

import types

import numpy as np
import pytest

from gpu_helpers import Workspace, dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


def _cfg(N, c, f):
    return types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=c,
        plasma_fineness=f)


@pytest.mark.parametrize("N,c,f", [(129, 2, 2), (217, 2, 2), (433, 3, 2)])
@pytest.mark.parametrize("before", [0, 1])
def test_push_mark_stays_out_of_other_depositions(oracle, N, c, f, before):
    say(f"deposit after a non-finite push N={N}, {before} depositions before")
    cfg = _cfg(N, c, f)
    w = Workspace(oracle, cfg)
    rng = np.random.default_rng(5)
    h = cfg.grid_step_size
    good = [.4 * h * rng.uniform(-1, 1, w.shape) for _ in range(2)]
    p = [.1 * rng.uniform(-1, 1, w.shape) for _ in range(3)]
    want = oracle.deposit(cfg, w.const.ro_initial, *good, w.const.m, w.const.q, *p, w.vp)
    dgood, dp = [dev(a) for a in good], [dev(a) for a in p]
    mid = w.shape[0] // 2
    bad = [t.clone() for t in dgood]
    bad[0][mid, mid] = float("nan")
    for _ in range(before):
        w.deposit(*dgood, dp)
    pushed = w.push(*bad, dp)
    for _ in range(2):
        for name, g, o in zip(("ro", "jx", "jy", "jz"), w.deposit(*dgood, dp), want):
            assert rel_l2(host(g), o) < 1e-12, name
    # the push's own result: the tiles around its particle
    for g in w.deposit(pushed[0], pushed[1], pushed[2:]):
        nan = np.isnan(host(g))
        assert nan.any() and nan.mean() < .1
    w.close()
