"""The deposition's tiles against the oracle at the sizes where their shape
changes (8-, 16- and 24-cell tiles, one and several rounds of blocks), with
every staging form (coarseness 1 reads the coarse particles unstaged), group
size, halo (displacements from rest to beyond the largest halo, which takes the
spill list) and with uniform and mixed masses and charges; and a deposition on
its own with inputs that its displacement bound must not trust.  FP64 sums in
another order: relative L2 <= 1e-12, as the other deposition tests."""

import types

import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


def _cfg(N, c, f):
    return types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=c,
        plasma_fineness=f)


def _run(oracle, cfg, cells, mixed, edit=None, compare=True, seed=0):
    import lcode3d_amd as lc
    _, _, const, vp, _ = oracle.init(cfg)
    rng = np.random.default_rng(seed)
    shape = const.m.shape
    xo, yo = (cells * cfg.grid_step_size * rng.uniform(-1, 1, shape) for _ in range(2))
    px, py, pz = (.3 * rng.uniform(-1, 1, shape) for _ in range(3))
    m, q = const.m.copy(), const.q.copy()
    if mixed:
        m *= rng.uniform(.5, 2, shape)
        q *= rng.uniform(.5, 2, shape)
    if edit:
        edit(xo, vp)
    args = (xo, yo, m, q, px, py, pz)
    dvp = types.SimpleNamespace(**{k: dev(getattr(vp, k)) for k in (
        "influence_prev", "influence_next", "fine_grid", "indices_prev", "indices_next")})
    got = lc.deposit(cfg, dev(const.ro_initial), *map(dev, args), dvp)
    torch.cuda.synchronize()
    return got, oracle.deposit(cfg, const.ro_initial, *args, vp) if compare else None


@pytest.mark.parametrize("N,c,f,cells,mixed", [
    (51, 2, 2, .3, False), (129, 1, 1, 0., False), (129, 2, 3, 2.2, True),
    (193, 3, 2, 6.5, True), (201, 3, 1, 1., False), (217, 2, 2, 4., True),
    (401, 1, 2, 1.3, True), (401, 3, 3, .9, False), (433, 2, 2, 2.9, False),
    (649, 3, 2, 5., True)])
def test_deposit_matches_oracle(oracle, N, c, f, cells, mixed):
    say(f"deposit tiles N={N} c={c} f={f} cells={cells} mixed={mixed}")
    got, want = _run(oracle, _cfg(N, c, f), cells, mixed)
    for name, g, w in zip(("ro", "jx", "jy", "jz"), got, want):
        assert rel_l2(host(g), w) < 1e-12, name


def _whole_cells(xo, vp):           # offsets of exactly 1 .. 6 cells
    xo[...] = (6.4 / 129) * np.resize(np.arange(-6, 7), xo.shape)


def _far_weights(xo, vp):           # a fine particle further out than its coarse ones
    xo[...] = 2.5 * 6.4 / 129
    vp.influence_prev[40] *= 3


@pytest.mark.parametrize("edit", [_whole_cells, _far_weights])
def test_deposit_alone_bounds_its_own_halo(oracle, edit):
    say(f"deposit alone, {edit.__name__}")
    import lcode3d_amd as lc
    lc.fault_count()
    got, want = _run(oracle, _cfg(129, 2, 2), .4, False, edit)
    assert lc.fault_count() == 0
    for name, g, w in zip(("ro", "jx", "jy", "jz"), got, want):
        assert rel_l2(host(g), w) < 1e-12, name


def test_deposit_alone_keeps_nan_local(oracle):
    say("deposit alone, one NaN offset")
    import lcode3d_amd as lc

    def one_nan(xo, vp):
        xo[30, 30] = np.nan

    got, _ = _run(oracle, _cfg(129, 2, 2), .4, False, one_nan, compare=False)
    bad = np.isnan(host(got[0]))
    assert bad.any() and not bad.all()
    with pytest.raises(FloatingPointError):
        cfg = _cfg(129, 2, 2)
        _, _, const, vp, st = lc.init(cfg)
        for _ in range(3):           # (the flag of a workspace shared with the step)
            st = lc.step(cfg, const, vp, st, 0)
            torch.cuda.synchronize()
