"""A deposition whose particles lie closer together than its config says (the config's
coarseness and fineness scale the charge and size the tiles' tables; the particle
grids are the caller's): within the tables' least sizes it is served, by one
round of 16- or 24-cell tiles and by several.  Against the oracle with the same
config, relative L2 <= 1e-12 as the other depositions."""

import copy
import types

import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,c,f,cells,said_c,said_f", [
    (321, 3, 2, 5., 8, 2), (433, 3, 2, 5., 8, 2), (433, 4, 3, 1.5, 6, 1), (721, 3, 2, 5., 8, 2)])
def test_denser_than_configured(oracle, N, c, f, cells, said_c, said_f):
    import lcode3d_amd as lc
    say(f"denser grid N={N} c={c} f={f}, said {said_c} {said_f}, {cells} cells")
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=c + 3, plasma_padding_steps=10, plasma_coarseness=c,
        plasma_fineness=f)
    _, _, const, vp, _ = oracle.init(cfg)
    said = copy.copy(cfg)
    said.plasma_coarseness, said.plasma_fineness = said_c, said_f
    rng = np.random.default_rng(N)
    shape = const.m.shape
    args = [cells * cfg.grid_step_size * rng.uniform(-1, 1, shape) for _ in range(2)]
    args += [const.m, const.q] + [.3 * rng.uniform(-1, 1, shape) for _ in range(3)]
    dvp = types.SimpleNamespace(**{k: dev(getattr(vp, k)) for k in (
        "influence_prev", "influence_next", "fine_grid", "indices_prev", "indices_next")})
    lc.fault_count()
    got = lc.deposit(said, dev(const.ro_initial), *map(dev, args), dvp)
    torch.cuda.synchronize()
    want = oracle.deposit(said, const.ro_initial, *args, vp)
    assert lc.fault_count() == 0
    for name, g, w in zip(("ro", "jx", "jy", "jz"), got, want):
        assert rel_l2(host(g), w) < 1e-12, name
