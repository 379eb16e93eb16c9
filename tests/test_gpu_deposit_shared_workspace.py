"""A step in a workspace that was made for a plasma of smaller coarseness with the same
particle counts (the package keys its workspaces by the counts): the outermost
coarse particles moved by 5.9 cells carry fine particles two tiles away from
their own, which the 3 x 3 neighbourhood of per-tile bounds does not hold at this
coarseness.  Against the oracle, one step, relative L2 <= 1e-11 as the other
one-step tests."""

import types

import numpy as np
import pytest

from gpu_helpers import dev, host, rel_l2, say, to_device_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,padding,c,f", [(217, 31, 6, 2), (201, 31, 7, 2), (217, 47, 7, 3)])
def test_coarser_plasma_in_the_same_workspace(oracle, N, padding, c, f):
    import lcode3d_amd as lc
    from lcode3d_amd import lcode as L
    say(f"shared workspace N={N} padding={padding} c={c} f={f}")
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=1e-3,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=c + 3, plasma_padding_steps=padding, plasma_coarseness=c,
        plasma_fineness=f)
    _, _, const, vp, st = oracle.init(cfg)
    nc = const.m.shape[0]
    cs = L._config_struct(cfg, nc, len(vp.fine_grid))
    cs.plasma_coarseness = 2
    L._workspace(cs)
    for axis, at in (("x_offt", (-1, slice(None))), ("x_offt", (0, slice(None))),
                     ("y_offt", (slice(None), -1)), ("y_offt", (slice(None), 0))):
        state = oracle.init(cfg)[4]
        off = np.zeros((nc, nc))
        off[at] = (1 if -1 in at else -1) * 5.9 * cfg.grid_step_size
        setattr(state, axis, off)
        want = oracle.step(cfg, const, vp, state, 0)
        lc.init(cfg)
        got = lc.step(cfg, lc.GPUArrays(**{k: dev(getattr(const, k)) for k in (
            "m", "q", "x_init", "y_init", "ro_initial")}),
            lc.GPUArrays(**{k: getattr(vp, k) for k in (
                "influence_prev", "influence_next", "indices_prev", "indices_next",
                "fine_grid")}), to_device_state(lc, state), 0)
        assert lc.fault_count(cfg, nc) == 0
        for name in ("ro", "x_offt", "y_offt"):
            assert rel_l2(host(getattr(got, name)), getattr(want, name)) < 1e-11, (axis, at, name)
