"""lcode_deposit in a workspace whose pushes met other states, through the C ABI: a
push of a state with a NaN must not reach the deposition of a finite one (which
is the oracle's, relative L2 <= 1e-12), and deposited itself it spoils the tiles
around its particle alone.  Both orders of the workspace's slots."""

import ctypes
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


class Workspace:
    """One workspace and the operators on it."""

    def __init__(self, oracle, cfg):
        from lcode3d_amd import _lib
        from lcode3d_amd import lcode as L
        self.lib, self.cfg = _lib.load(), cfg
        _, _, self.const, self.vp, _ = oracle.init(cfg)
        self.shape = self.const.m.shape
        self.keep = [dev(getattr(self.vp, k)) for k in (
            "influence_prev", "influence_next", "fine_grid", "indices_prev", "indices_next")]
        self.cvp = _lib.LcodeVirtParams(*(t.data_ptr() for t in self.keep))
        self.cs = L._config_struct(cfg, self.shape[0], self.keep[2].numel())
        self.ws = ctypes.c_void_p()
        _lib.check(self.lib.lcode_workspace_create(ctypes.byref(self.cs), ctypes.byref(self.ws)),
                   "create")
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.m, self.q, self.x, self.y, self.ro0 = (
            dev(getattr(self.const, k)) for k in ("m", "q", "x_init", "y_init", "ro_initial"))

    def push(self, xo, yo, p):
        n = self.cfg.grid_steps
        fields = [torch.zeros((n, n), dtype=torch.float64, device="cuda") for _ in range(6)]
        ins = [self.m, self.q, self.x, self.y, xo, yo, xo, yo, *p]
        outs = [torch.empty_like(xo) for _ in range(5)]
        ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*(t.data_ptr() for t in ts))  # noqa: E731
        rc = self.lib.lcode_move_smart(self.ws, ctypes.byref(self.cs),
                                       *[t.data_ptr() for t in ins], ptrs(fields), ptrs(outs),
                                       self.stream)
        torch.cuda.synchronize()
        assert rc == 0, self.lib.lcode_last_error()
        return outs

    def deposit(self, xo, yo, p):
        n = self.cfg.grid_steps
        outs = [torch.empty((n, n), dtype=torch.float64, device="cuda") for _ in range(4)]
        parts = [xo, yo, self.m, self.q, *p]
        rc = self.lib.lcode_deposit(
            self.ws, ctypes.byref(self.cs), self.ro0.data_ptr(), *[t.data_ptr() for t in parts],
            ctypes.byref(self.cvp), (ctypes.c_void_p * 4)(*(o.data_ptr() for o in outs)),
            self.stream)
        torch.cuda.synchronize()
        assert rc == 0, self.lib.lcode_last_error()
        return outs

    def close(self):
        torch.cuda.synchronize()
        self.lib.lcode_workspace_destroy(self.ws)


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
