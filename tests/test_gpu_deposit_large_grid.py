"""lcode_deposit_noalloc on a grid of more tiles than a word of the block table
holds (66049 tiles of 24 cells): the same plasma as on a small grid of the same cell size
lies in its middle, so the middle is the small grid's deposition (FP64 sums in
another order: relative L2 <= 1e-12) and the rest the ion background as it is."""

import ctypes
import types

import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, rel_l2, say

pytestmark = pytest.mark.gpu


def _cfg(N):
    return types.SimpleNamespace(
        grid_steps=N, grid_step_size=.05, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=3,
        plasma_fineness=2)


def test_more_tiles_than_table_words(oracle):
    from lcode3d_amd import _lib
    from lcode3d_amd import lcode as L
    lib = _lib.load()
    small, large = _cfg(217), _cfg(6145)
    _, _, const, vp, _ = oracle.init(small)
    rng = np.random.default_rng(3)
    shape = const.m.shape
    args = [small.grid_step_size * rng.uniform(-1, 1, shape) for _ in range(2)]
    args += [const.m, const.q] + [.3 * rng.uniform(-1, 1, shape) for _ in range(3)]
    parts = [dev(a) for a in args]
    keep = [dev(getattr(vp, k)) for k in (
        "influence_prev", "influence_next", "fine_grid", "indices_prev", "indices_next")]
    cvp = _lib.LcodeVirtParams(*(t.data_ptr() for t in keep))
    got = {}
    for cfg in (small, large):
        n = cfg.grid_steps
        say(f"deposit_noalloc {n}^2")
        ro0 = torch.full((n, n), .25, dtype=torch.float64, device="cuda")
        outs = [torch.full((n, n), np.nan, dtype=torch.float64, device="cuda") for _ in range(4)]
        cs = L._config_struct(cfg, shape[0], keep[2].numel())
        rc = lib.lcode_deposit_noalloc(
            ctypes.byref(cs), ro0.data_ptr(), *[p.data_ptr() for p in parts], ctypes.byref(cvp),
            (ctypes.c_void_p * 4)(*(o.data_ptr() for o in outs)),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.lcode_last_error()
        torch.cuda.synchronize()
        got[n] = outs
    lo = 6145 // 2 - 217 // 2
    for k, (a, b) in enumerate(zip(got[217], got[6145])):
        mid = b[lo:lo + 217, lo:lo + 217]
        assert rel_l2(host(mid), host(a)) < 1e-12, k
        mid.fill_(.25 if k == 0 else 0.)
        assert torch.equal(b, torch.full_like(b, .25 if k == 0 else 0.)), k
