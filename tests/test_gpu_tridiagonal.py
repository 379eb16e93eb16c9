"""The tridiagonal pass of the FFT field solvers (fields.hip pass B) at the
edges of its tiling: single rows and lines, whole and partial waves of rows
(48 per wave to 192 rows, 96 to 1536, 256 beyond).  The
solves differ from the oracle's transforms by rounding only: both are
backward stable and the measured differences are a few 1e-15, so the bound is
the field solves' 1e-12."""

import types

import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, rel_l2, say, smooth_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trick", [1, 0])
@pytest.mark.parametrize("N", [5, 7, 49, 51, 97, 193, 201, 769, 1537, 1601])
def test_solves_match_oracle(oracle, N, trick):
    import lcode3d_amd as lc
    say(f"tridiagonal N={N} trick={trick}")
    rng = np.random.default_rng(N)
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=trick, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=2,
        plasma_fineness=2)
    args = [smooth_field(rng, N) for _ in range(4)]
    beam = smooth_field(rng, N, .05)
    # jx, jy without a zero rim too: the cosine solve's end rows carry data
    dens = [smooth_field(rng, N, zero_rim=0) for _ in range(6)]
    got = [*lc.calculate_Ex_Ey_Bx_By(cfg, *map(dev, args), dev(beam), *map(dev, dens)),
           lc.calculate_Ez(cfg, dev(dens[1]), dev(dens[2])),
           lc.calculate_Bz(cfg, dev(dens[1]), dev(dens[2]))]
    torch.cuda.synchronize()
    want = [*oracle.calculate_Ex_Ey_Bx_By(cfg, *args, beam, *dens),
            oracle.calculate_Ez(cfg, dens[1], dens[2]),
            oracle.calculate_Bz(cfg, dens[1], dens[2])]
    for name, g, w in zip(("Ex", "Ey", "Bx", "By", "Ez", "Bz"), got, want):
        assert rel_l2(host(g), w) < 1e-12, name
