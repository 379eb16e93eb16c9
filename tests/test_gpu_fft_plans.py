"""The half-extension FFT of the field solvers (fields.hip passes A and C) over its
plans: every first radix (4 .. 20), every stage radix (2 .. 16), one to three
stages, lengths with kernels of their own and without, odd and even numbers of
first-stage rows, one wavefront to the most (448 threads), FP32 transforms up to the longest
(2049^2).

FP64: the transforms and the oracle's are backward stable, so the bound is the
field solves' 1e-12.  FP32: an FFT of L points with correctly rounded roots
errs by about log2(L) eps (eps = 6e-8) relative, twice per solve: 1.5e-6 of the
right-hand side, spread over all modes, of which the inverse of the operator raises the
lowest against those that carry the solution (by up to some tens); 1e-4 is also what
Ez of the mixed step is held to."""

import types

import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, rel_l2, say, smooth_field

pytestmark = pytest.mark.gpu

SIZES = [11, 13, 19, 31, 33, 41, 55, 65, 73, 81, 101, 151, 181, 217, 241, 257, 321, 361,
         451, 487, 513, 577, 601, 973, 1001, 1025, 1081, 1297, 1621, 1729, 1801]


def solve_and_compare(oracle, N, precision, bound):
    import lcode3d_amd as lc
    say(f"fft plan N={N} {precision}")
    rng = np.random.default_rng(N)
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=6.4 / N, xi_step_size=.05,
        field_solver_subtraction_trick=1, field_solver_variant_A=True,
        reflect_padding_steps=5, plasma_padding_steps=10, plasma_coarseness=2,
        plasma_fineness=2, field_solver_precision=precision)
    args = [smooth_field(rng, N) for _ in range(4)]
    beam = smooth_field(rng, N, .05)
    dens = [smooth_field(rng, N, zero_rim=0) for _ in range(6)]
    got = [*lc.calculate_Ex_Ey_Bx_By(cfg, *map(dev, args), dev(beam), *map(dev, dens)),
           lc.calculate_Ez(cfg, dev(dens[1]), dev(dens[2])),
           lc.calculate_Bz(cfg, dev(dens[1]), dev(dens[2]))]
    torch.cuda.synchronize()
    want = [*oracle.calculate_Ex_Ey_Bx_By(cfg, *args, beam, *dens),
            oracle.calculate_Ez(cfg, dens[1], dens[2]),
            oracle.calculate_Bz(cfg, dens[1], dens[2])]
    for name, g, w in zip(("Ex", "Ey", "Bx", "By", "Ez", "Bz"), got, want):
        assert rel_l2(host(g), w) < bound, name


@pytest.mark.parametrize("N", SIZES)
def test_fp64_plans_match_oracle(oracle, N):
    solve_and_compare(oracle, N, "fp64", 1e-12)


@pytest.mark.parametrize("N", [5, 33, 181, 361, 641, 1281, 1945, 2049])
def test_fp32_plans_match_oracle(oracle, N):
    solve_and_compare(oracle, N, "fp32", 1e-4)
