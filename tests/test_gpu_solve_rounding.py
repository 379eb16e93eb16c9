"""The Ez solve against 80-bit transforms, to within its rounding.

Both solve the five-point operator whose least eigenvalue is lam = 8 / h^2
sin^2(pi / (2 (N - 1))).  A rounding error e of the right-hand side or of its transform
reaches the solution as e / lam at most, and an error of the transform back stays as
it is.  With unit roundoff r an FFT of L points errs by at most about 4 r per doubling of L in
relative 2-norm (a butterfly's complex product with a rounded root and its sum), two
transforms 8 r log2(L); right-hand side, the recurrences along the other axis and
the scaling are held to 16 r.  The right-hand side's own error is relative to
|d jx / dx| + |d jy / dy|, which may cancel.  So, in 2-norms,

    |u - exact| <= r (8 log2(L) + 16) | |d jx / dx| + |d jy / dy| | / lam.

Plans as constants (L = 2 (N - 1) a power of two or five times one) and from kernel
arguments, FP64 transforms and FP32 ones (whose right-hand side is rounded to FP32)."""

import types

import numpy as np
import pytest
import scipy.fft
import torch

from gpu_helpers import dev, host, say

pytestmark = pytest.mark.gpu

X = np.longdouble


@pytest.mark.parametrize("N,precision", [
    (33, "fp64"), (41, "fp64"), (65, "fp64"), (81, "fp64"), (129, "fp64"), (161, "fp64"),
    (257, "fp64"), (301, "fp64"), (361, "fp64"), (451, "fp64"), (641, "fp64"), (801, "fp64"),
    (1025, "fp64"), (1081, "fp64"), (1281, "fp64"), (1801, "fp64"),
    (41, "fp32"), (81, "fp32"), (161, "fp32"), (361, "fp32"), (641, "fp32"), (2049, "fp32")])
def test_ez_rounding(N, precision):
    import lcode3d_amd as lc
    say(f"Ez rounding N={N} {precision}")
    h, L = 6.4 / N, 2 * (N - 1)
    cfg = types.SimpleNamespace(
        grid_steps=N, grid_step_size=h, xi_step_size=.05, field_solver_subtraction_trick=1,
        field_solver_variant_A=True, reflect_padding_steps=5, plasma_padding_steps=10,
        plasma_coarseness=2, plasma_fineness=2, field_solver_precision=precision)
    x = (np.arange(N) - N // 2) * h
    g = np.exp(-(x[:, None] ** 2 + (x[None, :] - .3) ** 2) / 1.5)
    jx, jy = (x[:, None] + .2) * g, (x[None, :] - .1) * g * np.cos(x[:, None])
    got = host(lc.calculate_Ez(cfg, dev(jx), dev(jy)))
    torch.cuda.synchronize()
    dx = (X(1) * jx[2:, 1:-1] - jx[:-2, 1:-1]) / (2 * X(h))
    dy = (X(1) * jy[1:-1, 2:] - jy[1:-1, :-2]) / (2 * X(h))
    lam = 4 / X(h) ** 2 * np.sin(np.arange(1, N - 1) * np.arccos(X(-1)) / (2 * (N - 1))) ** 2
    f = scipy.fft.dstn(-(dx + dy), type=1) / (lam[:, None] + lam[None, :]) / X(L) ** 2
    want = np.zeros((N, N), X)
    want[1:-1, 1:-1] = scipy.fft.dstn(f, type=1)
    r = 2. ** -53 if precision == "fp64" else 2. ** -24
    scale = np.sqrt(float(((abs(dx) + abs(dy)) ** 2).sum())) / float(2 * lam[0])
    bound = r * (8 * np.log2(L) + 16) * scale
    err = np.sqrt(float(((got - want) ** 2).sum()))
    say(f"  error {err:.2e}, bound {bound:.2e}, relative {err / np.sqrt(float((want ** 2).sum())):.2e}")
    assert err <= bound
