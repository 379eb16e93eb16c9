"""The U-Net's weight gradients at the edges of their reduction over blocks
(one block; a whole group of 32 partials; a ragged last group) against the
U-Net oracle, with the bounds of test_gpu_unet.py: the sums are FP32 in
another order there too, the rest is rare bfloat16 rounding flips."""

import numpy as np
import pytest
import torch

from gpu_helpers import rel_l2, say
from test_gpu_unet import _chw_to_bf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [2, 61, 66])   # 1, 32 and 51 blocks at level 0
def test_gradients_match_oracle(S):
    from lcode3d_amd.unet import UNetPredictor
    from oracle import unet_oracle as uo
    say(f"unet gradients S={S}")
    rng = np.random.default_rng(S)
    net = UNetPredictor(4 * S - 3, seed=0)
    params = [(w, rng.standard_normal(b.shape) * .05) for w, b in uo.init_params(seed=5)]
    net.set_params(params)
    x = uo.bf16(rng.standard_normal((uo.CIN, S, S)))
    t = rng.standard_normal((uo.COUT, S, S)) * .3
    xd = _chw_to_bf(x, S)
    net.forward(xd)
    net.backward(xd, torch.as_tensor(t.transpose(1, 2, 0).astype(np.float32),
                                     device="cuda").contiguous())
    ref = uo.forward(params, x, q=uo.bf16)
    grads = uo.backward(params, ref, uo.mse_grad(ref["y"], t)[1], q=uo.bf16)
    for k, ((gw, gb), (rw, rb)) in enumerate(zip(net.layer_arrays(net.grad), grads)):
        assert rel_l2(gw, rw) < 3e-2 and rel_l2(gb, rb) < 3e-2, k
