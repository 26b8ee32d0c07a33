"""The learned guess's gradient at the edges of its waves (64 samples), of its
blocks (4 waves) and of the chunks that its partial gradients are summed in (64),
against the NumPy reference; bars as in test_gpu_learned.py (bf16 roundings of the first hidden layer may fall either
way where the sums before them differ in the last bit)."""
import numpy as np
import pytest

import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 63, 64, 65, 256, 257, 64 * 64, 64 * 64 + 1, 770 * 64 + 63])
def test_gradient(count):
    from hydrogrp import mlp
    feat, target, _, _ = mlp.data(15, count)
    P = mlp.init_params(4) + np.random.default_rng(4).normal(0, 0.05, mlp.NP).astype(np.float32)
    loss, grad = mlp.loss_grad(P, feat, target)
    loss_ref, grad_ref = mlp_ref.loss_grad(P, feat, target, quantize=True)
    assert abs(loss - loss_ref) <= 1e-4 * loss_ref
    assert np.linalg.norm(grad - grad_ref) <= 2e-3 * np.linalg.norm(grad_ref)
