"""The gradient kernels at batches of one sample, around the sixteen samples of a workgroup and around the batch sizes at
which the weight sums are split (MLP_PARAMS = 9217 floats per part out of 64 per sample: two parts from 289 samples on,
three from 433), against the float64 oracle.  The sums are FP32 over at most 1000 terms of magnitude at most 1."""
import numpy as np
import pytest

import oracle_lib
import rampack_amd as ra
from test_mlp_oracle import random_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 288, 289, 432, 433, 1000])
def test_gradient_batch_sizes(batch):
    rng = np.random.Generator(np.random.PCG64(batch))
    theta = random_net(3)
    x = rng.uniform(-1, 1, (batch, 12)).astype(np.float32)
    y = (rng.random(batch) < 0.3).astype(np.float32)
    loss, grad = ra.mlp_gradient(theta, x, y)
    loss_o, grad_o, _ = oracle_lib.mlp_loss_grad(theta, x, y)
    assert loss == pytest.approx(loss_o, rel=1e-5)
    err = np.abs(grad - grad_o)
    assert np.all(err <= 1e-4 * np.abs(grad_o).max() + 1e-4 * np.abs(grad_o)), err.max()
