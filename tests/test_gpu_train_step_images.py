"""One training step is one launch behind the gradient: sum of the rows, Adam, and the new weights
into the BF16 images that the next gradient reads."""
import numpy as np
import pytest

from trixi_hip.learned_indicator import (IndicatorNeuralNetwork, init_params, khi_semidiscretization, loss_grad,
                                         train_step)

pytestmark = pytest.mark.gpu


# one element, one tile and one row, partial tiles, more tiles than gradient rows
@pytest.mark.parametrize("n", [1, 16, 277, 20000])
def test_step_is_adam_and_images_follow(n):
    import torch
    semi = khi_semidiscretization(2)
    rng = np.random.default_rng(n)
    x = np.zeros((n, 32), np.float32)
    x[:, :19] = rng.uniform(-1, 1, (n, 19))
    xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(rng.uniform(0, 1, n).astype(np.float32)).cuda()
    net = IndicatorNeuralNetwork(init_params(3))
    net.upload(semi)
    _, g = loss_grad(semi, xd, td)
    before = net.params.copy()
    train_step(semi, xd, td, 2e-3)
    after = net.download(semi).params.astype(np.float64)
    # step 1 of Adam: m / (1 - b1) = g, v / (1 - b2) = g^2 up to FP32 rounding (1 - 0.999f
    # alone is off by 2e-5 relative), where eps does not matter: 1e-4 of the step
    ref = before - 2e-3 * g.astype(np.float64) / (np.abs(g) + 1e-8)
    big = np.abs(g) > 1e-5
    assert np.max(np.abs(after - ref)[big], initial=0.0) < 1e-4 * 2e-3 + 2.0 ** -23 * np.max(np.abs(before))
    assert np.all(after[g == 0] == before[g == 0])
    # the images of a step and those of an upload of the same weights: same bits
    step = loss_grad(semi, xd, td)
    IndicatorNeuralNetwork(after.astype(np.float32)).upload(semi)
    fresh = loss_grad(semi, xd, td)
    assert step[0] == fresh[0] and np.array_equal(step[1], fresh[1])
    semi.close()
