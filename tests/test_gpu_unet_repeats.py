"""The network's gradient and training repeat bit for bit: the weight gradients
are sums over workgroups that are added in a fixed order. Sizes where a layer
has one workgroup, a few, and more than the 16 that are added side by side."""
import numpy as np
import pytest

import incrmt_amd as ia
from tests.test_gpu_unet import bf16, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nx", [(8, 9), (24, 40), (65, 48), (257, 257), (300, 700)])
def test_gradient_repeats(ny, nx):
    in3, target = sample(ny, nx, 3)
    nets = [ia.UNet(nx, ny, seed=5) for _ in range(2)]
    p = bf16(nets[0].get_params())
    got = []
    for net in nets:
        net.set_params(p)
        got += [net.gradient(in3, target) for _ in range(3)]
    assert np.any(got[0][1] != 0)
    for loss, grad in got[1:]:
        assert loss == got[0][0] and np.array_equal(grad, got[0][1])


def test_training_repeats():
    in3, target = sample(129, 130, 4)
    nets = [ia.UNet(130, 129, seed=6) for _ in range(2)]
    for net in nets:
        for _ in range(8):
            net.train_step(in3, target, 1e-3)
    assert np.array_equal(nets[0].get_params(), nets[1].get_params())
