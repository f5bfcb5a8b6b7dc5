"""The network's loss, gradient and predictions around the sizes of its training groups (csrc/learn_kernels.hip: sixteen
samples at a time, up to 64 workgroups): one sample, the edges of a group, and of the workgroups' shares.

Bars of test_gpu_learn: FP32 sums against the FP64 reference, 2e-4 of the largest gradient entry."""
import numpy as np
import pytest

from oracle import mlp
from sunhubbardmy_amd.learned import EffectiveAction
from test_gpu_learn import _rand_weights, _samples, relmax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 500, 1023, 1024, 1025, 2049])
def test_groups(n):
    x, norm = _samples(4, n)
    if n == 1:
        norm = _samples(4, 100)[1]
    net = EffectiveAction(capacity=n, seed=3)
    wts = _rand_weights(9)
    net.set_weights(wts)
    net.set_norm(norm)
    print("samples", n, flush=True)
    loss, g = net.loss_grad(x)
    l0, g0 = mlp.loss_grad(wts, norm, x)
    assert abs(loss - l0) < 2e-4 * l0
    assert relmax(g.astype(np.float64), g0) < 2e-4
    e, e0 = net.predict(x[:, :4]), mlp.forward(wts, norm, x[:, :4])
    assert relmax(e - norm[8], e0 - norm[8]) < 2e-5
    net.close()
