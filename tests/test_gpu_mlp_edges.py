"""The closure network's passes at the edges of their split: 64 samples a
workgroup, 16-sample groups of the weight gradients, 256 interleaved partial
sums of the bias gradients.  References and bounds as in test_gpu_mlp.py: the
oracle with the same BF16 roundings, whose distance is set by the rare
roundings that FP32 accumulation order flips."""
import numpy as np
import pytest

from test_gpu_mlp import M, _case, _net, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 64, 65, 129, 8193])
def test_forward_sizes(n):
    closure, p = _net(21)
    x, _, s = _case(n, 22)
    print("forward n =", n, flush=True)
    net = closure.Mlp(p, s)
    y = net.forward(x)
    net.close()
    assert _rel(y, M.forward(p, s, x, bf16_mode=True)) < 2e-3


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 400, 1111])
def test_gradient_sizes(n):
    closure, p = _net(23)
    x, t, s = _case(n, 24)
    print("loss_grad n =", n, flush=True)
    net = closure.Mlp(p, s)
    loss, g = net.loss_grad(x, t)
    net.close()
    lq, gq = M.loss_grad(p, s, x, t, bf16_mode=True)
    assert loss == pytest.approx(lq, rel=2e-3)
    assert _rel(g, gq) < 1e-2


def test_training_is_repeatable_and_epochs_report_their_own_loss():
    closure, p = _net(25)
    x, t, s = _case(1000, 26)
    net = closure.Mlp(p, s)
    a = net.train(x, t, epochs=3, batch=128, lr=1e-3, seed=5)
    pa = net.params()
    net.set_params(p)
    b = net.train(x, t, epochs=3, batch=128, lr=1e-3, seed=5)
    assert np.array_equal(a, b) and np.array_equal(pa, net.params())
    assert a[0] > a[1] > a[2] > 0.0
    net.close()
