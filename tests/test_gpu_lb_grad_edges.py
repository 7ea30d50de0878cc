"""The learned layer's gradient at the edges of its work split (64 samples a
wave, 256 a block, 512 blocks a round), against the same sums in float64.

Tolerance: the samples' forward and backward passes are in fp32, chains of at
most 32 + 32 + 12 products and sums, each rounded to 2^-24 of the partial sum:
76 * 2^-24 = 4.5e-6 of values of order one.  The residual takes part in the loss
and in the gradient twice (2 d), so both are held to twice that, of the larger
of one and the largest parameter's gradient (the loss); the sums over the
samples add nothing to speak of."""
import numpy as np
import pytest

from oracle import lb_mlp
from xfdtd_cuda_amd import learned

pytestmark = pytest.mark.gpu
TOL = 2 * 76 * 2.0 ** -24


@pytest.mark.parametrize("first,count", [(0, 1), (5, 63), (0, 64), (3, 65), (0, 255), (1, 257), (0, 4096), (7, 131072 + 65)])
def test_gradient_at_the_edges_of_the_split(first, count):
    rng = np.random.default_rng(count)
    smp = rng.uniform(-1, 1, (first + count, 13)).astype(np.float32)
    w = lb_mlp.init_weights(4, out_scale=0.5)
    k = 0.3
    t = learned.Trainer(smp, k).set_weights(w)
    loss, grad = t.grad(first, count)
    again = t.grad(first, count)
    t.close()
    xs, r = lb_mlp.targets(smp[first:], k, drop_zero=False)
    loss_n, grad_n = lb_mlp.loss_and_grad(w, xs, r)
    scale = np.abs(grad_n).max()
    assert np.abs(grad - grad_n).max() <= TOL * max(1.0, scale)
    assert abs(loss - loss_n) <= TOL * max(1.0, loss_n)
    assert again[0] == loss and np.array_equal(again[1], grad)
