"""The FP64 sums of the 16-channel network's training kernels (loss, head and mixing-layer
gradients): blocks that take one group of points, a remainder, or many groups each."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel
from pairs import links


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt,layers", [(1, 1, 1, 4), (0, 2, 3, 4), (0, 2, 3, 2), (1, 3, 5, 3),
                                                 (1, 11, 17, 4)])
def test_batch_gradient_is_the_mean_of_the_pairs(gpu, lattice, n, Lt, layers):
    """20, 126, 900 and 41,140 points per pair: below one group of 64, groups cut by the pair's
    end, and more groups (of 64 and, with two pairs, of 256) than the kernels have blocks.  A
    batch of two scales every FP32 value of the backward pass by 1/2 exactly, so its gradient
    differs from the mean of the single pairs' only where groups of points fall differently:
    the FP32 accumulation of 64 products, 64 * 2^-24 = 4e-6 relative; the loss is summed in
    FP64 throughout."""
    print(f"case lattice={lattice} n={n} Lt={Lt} layers={layers}", flush=True)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=0.3)
    D.update(*links(lattice, n, Lt))
    net = q.Net(D, layers=layers, seed=3)
    rng = np.random.default_rng(7)
    r, e = ((rng.normal(size=(2, D.N)) + 1j * rng.normal(size=(2, D.N))).astype(np.complex64) for _ in range(2))
    one = [net.loss_grad(r[b:b + 1], e[b:b + 1]) for b in (0, 1)]
    loss, g = net.loss_grad(r, e)
    assert abs(loss - 0.5 * (one[0][0] + one[1][0])) <= 1e-12 * loss
    assert rel(g, 0.5 * (one[0][1] + one[1][1])) < 4e-6
    again = net.loss_grad(r, e)
    assert again[0] == loss and np.array_equal(again[1], g)
