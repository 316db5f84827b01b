"""The 16-channel network's buffers grow with the batch: training, inference and training again in
every order of batch sizes give the results of a fresh network."""
import itertools

import numpy as np
import pytest

import qed3_amd as q
from pairs import links


@pytest.mark.gpu
@pytest.mark.parametrize("layers", [2, 5])
@pytest.mark.parametrize("sizes", list(itertools.permutations((1, 2, 4))))
def test_training_after_a_larger_inference(gpu, layers, sizes):
    print(f"case layers={layers} sizes={sizes}", flush=True)
    D = q.WilsonDirac(1, 2, 5, r=1.0, M5=0.1, at=0.3)
    D.update(*links(1, 2, 5))
    rng = np.random.default_rng(7)
    r, e = ((rng.normal(size=(4, D.N)) + 1j * rng.normal(size=(4, D.N))).astype(np.complex64) for _ in range(2))
    calls = [lambda net, B: net.loss_grad(r[:B], e[:B]), lambda net, B: net.apply(r[:B]),
             lambda net, B: net.apply_adj(r[:B])]
    net = q.Net(D, layers=layers, seed=3)
    for k, B in enumerate(sizes + sizes[::-1]):
        for call in calls if k % 2 else calls[::-1]:
            got, ref = call(net, B), call(q.Net(D, layers=layers, seed=3), B)
            assert all(np.array_equal(x, y) for x, y in zip(got, ref))
