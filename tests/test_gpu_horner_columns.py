"""The network's FP32 layers on lattices with many sites, where a thread takes a whole column (from
88,000 sites on), and just below, against the oracle."""
import numpy as np
import pytest

import oracle as O
import qed3_amd as q
from conftest import rel
from pairs import links, oracle_setup, source


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt,bc,layers", [(0, 94, 3, 0, 3), (1, 67, 2, 1, 2), (0, 94, 1, 0, 1),
                                                    (1, 66, 4, 0, 3)])
def test_apply_and_gradient_match_oracle(gpu, lattice, n, Lt, bc, layers):
    """88,362, 89,780 and 87,120 sites, the last range of 256 a part of one; accuracies as of the same
    layers on small lattices: 2e-6 of FP32 sums over at most 4 layers of 8 terms, 1e-5 and 1e-4 of the
    loss and its gradient."""
    print(f"case lattice={lattice} n={n} Lt={Lt} bc={bc} layers={layers}", flush=True)
    _, Do, at = oracle_setup(lattice, n, Lt, M5=0.05, bc=bc)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.05, at=at, bc=bc)
    sp, tp = links(lattice, n, Lt, seed=3, kappa=1.4)
    Do.update(sp, tp)
    D.update(sp, tp)
    rng = np.random.default_rng(layers)
    K = q.Precond(D, layers=layers)
    p = 1 + 0.1 * (rng.normal(size=layers + 4) + 1j * rng.normal(size=layers + 4))
    K.params = p
    v, e = source(lattice, n, Lt, seed=7), source(lattice, n, Lt, seed=8)
    for adj in (False, True):
        assert rel(K.apply(v, adjoint=adj), O.horner_apply(Do, layers, p, v, adjoint=adj)) < 2e-6
    loss, g = K.loss_grad(v[None], e[None])
    loss_o, g_o = O.horner_loss_grad(Do, layers, p, v[None], e[None])
    assert abs(loss - loss_o) < 1e-5 * loss_o
    assert rel(g, g_o) < 1e-4
