"""The learned method's parallel-in-time layers at every chunk length (4, 8 or 16 slices a lane
by the lattice's size, 16 on split blocks beyond 64 slices): K, K^dagger and K K^dagger by the
solver's kernels against the FP32 layers, which the oracle checks."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel
from pairs import geometry, links, source
from renumber import renumber


def _check(D, layers, v):
    K = q.Precond(D, layers=layers)
    rng = np.random.default_rng(4)
    K.params = 1 + 0.05 * (rng.normal(size=K.nparams) + 1j * rng.normal(size=K.nparams))
    adj = K.apply(v, adjoint=True)
    # binary16 fields and transports: the bounds the solver's kernels have against the oracle
    assert rel(K.apply_solver(v), K.apply(v)) < 5e-3
    assert rel(K.apply_solver(v, adjoint=True), adj) < 5e-3
    assert rel(K.apply_solver(v, both=True), K.apply(adj)) < 8e-3


@pytest.mark.gpu
@pytest.mark.parametrize("lattice", [0, 1])
@pytest.mark.parametrize("Lt", [1, 2, 3, 4, 5, 8, 29, 32, 33, 40, 61, 64, 65, 130])
def test_chunks_of_small_lattices(gpu, lattice, Lt):
    """Chunks of 4 up to 32 slices (whole, partial and single lanes), of 8 up to 64, split
    blocks beyond."""
    print(f"case lattice={lattice} Lt={Lt}", flush=True)
    D = q.WilsonDirac(lattice, 3, Lt, r=1.0, M5=0.05, at=0.3)
    D.update(*links(lattice, 3, Lt))
    _check(D, 3, source(lattice, 3, Lt, seed=9))


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt", [(0, 33, 11), (1, 47, 19), (1, 92, 50)])
def test_chunks_by_size(gpu, lattice, n, Lt):
    """Sizes on both sides of the rule: 340 waves (chunks of 4), 2,073 (8), 10,584 waves of
    chunks of 16."""
    print(f"case lattice={lattice} n={n} Lt={Lt}", flush=True)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.05, at=0.02)
    rng = np.random.default_rng(1)
    D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
    _check(D, 2, rng.normal(size=D.N) + 1j * rng.normal(size=D.N))


@pytest.mark.gpu
def test_randomly_numbered_tables_keep_to_lds(gpu):
    """A random numbering's halos (several times the range) leave no room for eight lanes'
    tiles: chunks of 16."""
    n, Lt = 12, 64
    g, _ = renumber(geometry(n), 5)
    D = q.WilsonDirac(0, n, Lt, r=1.0, M5=0.05, at=0.1, geometry=g)
    D.update(*links(0, n, Lt))
    _check(D, 2, source(0, n, Lt, seed=9))
