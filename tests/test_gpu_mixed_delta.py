"""The mixed solver's reliable update, once per chunk of iterations or, for a loose delta, after every
one: the solution and the counts do not depend on which, and one context goes from one to the other."""
import numpy as np
import pytest

import qed3_amd as q
from pairs import links, source

DELTAS = (0.1, 0.25, 0.26, 0.9, 0.1, 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt,chunk", [(1, 4, 9, 0), (0, 5, 6, 4)])
def test_solutions_at_any_delta(gpu, lattice, n, Lt, chunk):
    print(f"case lattice={lattice} n={n} Lt={Lt} chunk={chunk}", flush=True)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=0.3)
    D.update(*links(lattice, n, Lt, seed=5))
    b = source(lattice, n, Lt, seed=2)
    d_b = q.DeviceArray.from_numpy(b)
    x, y = q.DeviceArray(b.nbytes), q.DeviceArray(b.nbytes)
    for delta in DELTAS:
        # with kernel timing the update always follows every iteration
        ref, _ = D.solve_kernel_times(y, d_b, tol=1e-10, solver=q.CG_MIXED, delta=delta)
        for _ in range(2):
            rep = D.solve_device(x, d_b, tol=1e-10, solver=q.CG_MIXED, delta=delta, check_every=chunk)
            assert rep.status == 0 and rep.true_resid <= 1e-10
            assert (rep.iterations, rep.reliable_updates) == (ref.iterations, ref.reliable_updates)
            assert np.array_equal(x.to_numpy(np.complex128), y.to_numpy(np.complex128))
