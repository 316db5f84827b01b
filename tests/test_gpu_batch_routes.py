"""Both routes of the batched solve: few systems on their own streams, many small ones in shared
launches, and a mixture; every solution satisfies its own system."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel

TOL = 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(0, 4, 6)], [(1, 3, 5), (0, 5, 4), (1, 4, 8)],  # own streams
    [(k % 2, 2 + k % 4, 3 + k % 5) for k in range(40)],  # shared launches
    [(k % 2, 2 + k % 3, 4) for k in range(30)] + [(1, 40, 12)],  # both
], ids=["one", "few", "many", "mixed"])
def test_every_system_is_solved(gpu, shapes):
    rng = np.random.default_rng(3)
    ops, bs, d_b, d_x = [], [], [], []
    for k, (lat, n, Lt) in enumerate(shapes):
        D = q.WilsonDirac(lat, n, Lt, r=1.0, M5=0.05 + 0.01 * (k % 7), at=0.3)
        D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
        b = rng.normal(size=D.N) + 1j * rng.normal(size=D.N)
        if k == 1:
            b[:] = 0  # a zero source: done at the start
        ops.append(D)
        bs.append(b)
        d_b.append(q.DeviceArray.from_numpy(b))
        d_x.append(q.DeviceArray(b.nbytes))
    for _ in range(2):  # the second call reuses what the first has built
        reps = q.batch_solve(ops, d_x, d_b, tol=TOL)
        for D, b, x, r in zip(ops, bs, d_x, reps):
            assert r.status == 0
            res = b - D.DHD(x.to_numpy(np.complex128))
            # the solver's own FP64 residual; the host's norm differs by rounding alone
            assert np.linalg.norm(res) <= TOL * np.linalg.norm(b) * (1 + 1e-3)
    one = ops[0].solve(bs[0], tol=TOL, solver=q.CG_HALF)[0]
    # |A^-1| |b| TOL on each side, |A^-1| |b| / |x| below 50 at these masses
    assert rel(d_x[0].to_numpy(np.complex128), one) < 100 * TOL
