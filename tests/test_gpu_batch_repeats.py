"""Several sources on one context in a batched solve: a context listed more than once, small and
large (always on its own stream), alone and among others."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel

TOL = 1e-10
SMALL, SMALL6, LARGE = (1, 3, 5, 4), (0, 4, 6, 4), (1, 40, 16, 4)  # lattice, n, Lt, slices per block (0: default shape)


@pytest.mark.gpu
@pytest.mark.parametrize("listed", [
    [SMALL] * 2, [SMALL6] * 3, [LARGE] * 2, [LARGE] * 3, [(1, 8, 64, 1)] * 2, [(0, 16, 16, 0), (1, 15, 13, 0)] * 4,
    [SMALL, LARGE, SMALL6, LARGE, SMALL, SMALL], [SMALL] * 20, [SMALL, SMALL6] * 12 + [LARGE] * 2,
], ids=["small2", "small3", "large2", "large3", "blocks2", "default8", "mixed", "small20", "many"])
def test_each_source_gets_its_own_solution(gpu, listed):
    print("case", listed, flush=True)
    rng = np.random.default_rng(11)
    ctx = {}
    for lat, n, Lt, ts in listed:
        if (lat, n, Lt) not in ctx:
            D = ctx[lat, n, Lt] = q.WilsonDirac(lat, n, Lt, r=1.0, M5=0.1, at=0.3)
            D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
            if ts:
                D.set_tile(256, ts, 1, 0)
    ops = [ctx[s[:3]] for s in listed]
    bs = [rng.normal(size=D.N) + 1j * rng.normal(size=D.N) for D in ops]
    d_b = [q.DeviceArray.from_numpy(b) for b in bs]
    d_x = [q.DeviceArray(b.nbytes) for b in bs]
    for _ in range(2):  # the second call reuses what the first has built
        reps = q.batch_solve(ops, d_x, d_b, tol=TOL)
        for D, b, x, r in zip(ops, bs, d_x, reps):
            assert r.status == 0 and r.true_resid <= TOL
            res = b - D.DHD(x.to_numpy(np.complex128))
            # the solver's own FP64 residual; the host's norm differs by rounding alone
            assert np.linalg.norm(res) <= TOL * np.linalg.norm(b) * (1 + 1e-3)
    for k in {0, len(listed) - 1}:
        one = ops[k].solve(bs[k], tol=TOL, solver=q.CG_HALF)[0]
        # |A^-1| |b| TOL on each side, |A^-1| |b| / |x| below 50 at this mass
        assert rel(d_x[k].to_numpy(np.complex128), one) < 100 * TOL
