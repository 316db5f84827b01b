"""The shared launches of the batched solve, which twenty-four small systems take: each system against
the oracle, a NaN source among them, sources far outside the binary16 range, autotuned shapes, and
what the call leaves for the contexts' own solves.  The shared launches keep the links' own gauge, so
their solutions differ in the last bits from those of a context's own solve: that tells the route."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel
from pairs import links, oracle_setup, source

SHAPES = [(0, 2, 4, 0.1), (1, 2, 3, 0.05), (0, 4, 8, 0.02), (1, 4, 2, 0.2), (0, 1, 1, 0.15), (1, 1, 5, 0.08),
          (0, 3, 6, 0.12), (1, 3, 9, 0.1)]
COUNT = 24


def _build(tune=()):
    ops, refs, bs = [], [], []
    for k in range(COUNT):
        lat, n, Lt, M5 = SHAPES[k % len(SHAPES)]
        _, Do, at = oracle_setup(lat, n, Lt, M5=M5)
        sp, tp = links(lat, n, Lt, seed=40 + k, kappa=1.4)
        Do.update(sp, tp)
        D = q.WilsonDirac(lat, n, Lt, r=1.0, M5=M5, at=at)
        D.update(sp, tp)
        if k in tune:
            D.autotune()
        ops.append(D)
        refs.append(Do)
        bs.append(source(lat, n, Lt, seed=100 + k))
    return ops, refs, bs


def _batch(ops, bs, tol, **kw):
    d_b = [q.DeviceArray.from_numpy(b) for b in bs]
    d_x = [q.DeviceArray(b.nbytes) for b in bs]
    reps = q.batch_solve(ops, d_x, d_b, tol=tol, **kw)
    return [x.to_numpy(np.complex128) for x in d_x], reps


@pytest.mark.gpu
def test_every_system_matches_the_oracle(gpu):
    ops, refs, bs = _build(tune=(2, 5, 9))
    xs, reps = _batch(ops, bs, 1e-12)
    own = [D.solve(b, tol=1e-12, solver=q.CG_HALF) for D, b in zip(ops, bs)]
    assert not all(np.array_equal(x, o[0]) for x, o in zip(xs, own))  # not the own-stream route
    for x, r, Do, b, o in zip(xs, reps, refs, bs, own):
        assert r.status == 0 and r.true_resid <= 1e-12
        # 1e-12 residuals times |A^-1| |b| / |x| below 50 on each side
        assert rel(x, Do.solve(b, tol=1e-13)[0]) < 1e-10
        assert abs(o[1].iterations - r.iterations) <= 2
    assert len({r.iterations for r in reps}) > 1  # systems converge on their own


@pytest.mark.gpu
def test_nan_and_scaled_sources(gpu):
    ops, refs, bs = _build()
    scales = np.where(np.arange(COUNT) % 3 == 0, 1e-25, np.where(np.arange(COUNT) % 3 == 1, 1.0, 1e25))
    bs = [s * b for s, b in zip(scales, bs)]
    bad = (1, 11)
    for k in bad:
        bs[k][3] = np.nan
    xs, reps = _batch(ops, bs, 1e-11, raise_on_fail=False)
    for k, (x, r, Do, b, s) in enumerate(zip(xs, reps, refs, bs, scales)):
        if k in bad:
            assert r.status == 4
            continue
        assert r.status == 0 and r.true_resid <= 1e-11
        assert rel(x / s, Do.solve(b / s, tol=1e-13)[0]) < 1e-9


@pytest.mark.gpu
def test_own_solves_after_shared_launches(gpu):
    """The shared launches free the contexts' work fields: a context's next own solve allocates new
    ones and must not replay the chunk it captured on the old."""
    ops, _, bs = _build()
    fresh, _, _ = _build()
    for solver in (q.CG_HALF, q.CG_F64, q.CG_MIXED):
        ref = [fresh[k].solve(bs[k], tol=1e-10, solver=solver)[0] for k in (2, 7)]
        for _ in range(2):
            assert all(np.array_equal(ops[k].solve(bs[k], tol=1e-10, solver=solver)[0], x) for k, x in zip((2, 7), ref))
            _batch(ops, bs, 1e-10)
            hold = [q.DeviceArray(c * D.N) for D in ops for c in (4, 8, 16)]  # takes what was freed
            assert all(np.array_equal(ops[k].solve(bs[k], tol=1e-10, solver=solver)[0], x) for k, x in zip((2, 7), ref))
            del hold
