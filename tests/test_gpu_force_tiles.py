"""The force kernel's tiles of slices (whole, partial, a single slice, Lt of one and two where a
slice is its own time neighbour) and the owner of a link (either orientation, pentavalent
padding), against the oracle; the gauge update's one pass against the operator built from it."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel
from pairs import geometry, links, oracle_setup, source
from renumber import renumber


@pytest.mark.gpu
@pytest.mark.parametrize("lattice", [0, 1])
@pytest.mark.parametrize("n,Lt", [(1, 1), (2, 1), (2, 2), (3, 3), (2, 5), (4, 16), (3, 17), (2, 33), (3, 40)])
def test_force_matches_oracle(gpu, lattice, n, Lt):
    print(f"case lattice={lattice} n={n} Lt={Lt}", flush=True)
    L, Do, at = oracle_setup(lattice, n, Lt, M5=0.1)
    sp, tp = links(lattice, n, Lt)
    Do.update(sp, tp)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=at)
    D.update(sp, tp)
    eta = source(lattice, n, Lt, seed=3)
    fs, ft = D.force(eta)
    rs, rt = Do.force(eta)
    # FP64 sums of a few tens of products each: 1e-12 relative, as the force's other tests
    assert rel(fs, rs) < 1e-12
    assert rel(ft, rt) < 1e-12 or np.linalg.norm(rt) < 1e-12 * np.linalg.norm(rs)


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt", [(0, 61, 57), (1, 43, 61), (1, 228, 3)])
def test_force_by_sites_is_the_derivative_along_a_direction(gpu, lattice, n, Lt):
    """2.1, 2.3 and 3.1 M points: the form by sites (whole and partial tiles of slices and ranges,
    both links' orientations).  D is trigonometric in a common angle t added to a set of links, so
    for w = D eta at t = 0, sum_l F_l = -2 d/dt Re <w, D(t) eta>, and the derivative of
    a + b cos t + c sin t at 0 is (f(pi/2) - f(-pi/2)) / 2 exactly; the sums of 4 M products round
    at 1e-16 of the sum of their magnitudes, which sqrt(points) cancellations leave below 1e-10."""
    print(f"case lattice={lattice} n={n} Lt={Lt}", flush=True)
    rng = np.random.default_rng(2)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=0.02)
    sp, tp = rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V))
    eta = rng.normal(size=D.N) + 1j * rng.normal(size=D.N)
    D.update(sp, tp)
    w = D.mult(eta)
    fs, ft = D.force(eta)

    def f(dsp, dtp):
        D.update(sp + dsp, tp + dtp)
        return np.vdot(w, D.mult(eta)).real

    pick = rng.random(sp.shape) < 0.5
    tick = rng.random(tp.shape) < 0.5
    for got, a, b in ((fs[pick].sum(), pick, 0 * tick), (ft[tick].sum(), 0 * pick, tick)):
        h = np.pi / 2
        ref = -2 * (f(h * a, h * b) - f(-h * a, -h * b)) / 2
        scale = np.abs(fs).sum() if b is not tick else np.abs(ft).sum()
        assert abs(got - ref) < 1e-10 * scale, (got, ref, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("lattice", [0, 1])
def test_force_on_reversed_links_is_the_relabelled_force(gpu, lattice):
    n, Lt = 3, 6
    g, maps = renumber(geometry(n), 8)
    R = maps(lattice, Lt)
    sp, tp = links(lattice, n, Lt)
    eta = source(lattice, n, Lt, seed=3)
    A = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=0.2)
    A.update(sp, tp)
    B = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.1, at=0.2, geometry=g)
    B.update(R.spatial(sp), R.temporal(tp))
    fs, ft = A.force(eta)
    gs, gt = B.force(R.spinor(eta))
    assert rel(gs, R.spatial(fs)) < 1e-12
    assert rel(gt, R.temporal(ft)) < 1e-12


@pytest.mark.gpu
def test_gauge_update_from_device_and_host_agree_in_every_precision(gpu):
    """A second update goes through the tables the first solve has built (FP64, FP32, 16-bit)."""
    lattice, n, Lt = 0, 3, 7
    sp, tp = links(lattice, n, Lt, seed=2)
    D = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.2, at=0.2)
    D.update(*links(lattice, n, Lt, seed=1))
    v = source(lattice, n, Lt, seed=5)
    D.apply(q.OP_D, v, q.F16)
    F = q.WilsonDirac(lattice, n, Lt, r=1.0, M5=0.2, at=0.2)
    F.update(sp, tp)
    d_sp, d_tp = q.DeviceArray.from_numpy(sp), q.DeviceArray.from_numpy(tp)
    q.check(q.load().qed3_set_gauge(D._h, d_sp.ptr, d_tp.ptr, 1))
    for prec in (q.F64, q.F32, q.F16):
        assert np.array_equal(D.apply(q.OP_D, v, prec), F.apply(q.OP_D, v, prec))
