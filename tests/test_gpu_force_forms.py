"""The two forms of the force kernel, a thread per link and a thread per site, link by link: one and
two pairs, overwriting and accumulating, every range size, a random numbering."""
import numpy as np
import pytest

import qed3_amd as q
from pairs import geometry
from renumber import renumber


def _force(D, fields, c, init, form, fs, ft):
    d = [q.DeviceArray.from_numpy(f) for f in fields]
    p = [a.ptr for a in d] + [None] * (4 - len(d))
    d_s, d_t = q.DeviceArray.from_numpy(fs), q.DeviceArray.from_numpy(ft)
    q.check(q.load().qed3_force_bilinear(D._h, *p, c, init, form, d_s.ptr, d_t.ptr))
    return d_s.to_numpy(np.float64), d_t.to_numpy(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("lattice,n,Lt,tile", [(0, 1, 1, (64, 1, 1, 1)), (0, 4, 2, (64, 2, 1, 1)),
                                               (1, 5, 17, (128, 2, 1, 1)), (0, 7, 5, (256, 4, 1, 1)),
                                               (1, 7, 3, (256, 1, 1, 0)), (0, 11, 33, (256, 4, 1, 1))])
def test_by_sites_equals_by_links(gpu, lattice, n, Lt, tile, shuffled):
    """12 to 1,212 sites: less than a range, ranges and tiles of slices with remainders, one and two
    slices; shuffled, the halo of 256 sites is most of the lattice, and two pairs of such a range do
    not fit in LDS.  A link's value is a sum of at most 64 FP64 products whose terms exceed the
    largest value by less than 10: 64 * 10 * 2^-53 = 7e-14 of it."""
    print(f"case lattice={lattice} n={n} Lt={Lt} tile={tile} shuffled={shuffled}", flush=True)
    rng = np.random.default_rng(8)
    g = renumber(geometry(n), seed=3)[0] if shuffled else geometry(n)
    D = q.WilsonDirac(lattice, n, Lt, r=0.8, M5=0.1, at=0.3, geometry=g)
    D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
    D.set_tile(*tile)
    w = [rng.normal(size=D.N) + 1j * rng.normal(size=D.N) for _ in range(4)]
    fs0, ft0 = rng.normal(size=(Lt, D.E)), rng.normal(size=(Lt, D.V))
    for fields in (w[:2], w):
        for init in (1, 0):
            got, ref = (_force(D, fields, -1.7, init, form, fs0, ft0) for form in (2, 1))
            top = max(np.abs(ref[0]).max(), np.abs(ref[1]).max())
            for a, b in zip(got, ref):
                assert np.abs(a - b).max() <= 7e-14 * top
    # the forces' own choice at these sizes
    auto, ref = (_force(D, w, -1.7, 0, form, fs0, ft0) for form in (0, 1))
    assert all(np.array_equal(a, b) for a, b in zip(auto, ref))


@pytest.mark.gpu
def test_bad_arguments(gpu):
    D = q.WilsonDirac(0, 1, 2, r=1.0, M5=0.1, at=0.3)
    a = q.DeviceArray(16 * D.N)
    f = q.load().qed3_force_bilinear
    assert f(D._h, a.ptr, a.ptr, None, None, 1.0, 1, 0, a.ptr, a.ptr) == 5  # QED3_ERR_STATE: no gauge field
    D.update(np.zeros((2, D.E)), np.zeros((2, D.V)))
    assert f(D._h, a.ptr, a.ptr, a.ptr, None, 1.0, 1, 0, a.ptr, a.ptr) == 1
    assert f(D._h, a.ptr, a.ptr, None, None, 1.0, 1, 3, a.ptr, a.ptr) == 1
    assert f(D._h, None, a.ptr, None, None, 1.0, 1, 0, a.ptr, a.ptr) == 1
