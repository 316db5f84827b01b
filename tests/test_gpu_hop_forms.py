"""The two forms of a hop in the 16-bit-angle stencils: at r = 1 the projector form, otherwise the
general one.  r = 1 + 2^-22 is the nearest operator that takes the general form, so both are held
against each other and against FP64."""
import numpy as np
import pytest

import qed3_amd as q
from conftest import rel
from pairs import geometry, links
from renumber import renumber

NEAR = 1.0 + 2.0 ** -22


def _operator(lattice, n, Lt, r, tile, renumbered):
    kw = {"geometry": renumber(geometry(n), 5)[0]} if renumbered else {}
    D = q.WilsonDirac(lattice, n, Lt, r=r, M5=0.05, at=0.2, **kw)
    D.update(*links(lattice, n, Lt))
    D.set_tile(*tile)
    return D


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,n,Lt,tile,renumbered", [
    (0, 1, 1, (64, 1, 0, 0), False), (0, 5, 7, (64, 3, 1, 0), False), (0, 6, 9, (128, 4, 1, 1), False),
    (1, 3, 2, (64, 2, 0, 0), False), (1, 5, 6, (256, 4, 1, 1), False), (0, 9, 5, (256, 2, 1, 0), True)])
def test_forms_agree(gpu, lattice, n, Lt, tile, renumbered):
    print(f"case {lattice} {n} {Lt} {tile} {renumbered}", flush=True)
    one, near = (_operator(lattice, n, Lt, r, tile, renumbered) for r in (1.0, NEAR))
    rng = np.random.default_rng(2)
    v = (rng.normal(size=one.N) + 1j * rng.normal(size=one.N)).astype(np.complex64)
    h = v.real.astype(np.float16).astype(float) + 1j * v.imag.astype(np.float16).astype(float)
    for op in (q.OP_D, q.OP_DDAG, q.OP_DDAGD):
        a, b = one.apply(op, h, q.F16), near.apply(op, h, q.F16)
        # FP32 sums that differ by some 1e-6 round to another binary16 (2^-11 apart) at about
        # 1e-6 / 2^-11 of the points: 2^-11 sqrt(2e-3 n) = 2e-5 for n = 1, less than 2e-4
        assert rel(a, b) < 2e-4, op
        # binary16 results (2^-11 / sqrt 3 each, twice for D^dag D) and 5e-5 of angle rounding
        assert rel(a, one.apply(op, h)) < 2e-3, op
    ra, rb = (D.solve(h, tol=1e-11, solver=q.CG_HALF) for D in (one, near))
    assert ra[1].status == 0 and rb[1].status == 0
    res = h - one.DHD(ra[0])
    assert np.linalg.norm(res) <= 1e-11 * np.linalg.norm(h) * (1 + 1e-3)
    # the operators differ by 2.4e-7 and A^-1 is below 100 at this mass
    assert rel(ra[0], rb[0]) < 1e-4
