"""The solvers keep their captured chunk of iterations with the context: whatever a program
changes between two solves (buffers, source, links, tolerance, chunk length, launch shape,
network coefficients), the second solve gives the bits a fresh context gives."""
import numpy as np
import pytest

import qed3_amd as q
from pairs import links, source

N, LT, M5, AT = 4, 8, 0.1, 0.3


def _context(seed, lattice=1):
    D = q.WilsonDirac(lattice, N, LT, r=1.0, M5=M5, at=AT)
    D.update(*links(lattice, N, LT, seed=seed))
    return D


def _solve(D, K, b, x=None, **kw):
    d_b = q.DeviceArray.from_numpy(b)
    d_x = x or q.DeviceArray(b.nbytes)
    rep = (K or D).solve_device(d_x, d_b, **kw)
    return d_x.to_numpy(np.complex128), rep


def _change(what, D, K, kw):
    if what == "links":
        D.update(*links(D.lattice, N, LT, seed=99))
    elif what == "tile":
        D.set_tile(64, 2, 0, 1)
    elif what == "chunk":
        kw["check_every"] = 24
    elif what == "tol":
        kw["tol"] = 1e-8
    elif what == "coefficients" and K is not None:
        K.params = K.params * (1 + 0.03j)
    return kw


@pytest.mark.gpu
@pytest.mark.parametrize("solver", [q.CG_F64, q.CG_MIXED, q.CG_HALF, q.PCG])
@pytest.mark.parametrize("what", ["source", "links", "tile", "chunk", "tol", "coefficients"])
def test_second_solve_equals_a_fresh_context(gpu, solver, what):
    print(f"case solver={solver} what={what}", flush=True)
    b1, b2 = source(1, N, LT, seed=5), source(1, N, LT, seed=6)

    def make():
        D = _context(3)
        return D, (q.Precond(D, 3) if solver == q.PCG else None)

    base = dict(tol=1e-10) if solver == q.PCG else dict(tol=1e-10, solver=solver)
    D, K = make()
    keep = [_solve(D, K, b1, **base) for _ in range(2)]  # the second replays the first's chunk
    assert np.array_equal(keep[0][0], keep[1][0])
    kw = _change(what, D, K, dict(base))
    got, rep = _solve(D, K, b2, **kw)
    F, G = make()
    kw = _change(what, F, G, dict(base))
    ref, rep_ref = _solve(F, G, b2, **kw)
    assert (rep.iterations, rep.reliable_updates) == (rep_ref.iterations, rep_ref.reliable_updates)
    assert np.array_equal(got, ref)


@pytest.mark.gpu
def test_two_contexts_and_a_batch_keep_their_own(gpu):
    """Interleaved solves on two contexts of one shape, and the batched call that runs them
    together, do not replay each other's chunks."""
    A, B = _context(3), _context(4)
    b = source(1, N, LT, seed=5)
    ra, rb = (_solve(D, None, b, tol=1e-10, solver=q.CG_HALF)[0] for D in (_context(3), _context(4)))
    for _ in range(2):
        assert np.array_equal(_solve(A, None, b, tol=1e-10, solver=q.CG_HALF)[0], ra)
        assert np.array_equal(_solve(B, None, b, tol=1e-10, solver=q.CG_HALF)[0], rb)
    d_b = q.DeviceArray.from_numpy(b)
    xs = [q.DeviceArray(b.nbytes) for _ in range(2)]
    q.batch_solve([A, B], xs, [d_b, d_b], tol=1e-10)  # releases the contexts' work fields
    assert np.array_equal(_solve(A, None, b, tol=1e-10, solver=q.CG_HALF)[0], ra)
    assert np.array_equal(_solve(B, None, b, tol=1e-10, solver=q.CG_HALF)[0], rb)
