"""The multi-shift solve under any launch shape a context can be given."""
import numpy as np
import pytest

import qed3_amd as q

TOL = 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("Lt,tile", [(131073, (64, 1, 1, 0)), (131073, (64, 1, 1, 1)), (13, (64, 1, 0, 1)),
                                     (13, (256, 64, 1, 0))])
def test_shape_with_any_number_of_blocks(gpu, Lt, tile):
    """One range of sites, padded to eight, and 131,073 slices are eight blocks more than the
    reduction scratch has room for; a context takes that shape for its applications."""
    print(f"case Lt={Lt} tile={tile}", flush=True)
    rng = np.random.default_rng(4)
    D = q.WilsonDirac(0, 1, Lt, r=1.0, M5=0.3, at=0.5)
    D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
    D.set_tile(*tile)
    b = rng.normal(size=D.N) + 1j * rng.normal(size=D.N)
    shifts = [0.0, 0.5]
    for _ in range(2):  # the second solve replays what the first has captured
        xs, reps = q.multishift_solve(D, b, shifts, tol=TOL)
        for s, x, r in zip(shifts, xs, reps):
            assert r.status == 0
            # the solver's own FP64 residual; the host's norm differs by rounding alone
            assert np.linalg.norm(b - D.DHD(x) - s * x) <= TOL * np.linalg.norm(b) * (1 + 1e-3)
