"""Batched solves of contexts on a caller's stream: what the caller has queued there comes first, and
contexts on one stream are solved as well as those on their own."""
import numpy as np
import pytest
import torch

import qed3_amd as q
from conftest import rel

TOL = 1e-10


class At:
    def __init__(self, t):
        self.ptr = t.data_ptr()


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(1, 3, 5)] * 2, [(k % 2, 2 + k % 4, 3 + k % 5) for k in range(24)],
                                    [(0, 4, 6)] * 3 + [(1, 40, 16)] * 2], ids=["few", "many", "large"])
@pytest.mark.parametrize("which", ["all", "last"])
def test_sources_queued_on_the_callers_stream(gpu, shapes, which):
    """The sources are written on the caller's stream behind other work; a call that does not wait
    for them solves for zeros."""
    print(f"case systems={len(shapes)} which={which}", flush=True)
    rng = np.random.default_rng(5)
    st = torch.cuda.Stream()
    ops, bs = [], []
    for k, (lat, n, Lt) in enumerate(shapes):
        D = q.WilsonDirac(lat, n, Lt, r=1.0, M5=0.1, at=0.3)
        D.update(rng.vonmises(0.0, 1.4, (Lt, D.E)), rng.vonmises(0.0, 1.4, (Lt, D.V)))
        if which == "all" or k == len(shapes) - 1:
            D.set_stream(st.cuda_stream)
        ops.append(D)
        bs.append(rng.normal(size=D.N) + 1j * rng.normal(size=D.N))
    src = [torch.from_numpy(b).cuda() for b in bs]
    d_b = [torch.zeros_like(s) for s in src]
    for k, s in enumerate(src):
        if which == "last" and k < len(src) - 1:
            d_b[k].copy_(s)
    d_x = [q.DeviceArray(b.nbytes) for b in bs]

    for _ in range(2):  # the first call builds its tables, which waits by itself
        for k, d in enumerate(d_b):
            if which == "all" or k == len(src) - 1:
                d.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            torch.cuda._sleep(40_000_000)
            for d, s in zip(d_b, src):
                d.copy_(s)
        reps = q.batch_solve(ops, d_x, [At(b) for b in d_b], tol=TOL)
        for D, b, x, r in zip(ops, bs, d_x, reps):
            assert r.status == 0 and r.true_resid <= TOL
            # the solver's own FP64 residual; the host's norm differs by rounding alone
            assert rel(D.DHD(x.to_numpy(np.complex128)), b) <= TOL * (1 + 1e-3)
