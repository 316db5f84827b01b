"""What a multi-shift solve leaves allocated: up to 256 MiB of work fields stay with the context, more
are given back at its end."""
import gc

import numpy as np
import pytest
import torch

import qed3_amd as q
from pairs import links, source

MIB = 1 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("shifts", [18, 3])
def test_work_memory_is_given_back(gpu, shifts):
    """0.51 M points: twenty fields are 313 MiB, five 78.  The first solve with one shift has built
    everything else that a context keeps."""
    print(f"case shifts={shifts}", flush=True)
    n, Lt = 32, 50
    D = q.WilsonDirac(0, n, Lt, r=1.0, M5=0.2, at=0.3)
    D.update(*links(0, n, Lt, seed=5))
    b = source(0, n, Lt, seed=2)
    first = q.multishift_solve(D, b, [0.5], tol=1e-8)[0][0]
    gc.collect()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        xs, reps = q.multishift_solve(D, b, list(0.5 + 0.1 * np.arange(shifts)), tol=1e-8)
        assert all(r.status == 0 for r in reps)
        assert np.linalg.norm(xs[0] - first) <= 1e-6 * np.linalg.norm(first)
        del xs
        gc.collect()
        kept = before - torch.cuda.mem_get_info()[0]
        assert kept <= (16 if shifts == 18 else 80) * MIB, kept
