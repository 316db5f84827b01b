"""Where the angles of a gauge update may lie: the phases are made straight from the caller's arrays
only if they are aligned memory of the device; host memory given as device memory (pageable or
pinned) and unaligned addresses go through a copy, and a range beyond its allocation is refused."""
import ctypes as C

import numpy as np
import pytest
import torch

import qed3_amd as q
from pairs import links, source

LAT, N, LT = 0, 4, 6


class _Shifted(q.DeviceArray):
    """a's bytes 4 past an allocation's start"""

    def __init__(self, a):
        super().__init__(a.nbytes + 8)
        raw = np.zeros(a.nbytes + 8, np.uint8)
        raw[4:4 + a.nbytes] = a.view(np.uint8).reshape(-1)
        self.upload(raw)


def _place(kind, a):
    """(owner, address) of a copy of a"""
    if kind == "pageable":
        return a, a.ctypes.data
    if kind == "pinned":
        t = torch.from_numpy(a).pin_memory()
        return t, t.data_ptr()
    if kind == "inside":  # not at its allocation's start
        d = q.DeviceArray.from_numpy(np.concatenate([np.zeros(7), a.reshape(-1)]))
        return d, d.ptr.value + 56
    d = _Shifted(a) if kind == "unaligned" else q.DeviceArray.from_numpy(a)
    return d, d.ptr.value + (4 if kind == "unaligned" else 0)


def _set(D, s, t):
    return q.load().qed3_set_gauge(D._h, C.c_void_p(s), C.c_void_p(t), 1)


@pytest.mark.gpu
@pytest.mark.parametrize("ks,kt", [("device", "device"), ("inside", "inside"), ("pageable", "pageable"),
                                   ("pinned", "pinned"), ("unaligned", "unaligned"), ("device", "pageable"),
                                   ("pinned", "device")])
def test_angles_in_any_memory(gpu, ks, kt):
    print(f"case spatial={ks} temporal={kt}", flush=True)
    D = q.WilsonDirac(LAT, N, LT, r=1.0, M5=0.1, at=0.3)
    sp, tp = (np.ascontiguousarray(a) for a in links(LAT, N, LT, seed=5))
    b = source(LAT, N, LT, seed=2)
    D.update(sp, tp)
    ref = [D.mult(b), D.mult(b, q.F32), D.mult(b, q.F16)]
    D.update(0 * sp, 0 * tp)
    (own_s, s), (own_t, t) = _place(ks, sp), _place(kt, tp)
    assert _set(D, s, t) == 0
    assert all(np.array_equal(x, y) for x, y in zip(ref, [D.mult(b), D.mult(b, q.F32), D.mult(b, q.F16)]))


@pytest.mark.gpu
def test_a_short_range_is_refused(gpu):
    D = q.WilsonDirac(LAT, N, LT, r=1.0, M5=0.1, at=0.3)
    sp, tp = (np.ascontiguousarray(a) for a in links(LAT, N, LT, seed=5))
    d_s, d_t = q.DeviceArray.from_numpy(sp), q.DeviceArray.from_numpy(tp)
    short = q.DeviceArray.from_numpy(sp[:-1])
    assert _set(D, short.ptr.value, d_t.ptr.value) != 0
    assert _set(D, d_s.ptr.value, d_t.ptr.value) == 0  # and the context still works
    b = source(LAT, N, LT, seed=2)
    got = D.mult(b)
    D.update(sp, tp)
    assert np.array_equal(got, D.mult(b))
