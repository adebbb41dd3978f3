"""A batch and its cases end in any order."""
import ctypes as C

import numpy as np
import pytest

import fizzy_amd as F
from fizzy_amd import cases

pytestmark = pytest.mark.gpu

FIELDS = ["u", "v", "w", "p", "psi", "kappa"]
RATIOS = (10.0, 50.0, 200.0, 900.0)


def start(graphs=False, icheck=10):
    out = []
    for r in RATIOS:
        dc = F.DeviceCase(dict(cases.rising_bubble_3d(ng=(32, 16, 24), rho12=(r, 1.0)), icheck=icheck))
        dc.init()
        dc.set_graphs(graphs)
        dc.step(1)
        out.append(dc)
    return out


@pytest.mark.parametrize("gone", [[0], [0, 1], [3], [0, 1, 2, 3]], ids=lambda g: "-".join(map(str, g)))
def test_cases_end_before_their_batch(gone):
    """The first case, some or all of them are destroyed while the batch is
    there: it refuses to step, it is destroyed, and the others go on."""
    alone, batched = start(), start()
    try:
        b = F.CaseBatch(batched)
        b.step(2)
        for q in gone:
            batched[q].close()
        with pytest.raises(F.FizzyError, match="destroyed"):
            b.step(1)
        assert F.lib().fz_case_batch_step_begin(b._h, None) == -4
        b.close()
        for q in range(len(RATIOS)):
            if q not in gone:
                alone[q].step(4)
                batched[q].step(2)
                for k in FIELDS:
                    assert np.array_equal(alone[q].get(k), batched[q].get(k)), (q, k)
    finally:
        for dc in alone + batched:
            dc.close()


@pytest.mark.parametrize("gone", [0, 2])
def test_a_case_ends_inside_a_batched_step(gone):
    """Between the two halves of a batched step whose checks are due: the end
    reads the other cases' checks."""
    alone, batched = start(icheck=2), start(icheck=2)
    try:
        b = F.CaseBatch(batched)
        pending = C.c_int()
        F.call("fz_case_batch_step_begin", b._h, C.byref(pending))
        assert pending.value == 1
        batched[gone].close()
        killed = (C.c_int * len(RATIOS))()
        F.call("fz_case_batch_step_end", b._h, killed)
        assert list(killed) == [0] * len(RATIOS)
        b.close()
        for q in range(len(RATIOS)):
            if q != gone:
                alone[q].step(3)
                batched[q].step(2)
                assert np.array_equal(alone[q].scalars(), batched[q].scalars())
                for k in FIELDS:
                    assert np.array_equal(alone[q].get(k), batched[q].get(k)), (q, k)
    finally:
        for dc in alone + batched:
            dc.close()
