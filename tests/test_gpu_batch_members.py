"""A batch and its cases end in any order, and between the batch's steps its
cases are contexts of their own, each driven by a thread of its own."""
import ctypes as C
import threading

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


def each(work, items):
    """work(item) on a thread per item, all started together; their errors."""
    gate, errors = threading.Barrier(len(items)), []

    def body(x):
        try:
            gate.wait(30)
            work(x)
        except Exception as e:  # noqa: BLE001 (reported by the test's thread)
            errors.append(repr(e))

    threads = [threading.Thread(target=body, args=(x,)) for x in items]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    return errors


def test_members_of_a_batch_step_on_threads_of_their_own():
    """Steps that capture and replay graphs, on four threads at once, while
    the batch that the cases came from is still there."""
    alone, batched = start(), start(graphs=True)
    try:
        b = F.CaseBatch(batched)
        b.step(2)
        assert each(lambda dc: dc.step(5), batched) == []
        c = F.CaseBatch(batched[::-1])  # another first case: the cases' own steps come before its own
        c.step(3)
        for x, y in zip(alone, batched):
            x.step(10)
            for k in FIELDS:
                assert np.array_equal(x.get(k), y.get(k)), k
        b.close()
        c.close()
    finally:
        for dc in alone + batched:
            dc.close()


def test_members_of_a_batch_are_destroyed_by_their_threads():
    alone, batched = start(), start()
    try:
        b = F.CaseBatch(batched)
        b.step(2)
        assert each(lambda dc: dc.close(), batched[1:]) == []
        b.close()
        batched[0].step(2)
        alone[0].step(4)
        for k in FIELDS:
            assert np.array_equal(alone[0].get(k), batched[0].get(k)), k
    finally:
        for dc in alone + batched:
            dc.close()


@pytest.mark.parametrize("given", [0, 1, 2], ids=["first", "one", "all"])
def test_members_on_streams_of_the_caller(given):
    """Cases whose streams the caller gave (the first, another, all of them),
    with the caller's own work on them between the batch's steps."""
    hip = F.lib()  # (its own HIP runtime)
    alone = start()
    streams = [C.c_void_p() for _ in RATIOS]
    for st in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0  # non-blocking
    batched = []
    for q, r in enumerate(RATIOS):
        mine = given == 2 or q == given
        dc = F.DeviceCase(cases.rising_bubble_3d(ng=(32, 16, 24), rho12=(r, 1.0)),
                          stream=streams[q].value if mine else None)
        dc.init()
        dc.step(1)
        batched.append(dc)
    try:
        b = F.CaseBatch(batched)
        b.step(1)
        for _ in range(2):
            for dc in batched[::2]:
                dc.set("p", 1.25 * dc.get("p"))
            b.step(1)
        b.close()
        for dc in alone:
            dc.step(1)
        for _ in range(2):
            for q, dc in enumerate(alone):
                if q % 2 == 0:
                    dc.set("p", 1.25 * dc.get("p"))
                dc.step(1)
        for x, y in zip(alone, batched):
            y.step(1)
            x.step(1)
            for k in FIELDS:
                assert np.array_equal(x.get(k), y.get(k)), k
    finally:
        for dc in alone + batched:
            dc.close()
        for st in streams:
            hip.hipStreamDestroy(st)
