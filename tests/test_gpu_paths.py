"""Launch shapes chosen from the grid give the fields of any other choice.

The z-marching kernels (momentum, ACDI step, correction, normals) take their
planes per block from the grid; FZ_MARCH_PLANES, read when a context is made,
fixes the number. Every number gives the same fields bit for bit."""
import numpy as np
import pytest

import fizzy_amd as F
from fizzy_amd import cases

pytestmark = pytest.mark.gpu

FIELDS = ["u", "v", "w", "p", "psi", "kappa"]
BUBBLE = cases.rising_bubble_3d(ng=(72, 20, 40))
SPECS = {"fp64": BUBBLE, "mixed": dict(BUBBLE, precision="mixed", refine=1),
         "two-d": cases.hysing_2d(ng=(32, 2, 33)), "droplets": cases.vof_droplets(ng=(32, 24, 18), ndrop=2, r=0.6)}


def run(spec, nsteps, planes, monkeypatch):
    if planes:
        monkeypatch.setenv("FZ_MARCH_PLANES", str(planes))
    else:
        monkeypatch.delenv("FZ_MARCH_PLANES", raising=False)
    dc = F.DeviceCase(spec)
    try:
        dc.init()
        dc.step(nsteps)
        return {k: dc.get(k) for k in FIELDS}, dc.scalars()
    finally:
        dc.close()


@pytest.mark.parametrize("planes", [1, 3, 16, 64])
@pytest.mark.parametrize("name", list(SPECS))
def test_planes_per_block_agree_bitwise(name, planes, monkeypatch):
    a, sa = run(SPECS[name], 8, 0, monkeypatch)
    b, sb = run(SPECS[name], 8, planes, monkeypatch)
    for k in FIELDS:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(sa, sb)
