"""The kernels that large grids run, on small ones: the z-marching forms of the
phase-field step, the normals and the correction, with several planes a block."""
import numpy as np
import pytest

import fizzy_amd as F
import test_gpu_kernels as K
from fizzy_amd import cases

pytestmark = pytest.mark.gpu

FIELDS = ["u", "v", "w", "p", "psi", "kappa", "normx", "normy", "normz", "psiflx_x", "psiflx_y", "psiflx_z"]
MARCHING = {"FZ_ACDI_VARIANT": "3", "FZ_YOUNGS_VARIANT": "3", "FZ_CORREC_MY": "4"}
SPECS = {"bubble": cases.rising_bubble_3d(ng=(72, 20, 40)),
         "walls": dict(cases.hysing_2d(ng=(45, 2, 35)), ng=[45, 13, 35], l=[1.0, 13 / 45, 35 / 45])}


def run(spec, env, monkeypatch):
    for k in list(MARCHING) + ["FZ_MARCH_PLANES"]:
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    dc = F.DeviceCase(spec)
    try:
        dc.init()
        dc.step(8)
        return {k: dc.get(k) for k in FIELDS}, dc.scalars()
    finally:
        dc.close()


@pytest.mark.parametrize("planes", ["1", "3", "16"])
@pytest.mark.parametrize("name", list(SPECS))
def test_marching_kernels_agree_bitwise(name, planes, monkeypatch):
    a, sa = run(SPECS[name], {}, monkeypatch)
    b, sb = run(SPECS[name], dict(MARCHING, FZ_MARCH_PLANES=planes), monkeypatch)
    for k in FIELDS:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(sa, sb)


@pytest.mark.parametrize("seps_cells, raised", [(0.51, False), (2.0 ** 24, True)], ids=["flag-clear", "flag-raised"])
@pytest.mark.parametrize("planes", ["1", "5", "16"])
@pytest.mark.parametrize("variant", ["2", "3"], ids=["one-cell", "marching"])
@pytest.mark.parametrize("shape", K.SHAPES, ids=lambda s: "x".join(map(str, s[0])))
def test_normals_under_the_range_flag(shape, variant, planes, seps_cells, raised, rng, monkeypatch):
    """The one-cell kernel and the check-free marching one with its checked
    twin, each under a clear and a raised flag, against the oracle."""
    monkeypatch.setenv("FZ_YOUNGS_VARIANT", variant)
    monkeypatch.setenv("FZ_MARCH_PLANES", planes)
    n, l, gr = shape
    pair = K.Pair(n, l, "PPPPNN", gr)
    try:
        K.test_youngs_under_the_range_flag(pair, rng, seps_cells, raised)
    finally:
        pair.close()
