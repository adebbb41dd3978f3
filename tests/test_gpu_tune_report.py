"""The autotuner's report names the z solve that the case runs."""
import re

import pytest

import fizzy_amd as F
from fizzy_amd import cases

pytestmark = pytest.mark.gpu

THIN = dict(cases.rising_bubble_3d(ng=(512, 512, 3)), l=[1.0, 1.0, 3.0 / 512])


@pytest.mark.parametrize("spec, kinds, rows", [
    # a periodic z has one form for each number of rows
    (cases.vof_droplets(ng=(16, 16, 20), ndrop=1, r=0.6), ["registers"], [16]),
    (cases.vof_droplets(ng=(8, 8, 270), ndrop=1, r=0.6), ["registers"], [32]),
    (cases.vof_droplets(ng=(16, 16, 8), ndrop=1, r=0.6), ["chunks"], [16]),
    # pivots made at set-up: the columns in registers or the chunks that were faster
    (cases.rising_bubble_3d(ng=(16, 16, 32)), ["registers", "setup_pivots"], [8, 16]),
    # from 512x512 columns on, with or without a pivot array
    (THIN, ["no_pivots", "chunks"], [8, 16, 32]),
    (dict(THIN, precision="mixed"), ["no_pivots", "chunks", "pairs"], [8, 16, 32]),
], ids=["periodic", "periodic long", "periodic short", "walls", "columns", "fp32 columns"])
def test_report_names_the_z_solve(spec, kinds, rows):
    dc = F.DeviceCase(spec)
    try:
        dc.init()
        for cached in ("", " (cached)"):
            rep = dc.autotune(1)
            print(rep)
            m = re.match(r"tile_y=\d+ mom_variant=\d+ thomas_rows=(\d+)(x2|rc|) ms_per_step=[0-9.]+ thomas=(\w+)(.*)", rep)
            assert m and int(m.group(1)) in rows and m.group(3) in kinds and m.group(4) == cached
            assert m.group(2) == {"pairs": "x2", "no_pivots": "rc"}.get(m.group(3), "")
        dc.step(1)
        dc.sync()
    finally:
        dc.close()
