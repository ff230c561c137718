"""The wall force's sum over records by record count: below, at and past its
chunks of 1024 records, against the records' count on one record's term."""
import dataclasses

import numpy as np
import pytest

from code_mge_amd.grid import LevelGeom, body, hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrec", [1, 15, 16, 17, 1023, 1024, 1025, 2048, 3100])
def test_force_is_the_sum_in_record_order(require_gpu, nrec):
    """At the freestream start every record's mirror state follows from its own
    cells, so a level whose records are the body's, dealt out in order and
    repeated, has a force that is the ordered sum of single-record forces:
    equal bits."""
    n = (16, 16, 16)
    levels = hierarchy(n, (0.0, 0.0, 0.0), (0.8, 0.8, 0.8), 1, bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, distype="r1")
    g = level_geometry(levels[0], body("ellipsoid", center=(0.4, 0.4, 0.4), semi=(0.23, 0.21, 0.18)))

    def force(picks):
        recs = (type(g.recs[0]) * len(picks))()
        for m, k in enumerate(picks):
            recs[m] = g.recs[k]
        geom = LevelGeom(g.spec, g.xv, g.yv, g.zv, g.blank, recs, len(picks))
        with Case(dataclasses.replace(prm), levels, geoms=[geom], mxcyc=4) as c:
            c.init_flow()
            c.bc_cutcell(1)
            return np.array(c.wall_force(1))

    one = [force([k]) for k in range(g.nmir)]
    want = np.zeros(3)
    for m in range(nrec):
        want = want + one[m % g.nmir]
    got = force([m % g.nmir for m in range(nrec)])
    print(f"  {nrec} records of {g.nmir}: {got} {want}")
    assert np.array_equal(got, want)
