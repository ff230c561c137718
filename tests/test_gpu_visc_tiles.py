"""The viscous flux kernel by block size: remainders of its 16 x 4 x 4 tiles,
levels thinner than a tile, blank cells and wall records at tile edges, and
more wall records in one tile than the block has threads; one relaxation
against the oracle (FP64) and FP32 against FP64."""
import dataclasses

import numpy as np
import pytest

from code_mge_amd.grid import LevelGeom, body, hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case
from oracle.oracle import OracleCase
from tests.gpu_common import max_rel_to_field, perturbed_state

pytestmark = pytest.mark.gpu

# cells, repeats of the wall records
SHAPES = [((2, 2, 2), 1), ((3, 4, 5), 1), ((16, 4, 4), 1), ((17, 5, 5), 1), ((15, 3, 3), 1), ((33, 9, 8), 1),
          ((16, 16, 16), 1), ((18, 13, 14), 1), ((40, 22, 19), 1), ((48, 48, 2), 1), ((32, 20, 20), 3)]


@pytest.mark.parametrize("n,rep", SHAPES)
def test_one_viscous_relaxation(require_gpu, n, rep):
    """Tolerances: the fluxes' rounding is up to 1e-13 of the residual's
    largest value; quotients by widths keep their last bit or the next one,
    and a cell's record sum is added in the same order: 1e-12.  FP32: the
    same fluxes in 24 bits, 1e-13 * 2^29 = 5e-5, doubled"""
    h = 0.05
    levels = hierarchy(n, (0.0, 0.0, 0.0), tuple(h * m for m in n), 1, bctype=(-20,) * 6)
    prm = Params(mach=0.3, alpha_deg=3.0, beta_deg=1.0, eqntype="n", reynolds=20.0)
    bdy = None
    if min(n) >= 8:
        center, semi = tuple(0.5 * m for m in n), tuple(min(0.3 * m, 5.0) for m in n)
        if rep > 1:   # a thin plate: both of its sides in one tile
            center, semi = (24.0, 10.5, 12.0), (12.0, 1.1, 5.0)
        bdy = body("ellipsoid", center=tuple(h * c for c in center), semi=tuple(h * c for c in semi))
    g = level_geometry(levels[0], bdy)
    if rep > 1:
        recs = (type(g.recs[0]) * (g.nmir * rep))()
        for m in range(g.nmir * rep):
            recs[m] = g.recs[m % g.nmir]
        g = LevelGeom(g.spec, g.xv, g.yv, g.zv, g.blank, recs, g.nmir * rep)
        count = {}
        for r in recs:
            t = tuple((c - 2) // s for c, s in zip(r.ccid, (16, 4, 4)))
            count[t] = count.get(t, 0) + 1
        assert max(count.values()) > 320
    geoms = [g]
    orc = OracleCase(prm, geoms, mxcyc=4)
    got = {}
    for precision in (64, 32):
        with Case(dataclasses.replace(prm, precision=precision), levels, geoms=geoms, mxcyc=4) as gpu:
            gpu.init_flow()
            w, p = perturbed_state(gpu, 1, prm, seed=3)
            runs = [gpu] if precision == 32 else [gpu, orc]
            if precision == 64:
                orc.init_flow()
            for c in runs:
                c.upload(1, "w", w)
                c.upload(1, "p", p)
                c.bcond(1)
                c.bc_cutcell(1)
                c.timestep(1)
                c.euler(1, 1, 1, 1, 0, 0)
            got[precision] = gpu.download(1, "dw")
    e = max_rel_to_field(got[64], orc.download(1, "dw"))
    e32 = max_rel_to_field(got[32], got[64])
    print(f"  {n} nmir {g.nmir}: FP64 {e:.2e}, FP32 {e32:.2e}")
    assert np.isfinite(got[64]).all()
    assert e < 1e-12
    assert e32 < 1e-4
