"""Restriction and prolongation by level shape: the prolongation of eight fine
cells per thread (all directions halved) around its 64 x 4 tile, the general
one where a direction keeps its cells, blank cells, the correction and the
full-multigrid step; call by call against the oracle (FP64) and FP32 against
FP64."""
import dataclasses

import numpy as np
import pytest

from code_mge_amd.grid import body, hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case
from oracle.oracle import OracleCase
from tests.gpu_common import max_rel_to_field, perturbed_state

pytestmark = pytest.mark.gpu

# fine cells; halved in every direction unless odd
SHAPES = [(4, 4, 4), (6, 10, 4), (128, 8, 4), (130, 18, 6), (256, 4, 4), (16, 16, 3), (18, 5, 4), (32, 32, 32),
          (24, 26, 22)]


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("fmg", [False, True])
def test_restrict_relax_prolong(require_gpu, n, fmg):
    """Tolerances: a relaxation leaves up to 1e-13 of a field's largest value,
    the transfers' eight-term sums a few ulp more: 1e-12.  FP32: the same in
    24 bits, 1e-13 * 2^29 = 5e-5, doubled"""
    levels = hierarchy(n, (0.0, 0.0, 0.0), tuple(0.02 * m for m in n), 2, bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, beta_deg=1.0, smoo=0.6)
    bdy = None
    if min(n) >= 22:
        bdy = body("ellipsoid", center=tuple(0.01 * m for m in n), semi=tuple(0.005 * m for m in n))
    geoms = [level_geometry(s, bdy) for s in levels]
    orc = OracleCase(prm, geoms, mxcyc=4)
    got = {}
    for precision in (64, 32):
        with Case(dataclasses.replace(prm, precision=precision), levels, geoms=geoms, mxcyc=4) as gpu:
            gpu.init_flow()
            w, p = perturbed_state(gpu, 2, prm, seed=4)
            runs = [gpu] if precision == 32 else [gpu, orc]
            if precision == 64:
                orc.init_flow()
            for c in runs:
                c.upload(2, "w", w)
                c.upload(2, "p", p)
                c.bc_cutcell(2)
                c.bcond(2)
                c.timestep(2)
                c.euler(2, 1, 2, 2, 1, 0)
                c.movco(1)
                c.timestep(1)
                c.euler(1, 1, 1, 2, 0, 1)
                c.movfin(2, 1 if fmg else 2)
            got[precision] = {(l, f): gpu.download(l, f) for l, f in ((1, "wr"), (1, "w"), (2, "w"), (2, "p"))}
    for (l, f), a in got[64].items():
        e = max_rel_to_field(a, orc.download(l, f))
        e32 = max_rel_to_field(got[32][l, f], a)
        print(f"  {n} level {l} {f}: FP64 {e:.2e}, FP32 {e32:.2e}")
        assert np.isfinite(a).all()
        assert e < 1e-12, (l, f)
        assert e32 < 1e-4, (l, f)
