"""The residual smoothing's kernels by line length: planes held whole in LDS,
x rows and y/z lines in segments (lengths around every change of segment
length, kernel and thread count) and the sequential sweeps beyond 512 cells,
with blank cells inside lines where a body fits; one relaxation against the
oracle (FP64) and FP32 against FP64."""
import dataclasses

import numpy as np
import pytest

from code_mge_amd.grid import body, hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case
from oracle.oracle import OracleCase
from tests.gpu_common import max_rel_to_field, perturbed_state

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 4, 5), (8, 9, 16), (16, 17, 8), (17, 16, 33), (33, 70, 4), (64, 65, 17), (64, 69, 3),
          (127, 12, 129), (128, 128, 2), (129, 40, 3), (256, 5, 130), (257, 17, 2), (3, 257, 256), (2, 512, 300),
          (512, 3, 2), (513, 3, 2), (2, 513, 2), (3, 2, 513), (40, 36, 32)]


@pytest.mark.parametrize("n", SHAPES)
def test_one_smoothed_relaxation(require_gpu, n):
    """Tolerances: a relaxation's residual carries the fluxes' rounding, up to
    1e-13 of its largest value; the sweeps contract and add a few ulp: 1e-12.
    FP32: the same fluxes in 24 bits, 1e-13 * 2^29 = 5e-5, doubled"""
    levels = hierarchy(n, (0.0, 0.0, 0.0), tuple(0.01 * m for m in n), 1, bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, beta_deg=1.0, smoo=0.6)
    bdy = body("ellipsoid", center=tuple(0.005 * m for m in n), semi=tuple(0.0025 * m for m in n)) if min(n) >= 12 else None
    geoms = [level_geometry(s, bdy) for s in levels]
    orc = OracleCase(prm, geoms, mxcyc=4)
    got = {}
    for precision in (64, 32):
        with Case(dataclasses.replace(prm, precision=precision), levels, geoms=geoms, mxcyc=4) as gpu:
            gpu.init_flow()
            w, p = perturbed_state(gpu, 1, prm, seed=11)
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
    print(f"  {n} nmir {geoms[0].nmir}: FP64 {e:.2e}, FP32 {e32:.2e}")
    assert e < 1e-12
    assert e32 < 1e-4
