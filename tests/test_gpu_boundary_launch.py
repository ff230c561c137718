"""The boundary's launches: the far field's closed forms for air beside the
general powers, and the update, mirror states and faces of a smoothed stage
in one launch, against the oracle."""
import numpy as np
import pytest

from code_mge_amd.grid import body, hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case
from oracle.oracle import OracleCase
from tests.gpu_common import max_rel_to_field, perturbed_state

pytestmark = pytest.mark.gpu

FAR, SYM, PER, WALL = -20, -50, -60, -80


@pytest.mark.parametrize("gamma", [1.4, 1.3])
@pytest.mark.parametrize("n,bct", [((9, 3, 2), (FAR,) * 6), ((22, 17, 12), (FAR, WALL, PER, SYM, FAR, PER))])
def test_one_relaxation_every_cell(require_gpu, gamma, n, bct):
    """one five-stage relaxation from a state with inflow and outflow on every
    far face, ghost cells included.  The tolerance: a far state differs by a
    few ulp between the two sides (1e-15), which one stage's residual, a
    difference of fluxes some hundred times its size, lifts to 1e-13; 1e-12"""
    levels = hierarchy(n, (0.0, 0.0, 0.0), tuple(0.1 * m for m in n), 1, bctype=bct)
    prm = Params(mach=0.4, alpha_deg=3.0, beta_deg=1.0, gamma=gamma)
    bdy = body("sphere", center=tuple(0.05 * m for m in n), semi=(0.25,) * 3) if min(n) > 4 else None
    geoms = [level_geometry(s, bdy) for s in levels]
    orc = OracleCase(prm, geoms, mxcyc=4)
    with Case(prm, levels, geoms=geoms, mxcyc=4) as gpu:
        gpu.init_flow()
        orc.init_flow()
        w, p = perturbed_state(gpu, 1, prm, seed=3, amp=0.02)
        rng = np.random.Generator(np.random.PCG64(4))
        for m in (1, 2, 3):
            w[m] = w[m] + 0.05 * w[0] * rng.uniform(-1.0, 1.0, size=w[0].shape)
        p = (gamma - 1.0) * (w[4] - 0.5 * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) / w[0])
        for c in (gpu, orc):
            c.upload(1, "w", w)
            c.upload(1, "p", p)
            c.bcond(1)
            c.bc_cutcell(1)
            c.timestep(1)
            c.euler(1, 1, 1, 1, 0, 0)
        for f in ("w", "p"):
            e = max_rel_to_field(gpu.download(1, f), orc.download(1, f))
            print(f"  {f}: {e:.3e}")
            assert e < 1e-12, f
