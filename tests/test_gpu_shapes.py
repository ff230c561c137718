"""Launch shapes the library picks itself: a batch takes one stage-kernel
shape per level for all its cases, a shape forced on a case stays, and
neither changes a bit of any case's result."""
import numpy as np
import pytest

from code_mge_amd import configs
from code_mge_amd.grid import level_geometry
from code_mge_amd.solver import Batch, Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("distype,precision", [("c", 64), ("r2", 32)])
def test_batch_shape_with_tuned_forced_and_plain_cases(require_gpu, distype, precision):
    """one tuned, one forced and one plain case of different sizes, alone and
    in one batch: the same state and residual history"""
    alone, together = [], []
    for n, mode in ((24, "tuned"), (40, "forced"), (32, "plain")):
        prm, levels, bdy, _ = configs.ellipsoid3d(n=n, nlevel=3, semi=(0.9, 0.6, 0.5), box=4.0, mach=0.4,
                                                  alpha=3.0, distype=distype, precision=precision)
        geoms = [level_geometry(s, bdy) for s in levels]
        with Case(prm, levels, geoms=geoms, mxcyc=8) as c:
            c.init_flow()
            # a batch runs cycles on the finest level, with no full-multigrid start
            res = [c.cycles(3, 1, ncyc0=k)[0] for k in range(1, 7)]
            alone.append((np.array(res), c.download(3, "w")))
        c = Case(prm, levels, geoms=geoms, mxcyc=8)
        if mode == "forced":
            for lvl in (1, 2, 3):
                c.set_tile(lvl, 8, 3)
        c.init_flow()
        if mode == "tuned":
            c.autotune()
        together.append((mode, c))
    with Batch(log_cap=8) as b:
        slots = [b.add(c, 1e30, 6) for _, c in together]
        while b.run(2):
            pass
        logs = [b.log(s, cap=8) for s in slots]
    for (mode, c), lg, (la, wa) in zip(together, logs, alone):
        if mode == "forced":
            assert all(c.stage_tile(lvl) == (8, 3) for lvl in (1, 2, 3))
        assert np.array_equal(lg, la)
        assert np.array_equal(c.download(3, "w"), wa)
        c.close()
