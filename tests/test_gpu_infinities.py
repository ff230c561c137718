"""Infinite values go through the far field and the restriction as through the
reference's divisions and powers: an infinity stays one and becomes no NaN
where the reference has none."""
import numpy as np
import pytest

from code_mge_amd.grid import hierarchy, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case
from oracle.oracle import OracleCase
from tests.gpu_common import perturbed_state

pytestmark = pytest.mark.gpu

INF = np.inf
# component (5 the pressure) and value put into single cells next to the faces
ODD = [(0, INF), (0, 0.0), (0, 1e200), (1, INF), (1, -INF), (2, INF), (3, -INF), (5, INF), (5, 0.0), (0, 1e-300)]


def same_kind(a, b):
    """equal NaNs and infinities; the rest to the far state's rounding (1e-13)"""
    nan = np.isnan(a) == np.isnan(b)
    inf = np.isinf(a) | np.isinf(b)
    ok = nan & np.where(inf, a == b, True)
    fin = np.isfinite(a) & np.isfinite(b)
    return ok & np.where(fin, np.abs(np.where(fin, a - b, 0.0)) <= 1e-13 * (1.0 + np.abs(np.where(fin, b, 0.0))), True)


@pytest.mark.parametrize("gamma", [1.4, 1.3])
def test_far_field(require_gpu, gamma):
    n = (16, 16, 16)
    levels = hierarchy(n, (0.0, 0.0, 0.0), (1.6, 1.6, 1.6), 1, bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, beta_deg=1.0, gamma=gamma)
    geoms = [level_geometry(s, None) for s in levels]
    orc = OracleCase(prm, geoms, mxcyc=4)
    with Case(prm, levels, geoms=geoms, mxcyc=4) as gpu:
        gpu.init_flow()
        orc.init_flow()
        w, p = perturbed_state(gpu, 1, prm, seed=3)
        for f in range(6):          # each face: one odd cell in the middle of every second row
            for m, (c, v) in enumerate(ODD):
                q = [4 + 2 * (m % 5), 6 + 4 * (m // 5), 2 if f < 3 else 17]   # two in the plane, the face's layer
                x = {0: (q[2], q[0], q[1]), 1: (q[0], q[2], q[1]), 2: (q[0], q[1], q[2])}[f % 3]
                (p if c == 5 else w[c])[x[2], x[1], x[0]] = v
        out = []
        with np.errstate(all="ignore"):
            for c in (gpu, orc):
                c.upload(1, "w", w)
                c.upload(1, "p", p)
                c.bcond(1)
                out.append((c.download(1, "w"), c.download(1, "p")))
            (gw, gp), (ow, op) = out
            bad = ~np.concatenate([same_kind(gw, ow), same_kind(gp, op)[None]])
        inner = np.zeros(op.shape, dtype=bool)   # ghost cells with one ghost index
        for ax in range(3):
            g = [slice(2, -2)] * 3
            for s in (slice(0, 2), slice(-2, None)):
                g[ax] = s
                inner[tuple(g)] = True
        bad &= inner
        for b in np.argwhere(bad)[:20]:
            i = tuple(b)
            print("  component, k, j, i", i, gw[i] if i[0] < 5 else gp[i[1:]], ow[i] if i[0] < 5 else op[i[1:]])
        assert not bad.any()


@pytest.mark.parametrize("precision", [64, 32])
def test_restriction(require_gpu, precision):
    n = (16, 16, 16)
    levels = hierarchy(n, (0.0, 0.0, 0.0), (1.6, 1.6, 1.6), 2, bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, precision=precision)
    with Case(prm, levels, geoms=[level_geometry(s, None) for s in levels], mxcyc=4) as c:
        c.init_flow()
        dw = np.zeros((5,) + c.dims(2)[::-1])
        dw[1, 5, 6, 7], dw[3, 10, 10, 10] = INF, -INF
        c.upload(2, "dw", dw)
        c.movco(1)
        wr = c.download(1, "wr")
    assert not np.isnan(wr).any()
    assert np.isposinf(wr[1, 3, 4, 4]) and np.isneginf(wr[3, 6, 6, 6]) and np.isinf(wr).sum() == 2
