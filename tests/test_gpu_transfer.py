"""Field transfers between the host and a case through the pinned ring: small
(the caller's thread alone), several pieces (threads), a ragged last piece,
both directions and precisions, and from several threads at once."""
import threading

import numpy as np
import pytest

from code_mge_amd.grid import LevelSpec, level_geometry
from code_mge_amd.params import Params
from code_mge_amd.solver import Case

pytestmark = pytest.mark.gpu


def _case(n, precision):
    spec = LevelSpec(n=n, lo=(0.0, 0.0, 0.0), hi=(1.0, 1.0, 1.0), ratio=(2, 2, 2), bctype=(-20,) * 6)
    prm = Params(mach=0.4, alpha_deg=3.0, precision=precision)
    return Case(prm, [spec], geoms=[level_geometry(spec, None)], mxcyc=4), prm


def _round_trip(n, precision, seed, out):
    c, prm = _case(n, precision)
    rng = np.random.Generator(np.random.PCG64(seed))
    d = prm.derived()
    base = np.array([d["rho0"], d["rho0"] * d["u0"], d["rho0"] * d["v0"], d["rho0"] * d["w0"],
                     d["rho0"] * d["h0"] - d["p0"]])
    dev = rng.uniform(-0.5, 0.5, size=(5,) + c.dims(1)[::-1]).astype(np.float32).astype(np.float64)
    w = base[:, None, None, None] + dev
    q = rng.uniform(-1.0, 1.0, size=w.shape).astype(np.float32).astype(np.float64)
    c.init_flow()
    c.upload(1, "w", w)
    c.upload(1, "dw", q)
    out[seed] = (w, q, c.download(1, "w"), c.download(1, "dw"), precision, base)
    c.close()


def _check(w, q, w2, q2, precision, base):
    assert np.array_equal(q2, q)   # values of FP32 precision: exact either way
    if precision == 64:
        assert np.array_equal(w2, w)
    else:
        # the FP32 state is the deviation from the freestream: its rounding,
        # 2^-24 of at most 0.5, and the freestream's own FP32 rounding
        tol = 0.5 * 2.0 ** -24 + 2.0 * np.abs(base).max() * 2.0 ** -24
        assert np.abs(w2 - w).max() <= tol


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", [(3, 2, 2), (33, 31, 29), (70, 64, 61)])
def test_round_trip(require_gpu, n, precision):
    out = {}
    _round_trip(n, precision, 1, out)
    _check(*out[1])


def test_round_trips_from_threads(require_gpu):
    out = {}
    ts = [threading.Thread(target=_round_trip, args=((60, 50 + k, 40), 64 if k % 2 else 32, k, out)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(out) == 4
    for v in out.values():
        _check(*v)
