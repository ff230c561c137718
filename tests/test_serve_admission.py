"""Admission without a GPU: the launch shapes are timed for a request that is
admitted alone, and not for one that joins others, whose batch would not take
them."""
import threading

import pytest

from code_mge_amd import configs, serve


class FakeCase:
    tuned = 0

    def __init__(self, prm, levels, geoms, mxcyc):
        pass

    def init_flow(self):
        pass

    def autotune(self):
        FakeCase.tuned += 1

    def device_bytes(self):
        return 1000


@pytest.mark.parametrize("autotune", [True, False])
def test_timing_at_admission(monkeypatch, autotune):
    monkeypatch.setattr(serve, "Case", FakeCase)
    FakeCase.tuned = 0
    prm, levels, bdy, aref = configs.sphere3d(n=16, nlevel=2, box=4.0)
    srv = serve.Server(hbm_budget=1e12, autotune=autotune)
    srv._cv, srv._ready, srv._stop, srv._resident = threading.Condition(), [], False, 0
    counts = []
    for rid in range(3):
        req, case, got = srv._prepare(serve.Request(rid, 0.0, prm, levels, bdy, aref))
        counts.append(FakeCase.tuned)
        assert got == 1000 and isinstance(case, FakeCase)
    assert srv._resident == 3 and srv.used == 3000
    assert counts == ([1, 1, 1] if autotune else [0, 0, 0])
    srv._resident = 0   # all served
    srv._prepare(serve.Request(3, 0.0, prm, levels, bdy, aref))
    assert FakeCase.tuned == (2 if autotune else 0)
