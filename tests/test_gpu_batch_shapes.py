"""The stage launch shapes a batch's program takes: one per level for the cases
whose shape the library picks, tuned or not, and its own for a case whose
caller forced one."""
import pytest

from code_mge_amd import _ffi, configs
from code_mge_amd.solver import Batch, Case

pytestmark = pytest.mark.gpu


def make(n, mode, distype, precision):
    prm, levels, bdy, _ = configs.ellipsoid3d(n=n, nlevel=3, semi=(0.9, 0.6, 0.5), box=4.0, mach=0.4, alpha=3.0,
                                              distype=distype, precision=precision)
    c = Case(prm, levels, body=bdy, mxcyc=8)
    c.init_flow()
    for lvl in (1, 2, 3):
        if mode == "forced":
            c.set_tile(lvl, 8, 3)
        elif mode == "forced chunk":
            c.set_kc(lvl, 5)
    if mode in ("tuned", "tuned, chunk given back"):
        c.autotune()
    if mode == "tuned, chunk given back":
        for lvl in (1, 2, 3):
            c.set_kc(lvl, 5)
            c.set_kc(lvl, 0)
    return c


def run_batch(modes, distype, precision, n=24):
    """the modes' cases in one batch: their shapes by level, alone and in it"""
    cases = [make(n + 8 * k, m, distype, precision) for k, m in enumerate(modes)]
    alone = [[c.stage_tile(lvl) for lvl in (1, 2, 3)] for c in cases]
    with Batch(log_cap=8) as b:
        slots = [b.add(c, 1e30, 4) for c in cases]
        with pytest.raises(_ffi.MgeError):   # no program yet
            b.stage_tile(slots[0], 1)
        b.run(1)
        got = [[b.stage_tile(s, lvl) for lvl in (1, 2, 3)] for s in slots]
        with pytest.raises(_ffi.MgeError):
            b.stage_tile(slots[-1] + 1, 1)
    for c in cases:
        c.close()
    return got, alone


@pytest.mark.parametrize("distype,precision", [("c", 64), ("r2", 32)])
def test_common_and_forced_shapes(require_gpu, distype, precision):
    got, alone = run_batch(["tuned", "forced", "plain", "forced chunk"], distype, precision)
    print(got, alone)
    assert got[0] == got[2]
    assert got[1] == alone[1] and all(s == (8, 3) for s in got[1])
    assert got[3] == alone[3] and all(kc == min(5, n) for (_, kc), n in zip(got[3], (12, 24, 48)))


def test_given_back_chunk_is_not_forced(require_gpu):
    """a chunk length forced and given back (0) leaves the level to the library,
    tuned rows or not: the batch's common shape"""
    got, _ = run_batch(["plain", "tuned, chunk given back", "plain"], "r2", 32)
    print(got)
    assert got[0] == got[1] == got[2]


@pytest.mark.parametrize("distype,precision", [("c", 64), ("r2", 64), ("c", 32), ("r2", 32)])
def test_single_case_keeps_its_shape(require_gpu, distype, precision):
    """what was timed for the case, where that is not the library's pick either"""
    for n in (24, 32, 40, 64):
        plain, _ = run_batch(["plain"], distype, precision, n)
        got, alone = run_batch(["tuned"], distype, precision, n)
        print(n, "plain", plain, "tuned", alone)
        assert got == alone
