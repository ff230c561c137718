"""An error that other code of the thread left with the HIP runtime (here a
device number that does not exist) is not the library's: its calls go on."""
import ctypes

import pytest

from code_mge_amd import _ffi, configs
from code_mge_amd.solver import Case

pytestmark = pytest.mark.gpu


def test_calls_after_another_callers_error(require_gpu):
    hip = _ffi.lib().hipSetDevice   # the runtime the library is linked with
    hip.argtypes, hip.restype = [ctypes.c_int], ctypes.c_int
    prm, levels, bdy, _ = configs.cylinder2d(n=16, nz=2, nlevel=1, ffreeze=1e3)
    try:
        with Case(prm, levels, body=bdy, mxcyc=4) as c:
            c.init_flow()
            for call in (c.sync, lambda: c.cycles(1, 1), lambda: c.download(1, "w"), lambda: c.euler(1, 1, 1, 1, 0, 0),
                         lambda: c.upload_solut(1), lambda: c.upload_solut(1, noalloc=True), lambda: c.wall_force(1),
                         lambda: c.autotune(), lambda: c.bcond(1)):
                assert hip(1 << 20) != 0
                call()
    finally:
        _ffi.lib().hipGetLastError()
