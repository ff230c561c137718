"""Fields of more pieces than the transfer ring has places (and a ragged last
one), both ways, from one thread and from several."""
import threading

import pytest

from tests.test_gpu_transfer import _check, _round_trip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [((120, 110, 100), 64), ((150, 130, 120), 32)])
def test_ring_reuse(require_gpu, n, precision):
    out = {}
    _round_trip(n, precision, 1, out)
    _check(*out[1])


def test_ring_reuse_from_threads(require_gpu):
    """six threads: more than there are rings"""
    out = {}
    ts = [threading.Thread(target=_round_trip, args=((110 + k, 100, 90), 64 if k % 2 else 32, k, out)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert len(out) == 6
    for v in out.values():
        _check(*v)
