"""A checkpoint carries the form of the kernels that wrote it.

A batch restored from one takes the same kernels (packed or in-place close
pairs, one launch per step or one per phase), whatever it was created with, and
goes on bit for bit.  Files of before the field existed (0 in its place) leave
the batch as it is.
"""
import numpy as np
import pytest

from test_gpu_fused import THERMO, _gas
from test_gpu_routes import KEYS, _final

pytestmark = pytest.mark.gpu

OPTS = dict(dt=0.003, verlet_skin=0.05, seed=3, **THERMO["langevin"])
FORM_AT = 76   # of the header: 8 bytes of magic, 4 ints, 3 long longs, 7 ints


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _batch(hip, monkeypatch, pack, fuse):
    monkeypatch.setenv("OXH_PERSIST", "0")
    monkeypatch.setenv("OXH_FORCE_LANES", "8")
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    monkeypatch.setenv("OXH_PACK", str(pack))
    monkeypatch.setenv("OXH_FUSE", str(fuse))
    return hip.HIPBatch(_gas(5, 40, 17), **OPTS)


@pytest.mark.parametrize("pack,fuse", [(0, 1), (1, 0), (1, 1), (0, 0)])
def test_restored_batch_takes_the_same_kernels(hip, monkeypatch, pack, fuse):
    with _batch(hip, monkeypatch, pack, fuse) as a:
        a.run(70)
        ck = a.checkpoint()
        a.run(90)
        want = _final(a, 0)
    assert int.from_bytes(ck[FORM_AT:FORM_AT + 4], "little") != 0
    with _batch(hip, monkeypatch, 1 - pack, 1 - fuse) as b:
        b.run(3)
        b.restore(ck)
        assert b.stats()["pack"] == bool(pack) and b.routes()["one_launch"] == bool(fuse)
        b.run(90)
        got = _final(b, 0)
    for key in KEYS:
        assert np.array_equal(want[key], got[key]), key


def test_files_without_the_field(hip, monkeypatch):
    with _batch(hip, monkeypatch, 1, 1) as a:
        a.run(70)
        ck = bytearray(a.checkpoint())
        a.run(20)
        want = _final(a, 0)
    ck[FORM_AT:FORM_AT + 4] = bytes(4)
    with _batch(hip, monkeypatch, 0, 0) as b:
        b.restore(bytes(ck))
        assert not b.stats()["pack"] and not b.routes()["one_launch"]
        b.run(20)
        got = _final(b, 0)
    for key in KEYS:
        assert np.array_equal(want[key], got[key]), key
