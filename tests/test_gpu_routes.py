"""Which kernels a batch's steps take, and that the choice leaves no trace.

`routes()` says whether steps take one launch each; the comparisons of
test_gpu_fused.py are between two paths only if it differs between them, here
for the same systems.  A trajectory has the same bits whichever path its steps
take, whether the close pairs are evaluated packed or in place, and however a
run is cut into calls (a chunk's first and last half steps are kernels of their
own): bit for bit, since a pool's slots and a restored checkpoint rely on it.
"""
import numpy as np
import pytest

from test_gpu_fused import THERMO, _gas

pytestmark = pytest.mark.gpu

KEYS = ("pos", "a1", "a3", "vel", "L", "F", "T")


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _final(b, k):
    F, T, _ = b.forces(k)
    return dict(b.state(k), F=F, T=T)


def _run(hip, monkeypatch, ss, steps, fuse=1, pack=0, lanes=8, **opts):
    monkeypatch.setenv("OXH_FUSE", str(fuse))
    monkeypatch.setenv("OXH_PACK", str(pack))
    monkeypatch.setenv("OXH_PERSIST", "0")
    monkeypatch.setenv("OXH_FORCE_LANES", str(lanes))
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    per = [dict(seed=100 + k) for k in range(len(ss))]
    with hip.HIPBatch(ss, options=per, dt=0.003, verlet_skin=0.05, refresh_vel=True, **opts) as b:
        assert b.routes()["one_launch"] == bool(fuse)
        for n in steps:
            b.run(n)
        assert b.routes()["one_launch"] == bool(fuse)
        return [_final(b, k) for k in range(len(ss))]


def _equal(x, y):
    for a, b in zip(x, y):
        for key in KEYS:
            assert np.array_equal(a[key], b[key]), (key, np.abs(a[key] - b[key]).max())


@pytest.mark.parametrize("thermo", list(THERMO))
@pytest.mark.parametrize("sizes", [[(1, 5)], [(31, 19)], [(1, 9), (33, 17), (4, 21)]])
def test_same_bits_on_every_path(hip, monkeypatch, thermo, sizes):
    ss = [_gas(5 + k, n, bp) for k, (n, bp) in enumerate(sizes)]
    want = _run(hip, monkeypatch, ss, [130], **THERMO[thermo])
    _equal(want, _run(hip, monkeypatch, ss, [37, 1, 20, 72], **THERMO[thermo]))
    _equal(want, _run(hip, monkeypatch, ss, [130], pack=1, **THERMO[thermo]))
    _equal(want, _run(hip, monkeypatch, ss, [130], fuse=0, **THERMO[thermo]))
    _equal(want, _run(hip, monkeypatch, ss, [65, 65], fuse=0, pack=1, **THERMO[thermo]))


@pytest.mark.parametrize("lanes", [2, 4, 16, 32])
def test_same_bits_for_other_lanes(hip, monkeypatch, lanes):
    ss = [_gas(5, 1, 9), _gas(6, 33, 17), _gas(7, 7, 13)]
    want = _run(hip, monkeypatch, ss, [96], lanes=lanes, **THERMO["langevin"])
    _equal(want, _run(hip, monkeypatch, ss, [31, 65], lanes=lanes, pack=1, **THERMO["langevin"]))
    _equal(want, _run(hip, monkeypatch, ss, [96], lanes=lanes, fuse=0, **THERMO["langevin"]))


def test_paths_that_are_not_one_launch(hip, monkeypatch):
    s = _gas(3, 30, 20)
    with hip.HIPBatch(s, backend_precision="double") as b:
        assert not b.routes()["one_launch"]
    with hip.HIPBatch(_gas(3, 1, 9)) as b:      # workgroup engine
        assert not b.routes()["one_launch"]
    monkeypatch.setenv("OXH_FORCE_LANES", "8")
    monkeypatch.setenv("OXH_FAR_LANES", "8")
    with hip.HIPBatch(s) as b:
        assert not b.routes()["one_launch"]
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    with hip.HIPBatch(s) as b:
        assert b.routes()["one_launch"]
        b.set_external_forces([dict(type="trap", particle=0, stiff=1.0, pos0=s.pos[0], dir=(0.0, 0.0, 1.0))])
        assert not b.routes()["one_launch"]


def test_second_buffers_only_while_steps_use_them(hip, monkeypatch):
    """Device bytes held, against a batch that never takes one launch per step."""
    s = _gas(3, 100, 20)
    monkeypatch.setenv("OXH_FORCE_LANES", "8")

    def held(fuse, far):
        monkeypatch.setenv("OXH_FUSE", str(fuse))
        monkeypatch.setenv("OXH_FAR_LANES", str(far))
        return hip.HIPBatch(s, dt=0.003, verlet_skin=0.05, seed=3, **THERMO["langevin"])

    with held(0, 0) as b:
        base = b.stats()["device_bytes"]
        b.run(120)
        want = _final(b, 0)
    with held(1, 8) as b:
        assert b.stats()["device_bytes"] == base
    with held(1, 0) as b:
        used = b.stats()["device_bytes"]
        assert used >= base + 112 * s.N
        b.run(40)
        ck = b.checkpoint()
        b.set_external_forces([dict(type="trap", particle=0, stiff=1.0, pos0=s.pos[0], dir=(0.0, 0.0, 1.0))])
        less = b.stats()["device_bytes"]
        assert less < used - 112 * s.N
        b.run(10)
        b.set_external_forces([])
        b.restore(ck)
        b.run(80)
        assert b.routes()["one_launch"] and b.stats()["device_bytes"] >= used
        got = _final(b, 0)
    for key in KEYS:
        assert np.array_equal(want[key], got[key]), key


@pytest.mark.parametrize("lanes", [None, 1, 2])
def test_packed_form_of_pools(hip, monkeypatch, lanes):
    """OXH_PACK=0 and one lane per nucleotide keep a pool in place; the bits are those of the packed form."""
    jobs = [_gas(1, 30, 20), _gas(2, 3, 11), _gas(3, 9, 31)]
    if lanes:
        monkeypatch.setenv("OXH_FORCE_LANES", str(lanes))
    got = []
    for pack in (1, 0, None):
        if pack is None:
            monkeypatch.delenv("OXH_PACK")
        else:
            monkeypatch.setenv("OXH_PACK", str(pack))
        with hip.HIPPool([2048] * 3) as p:
            assert p.stats()["pack"] == (lanes != 1 and pack != 0)
            for k, s in enumerate(jobs):
                p.admit(k, s, 60 + 20 * k, seed=7 + k, dt=0.003, verlet_skin=0.05, refresh_vel=True, **THERMO["langevin"])
            p.run(120)
            got.append([_final(p, k) for k in range(3)])
    _equal(got[0], got[1])
    _equal(got[0], got[2])


def test_packed_form_is_reported_only_where_there_is_one(hip, monkeypatch):
    from test_gpu_rna import load_rna
    monkeypatch.setenv("OXH_PACK", "1")
    with hip.HIPPool([256] * 2) as p:   # workgroup engine
        assert p.stats()["engine"] == "workgroup" and not p.stats()["pack"]
    monkeypatch.setenv("OXH_FORCE_LANES", "4")
    s, opts, _ = load_rna("rna_ff16_nohb")
    with hip.HIPBatch(s, **opts) as b:
        assert not b.stats()["pack"]
    monkeypatch.setenv("OXH_PERSIST", "0")
    with hip.HIPBatch(_gas(3, 30, 20), backend_precision="double") as b:
        assert not b.stats()["pack"]
