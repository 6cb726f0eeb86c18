"""List rows longer than the one-launch step's LDS keys (512 entries).

Such rows are put in order cell by cell instead.  They are the rows of the
per-phase path, so trajectories keep their bits (as in test_gpu_routes.py),
also where a cell holds more particles than a group has lanes; the batch stays on one launch per step, and so does a pool that takes a job
with such rows: the other slots' jobs are those of a pool of one.
"""
import numpy as np
import pytest

from test_gpu_fused import THERMO, _gas
from test_gpu_routes import KEYS, _equal, _final, _run

pytestmark = pytest.mark.gpu

OPTS = dict(dt=0.003, verlet_skin=0.05, refresh_vel=True, **THERMO["langevin"])


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _dense(nx, bp, lz, salt):
    from oxdna_amd import systems
    return systems.duplex_bundle(2, nx=nx, ny=nx, bp=bp, spacing=2.6, lz=lz, tc=30.0, salt=salt)


# rows of 512 entries and around, about 1,000, and long ones from cells of 50 particles
@pytest.mark.parametrize("nx,bp,lz,salt", [(8, 40, 18.5, 0.115), (8, 40, 18.5, 0.08), (12, 66, 28.5, 0.03)])
def test_long_rows_keep_the_bits(hip, monkeypatch, nx, bp, lz, salt):
    s = _dense(nx, bp, lz, salt)
    monkeypatch.setenv("OXH_CELL_BUILD", "0")
    monkeypatch.setenv("OXH_FAR_BACK", "0")
    monkeypatch.setenv("OXH_EDGE", "0")
    got = [_run(hip, monkeypatch, [s], [64, 7], fuse=fuse, pack=1, **THERMO["langevin"]) for fuse in (1, 0)]
    with hip.HIPBatch(s) as b:
        assert b.stats()["mean_neigh"] > 450
    _equal(*got)


def test_a_job_with_long_rows_leaves_the_others_alone(hip):
    jobs = [_gas(1, 30, 20), _dense(8, 30, 14.5, 0.08), _gas(3, 40, 31)]
    steps = [300, 100, 260]
    with hip.HIPPool([4096] * 3) as p:
        for k in (0, 2, 1):
            p.admit(k, jobs[k], steps[k], seed=7 + k, **OPTS)
            assert p.routes()["one_launch"]
            p.run(40)
        assert p.stats()["mean_neigh"] > 400   # two of three jobs have short rows
        p.run(300)
        assert list(p.status()["done"]) == steps
        assert p.routes()["one_launch"]
        mixed = [_final(p, k) for k in range(3)]
    for k in range(3):
        with hip.HIPPool([4096]) as p:
            p.admit(0, jobs[k], steps[k], seed=7 + k, **OPTS)
            p.run(400)
            alone = _final(p, 0)
        for key in KEYS:
            assert np.array_equal(alone[key], mixed[k][key]), (k, key)
