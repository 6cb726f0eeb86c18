"""One launch per MD step against one kernel per phase (OXH_FUSE=0).

The two paths run the same per-particle functions on the same lists, so
trajectories agree to FP32 rounding of the torque sums (the compiler may fuse
multiply-adds differently in the two kernels): 1e-6 after up to 130 steps, the
engines' bar, with the same number of list builds.  Sizes: below and above one
workgroup, without cells and with full-size cells, an uneven batch of both;
step counts that leave a whole chunk, a partial one, a single step and odd and
even numbers of buffer exchanges; every thermostat (Bussi's activations break
the chain of launches); slot pools whose jobs end inside a chunk.  A dense
system whose rows are longer than the step kernel sorts goes back to one
kernel per phase within the run.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THERMO = {
    "langevin": dict(thermostat="langevin", diff_coeff=2.5),
    "bussi": dict(thermostat="bussi", newtonian_steps=10, bussi_tau=100),
    "brownian": dict(thermostat="john", diff_coeff=2.5, newtonian_steps=7),
    "nve": dict(thermostat="no"),
}


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _gas(seed, n, bp, tc=40.0):
    from oxdna_amd import systems
    rng = np.random.default_rng(seed)
    b = systems._Builder()
    side = int(np.ceil(n ** (1.0 / 3.0)))
    a = max(12.0, 0.4 * bp + 4.0)
    for k in range(n):
        c = (np.array([k % side, k // side % side, k // side ** 2]) + 0.5) * a
        systems.add_duplex(b, rng.integers(0, 4, bp), c, systems.random_rotation(rng))
    return b.build([side * a] * 3, "gas", T=systems.celsius(tc), salt=0.5)


def _run(hip, monkeypatch, ss, fuse, steps, **opts):
    monkeypatch.setenv("OXH_FUSE", str(fuse))
    monkeypatch.setenv("OXH_PERSIST", "0")
    monkeypatch.setenv("OXH_FORCE_LANES", "8")
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    per = [dict(seed=100 + k) for k in range(len(ss))]
    with hip.HIPBatch(ss, options=per, dt=0.003, verlet_skin=0.05, refresh_vel=True, **opts) as b:
        for n in steps:
            b.run(n)
        return [dict(b.state(k), F=b.forces(k)[0], rebuilds=b.info(k)[0]) for k in range(len(ss))]


def _agree(x, y, tol=1e-6):
    for a, b in zip(x, y):
        assert a["rebuilds"] == b["rebuilds"]
        for key in ("pos", "a1", "a3", "vel", "L"):
            assert np.abs(a[key] - b[key]).max() <= tol, (key, np.abs(a[key] - b[key]).max())
        assert np.abs(a["F"] - b["F"]).max() <= 1e-5 * np.abs(b["F"]).max()


@pytest.mark.parametrize("thermo", list(THERMO))
@pytest.mark.parametrize("sizes", [[(1, 5)], [(7, 13)], [(31, 19)], [(1, 9), (33, 17), (4, 21)]])
def test_one_launch_per_step_agrees(hip, monkeypatch, thermo, sizes):
    ss = [_gas(5 + k, n, bp) for k, (n, bp) in enumerate(sizes)]
    for steps in ([64], [130], [37, 1, 20]):
        _agree(_run(hip, monkeypatch, ss, 1, steps, **THERMO[thermo]), _run(hip, monkeypatch, ss, 0, steps, **THERMO[thermo]))


@pytest.mark.parametrize("pack", [0, 1])
def test_packed_and_in_place(hip, monkeypatch, pack):
    monkeypatch.setenv("OXH_PACK", str(pack))
    ss = [_gas(3, 30, 20), _gas(4, 3, 11)]
    _agree(_run(hip, monkeypatch, ss, 1, [96], **THERMO["langevin"]), _run(hip, monkeypatch, ss, 0, [96], **THERMO["langevin"]))


def test_pool_jobs_that_end_inside_a_chunk(hip, monkeypatch):
    ss = [_gas(1, 2, 16), _gas(2, 30, 20), _gas(3, 9, 31)]
    steps = [23, 129, 64]
    got = []
    for fuse in (1, 0):
        monkeypatch.setenv("OXH_FUSE", str(fuse))
        with hip.HIPPool([2048] * 4) as p:
            for k, (s, n) in enumerate(zip(ss, steps)):
                p.admit(k, s, n, dt=0.003, verlet_skin=0.05, refresh_vel=True, seed=7 + k, **THERMO["langevin"])
            p.run(40)
            p.run(200)
            assert list(p.status()["done"][:3]) == steps
            got.append([dict(p.state(k), F=p.forces(k)[0], rebuilds=p.info(k)[0]) for k in range(3)])
    _agree(*got)


def test_rows_longer_than_the_step_kernel_sorts(hip, monkeypatch):
    from oxdna_amd import systems
    s = systems.duplex_bundle(2, nx=8, ny=8, bp=40, spacing=2.6, lz=18.5, tc=30.0, salt=0.08)
    monkeypatch.setenv("OXH_CELL_BUILD", "0")
    monkeypatch.setenv("OXH_FAR_BACK", "0")
    monkeypatch.setenv("OXH_EDGE", "0")
    got = []
    for fuse in (1, 0):
        got.append(_run(hip, monkeypatch, [s], fuse, [64, 10], **THERMO["langevin"]))
    monkeypatch.setenv("OXH_FUSE", "0")
    with hip.HIPBatch(s) as b:
        assert b.stats()["mean_neigh"] > 512   # the case this test is for
    _agree(*got)


@pytest.mark.parametrize("lanes", [2, 4, 16, 32])
def test_rows_of_several_particles(hip, monkeypatch, lanes):
    # systems that end inside a group's rows, some with cells
    ss = [_gas(5, 1, 5), _gas(6, 1, 9), _gas(7, 3, 11), _gas(8, 33, 17), _gas(9, 7, 13)]
    per = [dict(seed=100 + k) for k in range(len(ss))]
    got = []
    for fuse in (1, 0):
        monkeypatch.setenv("OXH_FUSE", str(fuse))
        monkeypatch.setenv("OXH_PERSIST", "0")
        monkeypatch.setenv("OXH_FORCE_LANES", str(lanes))
        with hip.HIPBatch(ss, options=per, dt=0.003, verlet_skin=0.05, refresh_vel=True, **THERMO["langevin"]) as b:
            b.run(96)
            got.append([dict(b.state(k), F=b.forces(k)[0], rebuilds=b.info(k)[0]) for k in range(len(ss))])
    _agree(*got)
