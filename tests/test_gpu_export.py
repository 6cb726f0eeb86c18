"""What the host reads: state and forces in the caller's order, sums per system.

Sizes on both sides of what a kernel writes straight into page-locked memory
(546 nt of state), and where one half, both halves and a part of a third are
filled; the middle system of three, in Hilbert order.  Positions, velocities
and momenta come back as they were set, to the bit; axes to the rounding of a
quaternion (1e-14, bar 1e-12).  Sums against numpy's over the same arrays:
FP64 sums of n terms in another order differ by less than n times 1e-16 of the
sum of magnitudes (bar 1e-11); the terms against the FP32 energies by the
latter's rounding (6e-8 of the sum of magnitudes, bar 1e-6).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _gas(seed, n, bp):
    from oxdna_amd import systems
    rng = np.random.default_rng(seed)
    b = systems._Builder()
    side = int(np.ceil(n ** (1.0 / 3.0)))
    a = max(12.0, 0.4 * bp + 4.0)
    for k in range(n):
        c = (np.array([k % side, k // side % side, k // side ** 2]) + 0.5) * a
        systems.add_duplex(b, rng.integers(0, 4, bp), c, systems.random_rotation(rng))
    return b.build([side * a] * 3, "gas", T=systems.celsius(30.0), salt=0.5)


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("n,bp", [(1, 8), (21, 13), (1, 274), (500, 9), (514, 17), (600, 20)])
def test_reads(hip, n, bp, precision):
    rng = np.random.default_rng(5)
    ss = [_gas(1, 2, 8), _gas(2, n, bp), _gas(3, 1, 11)]
    with hip.HIPBatch(ss, dt=0.003, verlet_skin=0.05, refresh_vel=True, backend_precision=precision) as b:
        want = {k: np.asarray(getattr(ss[1], k)) for k in ("pos", "a1", "a3")}
        want["vel"], want["L"] = rng.normal(size=(2, ss[1].N, 3))
        b.set_state(sys=1, **want)
        b.hilbert_sort()
        b.compute_forces()
        got = b.state(1)
        for k in ("pos", "vel", "L"):
            assert np.array_equal(got[k], want[k]), k
        for k in ("a1", "a3"):
            assert np.abs(got[k] - want[k]).max() < 1e-12, k
        E = b.forces(1)[2]
        e = b.energies()[1]
        assert abs(e[0] - E.sum()) < 1e-11 * np.abs(E).sum()
        assert abs(e[2] - 0.5 * (want["vel"] ** 2).sum()) < 1e-11 * e[2]
        assert abs(e[3] - 0.5 * (want["L"] ** 2).sum()) < 1e-11 * e[3]
        split = b.energy_split(1)
        assert abs(split.sum() - E.sum()) < 1e-6 * np.abs(split).sum()
        kinetic = b.stress(1)[1]
        v = want["vel"]
        for c, (x, y) in enumerate([(0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)]):
            assert abs(kinetic[c] - (v[:, x] * v[:, y]).sum()) < 1e-11 * np.abs(v[:, x] * v[:, y]).sum()
