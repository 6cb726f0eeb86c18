"""Every oxRNA2 pair term of lone nucleotide pairs, against the model in 64 bits.

The kernel skips a term unless every cosine is inside its window, and takes
sines of angles from a polynomial (mixed) or a reciprocal root (all-FP64).
Pairs at random separations and orientations fall on both sides of every
window; a term that a window leaves out wrongly is missing whole.  Others have
angles of exactly 0 and pi, and close to them, in hydrogen bonding, cross
stacking and coaxial stacking: the guard of a small sine, and the reflected
angles pi - theta and 2 pi - theta.  Reference: the energy of the model in
plain 64-bit torch, forces and torques as its derivatives by autograd
(perf/cases.py), with one exception of the model's own: the derivative by a
reflected angle divides by that angle's sine, and its pi is the FP32 one, so
that the two sines differ by 8.7e-8.  Its arc cosine, which stops 1e-15 short
of 1, is replaced by one that does not.

Bars, of the largest force: all-FP64 1e-9, the force tests'.  Mixed 3e-5: an
FP32 angle theta carries 2^-24 / sin(theta), its sine that by 1 / sin(theta)
again, 1.7e-5 of a factor's derivative at theta = 0.06.  Closer to 0 and pi only
the exact angles are compared in that form, and closer than 1.5e-4 in the other,
where the model's guard stands in for a ratio (sin^2 up to 1e-8).
"""
import numpy as np
import pytest

from test_gpu_packed import _random_pairs

pytestmark = pytest.mark.gpu

BAR = {"mixed": 3e-5, "double": 1e-9}
SMALL = {"mixed": 0.06, "double": 1.5e-4}
BASE, STACK = float(np.float32(0.4)), float(np.float32(0.34))   # the model's site positions


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


class _ModelPi(float):
    """PI of the model: PI - t and 2 PI - t with derivatives by t of -sin(t) / |sin(PI - t)|."""

    def __rmul__(self, n):
        return _ModelPi(n * float(self))

    def __sub__(self, t):
        u = float(self) - t.detach()
        return u - (t - t.detach()) * (t.detach().sin() / u.sin().abs())


def _acos(c):
    """The arc cosine, 0 and pi included; no derivative there (it multiplies a zero vector)."""
    import torch
    v = c.detach().clamp(-1.0, 1.0)
    sin2 = (1.0 - v) * (1.0 + v)
    slope = torch.where(sin2 > 2e-15, -1.0 / sin2.clamp_min(1e-30).sqrt(), torch.zeros_like(v))
    return torch.acos(v) + slope * (c - c.detach())


def _unit(v):
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _turn(v, axis, angle):
    return v * np.cos(angle) + np.cross(axis, v) * np.sin(angle) + axis * np.dot(axis, v) * (1.0 - np.cos(angle))


def _aligned(seed):
    """Pairs with angles of 0, pi and close to them."""
    from oxdna_amd import systems
    rng = np.random.default_rng(seed)
    rows = []
    for tilt in (0.0, 1e-3, 1e-2, 0.05, 0.1, 0.2):
        for kind in ("hb", "crst", "cxst"):
            for flip in (1.0, -1.0):
                for _ in range(6):
                    q, r = np.linalg.qr(rng.normal(size=(3, 3)))
                    q = q * np.sign(np.diag(r))
                    a1, a2, a3 = (np.eye(3) if tilt == 0.0 else q * np.sign(np.linalg.det(q))).T
                    if kind == "hb":        # t1 = t2 = t3 = 0, t4 = pi or 0
                        b1, b3, d, arm = -a1, -flip * a3, a1 * rng.uniform(0.35, 0.6), BASE
                    elif kind == "crst":    # t7, t8 = 0 or pi
                        b1, b3, d, arm = -a1, flip * a3, a3 * rng.uniform(0.42, 0.58) * rng.choice([-1.0, 1.0]), BASE
                    else:                   # t1 = pi, t4 = 0, t5, t6 = 0 or pi
                        b1, b3, d, arm = a1, a3, flip * a3 * rng.uniform(0.42, 0.58), STACK
                    axis, other = _unit(rng.normal(size=(2, 3)))
                    if tilt > 0.0:   # every angle by another amount
                        b1, b3, d = _turn(b1, axis, tilt), _turn(b3, axis, tilt), _turn(d, other, 0.7 * tilt)
                    rows.append((a1, a3, arm * a1 + d - arm * b1, b1, b3))
    n = len(rows)
    side = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 8.0 + 4.0
    a1, a3, dq, b1, b3 = (np.stack(v) for v in zip(*rows))
    none = np.full(2 * n, -1, np.int32)
    two = lambda x, y: np.stack([x, y], 1).reshape(-1, 3)  # noqa: E731
    bt = np.tile([0, 3], n).astype(np.int32)
    return systems.System(pos=two(g, g + dq), a1=two(a1, b1), a3=two(a3, b3), btype=bt, n3=none, n5=none.copy(),
                          strand=np.arange(2 * n, dtype=np.int32), box=np.array([side * 8.0] * 3), T=systems.celsius(25.0), salt=0.5,
                          name="aligned")


def _smallest_angle(s):
    """The smallest angle to 0 or pi of each pair's cosines that is not 0 or pi itself, for both its nucleotides."""
    p, q = slice(0, None, 2), slice(1, None, 2)
    r = s.pos[q] - s.pos[p]
    d = [_unit(r + arm * (s.a1[q] - s.a1[p])) for arm in (BASE, STACK)]
    c = [(s.a1[p] * s.a1[q]).sum(1), (s.a3[p] * s.a3[q]).sum(1)]
    for u in d:
        c += [(x * u).sum(1) for x in (s.a1[p], s.a1[q], s.a3[p], s.a3[q])]
    t = np.arccos(np.minimum(np.abs(c), 1.0))
    return np.repeat(np.where(t < 1e-6, np.inf, t).min(0), 2)


@pytest.mark.parametrize("precision", ["mixed", "double"])
def test_pairs_against_64_bits(hip, monkeypatch, precision):
    import torch
    from perf import cases
    monkeypatch.setattr(torch.cuda, "is_available", lambda: False)   # the reference on the CPU
    monkeypatch.setattr(cases, "PI", _ModelPi(cases.PI))
    monkeypatch.setattr(cases, "_acos", _acos)
    monkeypatch.setenv("OXH_FORCE_LANES", "4")
    ss = [_random_pairs(450, 11 + k) for k in range(4)] + [_aligned(5)]
    with hip.HIPBatch(ss, backend_precision=precision, interaction_type="RNA2") as b:
        b.compute_forces()
        got = [b.forces(k) for k in range(len(ss))]
        split = [b.energy_split(k) for k in range(len(ss))]
    active = np.zeros(3, int)
    for k, s in enumerate(ss):
        ex = cases._Exact([s], "RNA2")
        pos, quat = torch.from_numpy(s.pos), torch.from_numpy(hip.quat_from_frame(s.a1, s.a3))
        F, T, share, _ = ex.forces(pos, quat, ex.pairs(pos, 0.0))
        F, T = F.numpy(), T.numpy()
        terms = np.stack([share[t].numpy() for t in ("hb", "crst", "cxst")])
        active += (np.abs(terms) > 1e-6).sum(1) // 2
        # pairs without steep overlap, and without angles that the form cannot resolve
        soft = (np.linalg.norm(F, axis=1) < 50.0) & (_smallest_angle(s) >= SMALL[precision])
        assert soft.sum() > 0.15 * s.N   # most tilted pairs are below SMALL
        bar = BAR[precision]
        for name, x, y in (("force", got[k][0], F), ("torque", got[k][1], T)):
            worst = np.abs(x - y)[soft].max() / np.abs(y[soft]).max()
            print(precision, s.name, k, name, "%.2e" % worst, flush=True)
            assert worst <= bar, (name, k)
        E = sum(v.numpy() for v in share.values())
        assert np.abs(got[k][2] - E)[soft].max() <= bar * np.abs(E[soft]).max()
        want = np.array([float(share[t].sum()) for t in cases._TERMS])
        assert np.all(np.abs(split[k] - want)[4:] <= bar * np.abs(want[4:]).sum())
    # every term is met, and left out, by many pairs
    pairs = sum(s.N for s in ss) // 2
    assert np.all(active > 40) and np.all(active < pairs - 400), active
