"""The packed close kernel (HB and CRST from LDS work lists, bonds by whole
waves) and the cosine windows that leave pairs out of them.

  - packed and in-place kernels give the same bits where their workgroups are
    partly filled, hold particles without close pairs, or end inside a
    particle group: sizes around the 256-thread workgroup for 2, 4, 8 and 32
    lanes per nucleotide, down to one nucleotide;
  - every pair term of isolated nucleotide pairs at random separations and
    orientations, so that separations and cosines fall on both sides of every
    window, against the FP64 oracle.  A pair that a window left out wrongly
    would miss a whole term: its force would be off by more than the bar.
    Bar: 1e-5 of the largest force, FP32 terms (the force tests' bar), 1e-9
    all-FP64.
"""
import numpy as np
import pytest

from _common import vec_rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


def _strands(lengths, seed):
    """Single helix strands side by side, 2.2 apart, with thermal displacements."""
    from oxdna_amd import systems
    rng = np.random.default_rng(seed)
    b = systems._Builder()
    side = int(np.ceil(np.sqrt(len(lengths))))
    for k, n in enumerate(lengths):
        pos, a1, a3 = systems.duplex_geometry(max(n, 2), perp=(1.0, 0.0, 0.0))
        b.add_strand(pos[:n] + np.array([3.0 + 2.2 * (k % side), 3.0 + 2.2 * (k // side), 1.0]), a1[:n], a3[:n], rng.integers(0, 4, n))
    s = b.build([60.0, 60.0, 60.0], "strands", T=systems.celsius(30.0), salt=0.5)
    s.pos = s.pos + 0.01 * rng.normal(size=s.pos.shape)
    return s


@pytest.mark.parametrize("lanes", [2, 4, 8, 32])
@pytest.mark.parametrize("lengths", [[1], [2], [7], [8, 1], [31, 2], [33], [63, 1], [65], [40, 40, 40, 9], [61, 60, 60, 60, 20]])
def test_packed_equals_in_place_at_workgroup_edges(hip, monkeypatch, lanes, lengths):
    s = _strands(lengths, 3)
    monkeypatch.setenv("OXH_PERSIST", "0")
    monkeypatch.setenv("OXH_EDGE", "0")
    monkeypatch.setenv("OXH_FORCE_LANES", str(lanes))
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    got = []
    for pack in (0, 1):
        monkeypatch.setenv("OXH_PACK", str(pack))
        with hip.HIPBatch(s) as b:
            assert b.stats()["pack"] == bool(pack)
            b.compute_forces()
            got.append((*b.forces(), b.energy_split(), b.hb_count()))
    for x, y in zip(*got):
        assert np.array_equal(x, y)


def _random_pairs(n, seed):
    """n pairs of lone nucleotides, 8 apart, each pair at a random separation of base or stacking sites below 0.9."""
    from oxdna_amd import systems
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 8.0 + 4.0

    def frames():
        a1 = rng.normal(size=(n, 3))
        a1 /= np.linalg.norm(a1, axis=1, keepdims=True)
        a3 = rng.normal(size=(n, 3))
        a3 -= a1 * (a3 * a1).sum(1, keepdims=True)
        return a1, a3 / np.linalg.norm(a3, axis=1, keepdims=True)

    a1, a3 = frames()
    b1, b3 = frames()
    # half of the partners nearly antiparallel in a1 and parallel or antiparallel in a3, where HB, CRST and CXST live
    near = rng.random(n) < 0.75
    sign = np.where(rng.random((n, 1)) < 0.5, 1.0, -1.0)
    flip = np.where(rng.random((n, 1)) < 0.5, 1.0, -1.0)
    c1 = flip * a1 + 0.6 * rng.normal(size=(n, 3))
    c1 /= np.linalg.norm(c1, axis=1, keepdims=True)
    c3 = sign * a3 + 0.6 * rng.normal(size=(n, 3))
    c3 -= c1 * (c3 * c1).sum(1, keepdims=True)
    c3 /= np.linalg.norm(c3, axis=1, keepdims=True)
    b1, b3 = np.where(near[:, None], c1, b1), np.where(near[:, None], c3, b3)
    d = rng.normal(size=(n, 3)) + np.where(rng.random((n, 1)) < 0.5, 1.5, 0.0) * a1
    d *= (rng.uniform(0.33, 0.9, n) / np.linalg.norm(d, axis=1))[:, None]
    arm = np.where(rng.random((n, 1)) < 0.7, 0.4, 0.34)
    q = g + arm * a1 + d - arm * b1
    bt = rng.integers(0, 4, n)
    keep = np.ones(2 * n, bool)
    pos = np.stack([g, q], 1).reshape(-1, 3)
    x1, x3 = np.stack([a1, b1], 1).reshape(-1, 3), np.stack([a3, b3], 1).reshape(-1, 3)
    types = np.stack([bt, np.where(rng.random(n) < 0.8, 3 - bt, rng.integers(0, 4, n))], 1).reshape(-1)
    none = np.full(2 * n, -1, np.int32)
    return systems.System(pos=pos[keep], a1=x1, a3=x3, btype=types.astype(np.int32), n3=none, n5=none.copy(), strand=np.arange(2 * n, dtype=np.int32),
                          box=np.array([side * 8.0] * 3), T=systems.celsius(25.0), salt=0.5, name="pairs")


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("pack", [0, 1])
def test_random_pairs_against_oracle(hip, monkeypatch, precision, pack):
    from oracle import pyoracle as po
    if precision == "double" and pack:
        pytest.skip("the all-FP64 kernels have no packed form")
    s = _random_pairs(2000, 11)
    ref = po.forces(po.Params(T=s.T, salt=s.salt), s)
    # every term of lone pairs is met: excluded volume, HB, CRST, CXST
    assert np.all(np.abs(ref["E8"][[3, 4, 5, 6]]) > 0)
    monkeypatch.setenv("OXH_EDGE", "0")
    monkeypatch.setenv("OXH_FORCE_LANES", "4")
    monkeypatch.setenv("OXH_FAR_LANES", "0")
    monkeypatch.setenv("OXH_PACK", str(pack))
    with hip.HIPBatch(s, backend_precision=precision) as b:
        b.compute_forces()
        F, T, E = b.forces()
        split = b.energy_split()
    bar = 1e-5 if precision == "mixed" else 1e-9
    # pairs without steep overlap, each against the largest force among them
    soft = np.linalg.norm(ref["F"], axis=1) < 50.0
    assert soft.sum() > 2000
    for x, y in ((F, ref["F"]), (T, ref["T"])):
        assert np.abs(x - y)[soft].max() <= bar * np.abs(y[soft]).max()
    assert vec_rel_err(F, ref["F"])[0] <= bar
    assert np.all(np.abs(split - ref["E8"]) <= bar * np.abs(ref["E8"]).sum())
