"""Force calls on the caller's buffers whose states come and go.

A call first evaluates the forces on the lists in hand, and every force kernel
leaves the batch alone when the state asks for new lists; after two such calls
in a row a batch without cells queues its lists at once.  For each form of the
force kernels (in place, packed, half-list, far pairs in their own kernel,
all-FP64 with and without it, the workgroup engine, oxRNA2, with external
forces): states that move further than the skin, four in a row, then states
that hold, then both in turn.  Additions against the oracle at the force
tests' bars (1e-5 of the largest force, 1e-9 all-FP64; oxRNA2 against a batch
created with that state, 1e-5), one list build for each state that needs one
and none otherwise.
"""
import numpy as np
import pytest

from _common import load_golden, oracle_params, vec_rel_err
from _hipmem import DeviceArray

pytestmark = pytest.mark.gpu

GRID = dict(OXH_PERSIST="0", OXH_EDGE="0", OXH_FORCE_LANES="4", OXH_FAR_LANES="0", OXH_PACK="0")
FORMS = {
    "in_place": GRID,
    "packed": dict(GRID, OXH_PACK="1"),
    "half_list": dict(GRID, OXH_EDGE="1"),
    "far_kernel": dict(GRID, OXH_FAR_LANES="8"),
    "half_list_far_kernel": dict(GRID, OXH_EDGE="1", OXH_FAR_LANES="8"),
    "double": GRID,
    "double_far_kernel": dict(GRID, OXH_FAR_LANES="8"),
    "workgroup": {},
    "rna": GRID,
    "external": GRID,
    "cells": GRID,
    "cells_far_kernel": dict(GRID, OXH_FAR_LANES="8"),
}


@pytest.fixture(scope="module")
def hip():
    from oxdna_amd import _lib, backend
    assert _lib.device_count() >= 1, "no GPU visible"
    return backend


@pytest.mark.parametrize("form", list(FORMS))
def test_states_that_come_and_go(hip, monkeypatch, form):
    from oracle import pyoracle as po
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(3)
    if form == "rna":
        from test_gpu_rna import load_rna
        s, opts, _ = load_rna("rna_contacts_nohb")
    elif form.startswith("cells"):
        from test_gpu_fused import _gas
        s, opts = _gas(4, 30, 20), {}   # 1,200 nt
    else:
        s, opts, _ = load_golden("dense_md_excl_30C")
    double = form.startswith("double")
    if double:
        opts = dict(opts, backend_precision="double")
    ft = np.float64 if double else np.float32
    bar = 1e-9 if double else 1e-5
    trap = dict(type="trap", particle=3, stiff=2.0, pos0=(1.0, 2.0, 3.0), dir=(0.0, 0.0, 1.0))

    def expected(t):
        if form == "rna":
            with hip.HIPBatch(t, **opts) as f:
                return f.forces()[:2]
        ref = po.forces(oracle_params(t, opts) if opts else po.Params(T=t.T, salt=t.salt), t)
        F = ref["F"].copy()
        if form == "external":
            F[3] += 2.0 * (np.array([1.0, 2.0, 3.0]) - t.pos[3])
        return F, ref["T"]

    with hip.HIPBatch(s, **opts) as b:
        assert b.stats()["engine"] == ("workgroup" if form == "workgroup" else "grid-edge" if form.startswith("half") else "grid")
        if form == "external":
            b.set_external_forces([trap])
        at, builds = s.pos.copy(), b.info()[0]
        for move in [0, 1, 1, 1, 1, 0, 0, 1, 1, 0, 1, 0]:
            t = s.copy()
            if move:
                at = at + 0.3 * rng.normal(size=3)          # all of it, by more than the skin
            t.pos = at + 0.002 * rng.normal(size=s.pos.shape)   # and less than it
            q = hip.quat_from_frame(s.a1, s.a3)
            pos = np.zeros((s.N, 4))
            pos[:, :3] = t.pos
            pre = rng.normal(size=(2, s.N, 4)).astype(ft)
            dF, dT = DeviceArray(pre[0]), DeviceArray(pre[1])
            d_pos, d_quat = DeviceArray(pos), DeviceArray(q)
            b.interaction_forces(d_pos.ptr, d_quat.ptr, dF.ptr, dT.ptr)
            b.sync()
            F, T = expected(t)
            for got, p, want in ((dF, pre[0], F), (dT, pre[1], T)):
                add = got.numpy()[:, :3].astype(np.float64) - p[:, :3]
                assert vec_rel_err(add, want)[0] <= 10 * bar, (form, move)   # rounding of the additions onto O(1) values
            builds += move
            assert b.info()[0] == builds, (form, move)


def test_far_kernel_of_calls_alone(hip):
    """24 bundles of 960 nt with long rows (633 far pairs each): steps keep
    the far pairs inline for the sake of one launch, force calls on the
    caller's buffers take the far kernel, which is 6 % faster for them."""
    from oracle import pyoracle as po
    from oxdna_amd import systems
    ss = [systems.duplex_bundle(2 + k, nx=4, ny=4, bp=30, spacing=2.6, lz=14.3, tc=30.0, salt=0.1) for k in range(24)]
    n = sum(s.N for s in ss)
    pos = np.zeros((n, 4))
    pos[:, :3] = np.concatenate([s.pos for s in ss])
    d_pos = DeviceArray(pos)
    d_quat = DeviceArray(np.concatenate([hip.quat_from_frame(s.a1, s.a3) for s in ss]))
    dF, dT = DeviceArray.zeros((n, 4), np.float32), DeviceArray.zeros((n, 4), np.float32)
    with hip.HIPBatch(ss) as b:
        before = b.stats()
        assert b.routes()["call_far_lanes"] > 0
        b.interaction_forces(d_pos.ptr, d_quat.ptr, dF.ptr, dT.ptr)
        b.sync()
        assert b.stats() == before
    first = 0
    for k, s in enumerate(ss):
        if k in (0, 23):
            ref = po.forces(po.Params(T=s.T, salt=s.salt), s)
            assert vec_rel_err(dF.numpy()[first:first + s.N, :3].astype(np.float64), ref["F"])[0] <= 1e-5
            assert vec_rel_err(dT.numpy()[first:first + s.N, :3].astype(np.float64), ref["T"])[0] <= 1e-5
        first += s.N
