"""Force calls without allocation, before and after oxh_noalloc_init.

The entry point itself allocates nothing: until the library is set up on the
GPU by oxh_noalloc_init, topology and error word go through static memory.
Both ways give the same bits, and refuse the same calls.  What a process has
set up stays, so the calls before it run in a process of their own.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import ctypes as C, sys
sys.path[:0] = [%r, %r]
import numpy as np
from _common import load_golden
from _hipmem import DeviceArray, Stream
from oxdna_amd import _lib, backend, systems


def call(s, precision, stream=None, **opts):
    pos = np.zeros((s.N, 4))
    pos[:, :3] = s.pos
    ft = np.float64 if precision == "double" else np.float32
    d_pos, d_quat = DeviceArray(pos), DeviceArray(backend.quat_from_frame(s.a1, s.a3))
    F, T = DeviceArray.zeros((s.N, 4), ft), DeviceArray.zeros((s.N, 4), ft)
    keep = []
    d = backend.make_desc(s, keep, backend_precision=precision, **opts)
    rc = _lib.lib().oxh_interaction_compute_forces_noalloc(0, C.byref(d), d_pos.ptr, d_quat.ptr, F.ptr, T.ptr, stream)
    return rc, F.numpy(), T.numpy()


stream = Stream()
jobs = []
for name in ("gas8_25C_0.5M", "bundle_md_30C"):
    s, opts, _ = load_golden(name)
    jobs += [(s, p, st, opts) for p in ("mixed", "double") for st in (None, stream.handle)]
crowd = systems.duplex_bundle(3, nx=5, ny=5, bp=20, spacing=2.6, lz=14.0, tc=30.0, salt=0.03)   # over 256 neighbours
first = [call(s, p, st, **o) for s, p, st, o in jobs]
refused = call(crowd, "mixed")
assert refused[0] != 0 and not refused[1].any(), refused[0]
for _ in range(2):
    assert _lib.lib().oxh_noalloc_init(0) == 0
then = [call(s, p, st, **o) for s, p, st, o in jobs]
assert call(crowd, "mixed")[0] == refused[0]
for a, b in zip(first, then):
    assert a[0] == b[0] == 0 and a[1].any()
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
assert call(*jobs[0][:2], **jobs[0][3])[0] == 0
print("done", len(first))
"""


@pytest.mark.gpu
def test_same_bits_before_and_after():
    r = subprocess.run([sys.executable, "-c", CHILD % (ROOT, os.path.join(ROOT, "tests"))], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("done 8"), r.stdout + r.stderr


@pytest.mark.parametrize("device", [-1, 64])
def test_init_refuses_devices_out_of_range(device):
    from oxdna_amd import _lib
    lib = _lib.lib()
    assert lib.oxh_noalloc_init(device) == 1 and b"bad device" in lib.oxh_last_error()
