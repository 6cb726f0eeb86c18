"""The work that a program has this package do, as cases that can be timed.

A case is a dict of plain values.  Five kinds, after the package's uses:

  noalloc  one force evaluation of one small system through the entry point
           for callers that cannot allocate (`interaction_forces_noalloc`);
  forces   one force evaluation on the caller's device buffers
           (`HIPBatch.interaction_forces`), the reference program's plug-in
           surface: every MD step of such a program is one call;
  md       a run between two printed configurations: `HIPBatch.run`, then
           every system's state;
  pool     one round of a job server: jobs of uneven size and length admitted
           into a slot pool, run to their ends, their states taken and the
           slots released;
  observe  what is printed every so many steps, on the current state:
           energies, the split by term, stress, hydrogen bonds and forces.

Systems are the layouts of the package's workload builder (duplex gas,
hexagonal duplex bundle, single strands, hairpins, oxRNA duplexes) with
thermal displacements.  The mixed form (FP32 pair terms) hands its results
back in FP32, the all-FP64 form in FP64.

`exact` evaluates the same model in 64 bits with plain torch: the energy as
the model defines it, forces and torques as its derivatives by autograd, the
integrator and the thermostats with their counter-based noise.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from oxdna_amd import backend, systems

DT, SKIN, DIFF = 0.003, 0.05, 2.5
SIGMA_POS, SIGMA_ROT = 0.01, 0.02   # displacements of a relaxed helix, per component (no steep overlaps)


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest call: one 20-bp duplex, forces for a caller that cannot allocate
        dict(name="noalloc_duplex40", kind="noalloc", model="DNA2", precision="mixed", layout="gas", n=1, length=20, salt=0.5, tc=20.0),
        # plug-in force calls: the duplex gas (24,576 nt), the dense bundle (196,608 nt, low salt: long Debye-Hueckel range) ...
        dict(name="forces_gas24576", kind="forces", model="DNA2", precision="mixed", layout="gas", n=512, length=24, salt=0.5, tc=25.0),
        dict(name="forces_bundle196608", kind="forces", model="DNA2", precision="mixed", layout="bundle", n=32, ny=32, length=96, salt=0.2, tc=30.0),
        # ... an odd-sized bundle all in FP64 (backend_precision = double), and a set of oxRNA2 systems
        dict(name="forces_bundle53352_double", kind="forces", model="DNA2", precision="double", layout="bundle", n=19, ny=18, length=78, salt=0.2, tc=30.0),
        dict(name="forces_rna24x1024", kind="forces", model="RNA2", precision="mixed", layout="rna", n=24, length=32, salt=1.0, tc=37.0),
        # MD runs: one duplex alone (latency), a batch of 256 uneven hairpins, a small odd system without cells, the gas and the bundle
        dict(name="md_duplex40", kind="md", model="DNA2", precision="mixed", layout="gas", n=1, length=20, salt=0.5, tc=20.0, thermostat="langevin", steps=512),
        dict(name="md_hairpins256", kind="md", model="DNA2", precision="mixed", layout="hairpins", n=256, length=0, salt=0.5, tc=25.0, thermostat="langevin", steps=512),
        dict(name="md_strands777", kind="md", model="DNA2", precision="mixed", layout="strands", n=21, length=37, salt=0.5, tc=45.0, thermostat="john", steps=448),
        dict(name="md_gas24576", kind="md", model="DNA2", precision="mixed", layout="gas", n=512, length=24, salt=0.5, tc=25.0, thermostat="bussi", steps=300),
        dict(name="md_bundle196608", kind="md", model="DNA2", precision="mixed", layout="bundle", n=32, ny=32, length=96, salt=0.2, tc=30.0, thermostat="langevin", steps=192),
        # a job server's round: eight slots of up to 2,048 nt
        dict(name="pool_jobs8", kind="pool", model="DNA2", precision="mixed", layout="mix", n=8, length=2048, salt=0.5, tc=40.0, thermostat="langevin", steps=320),
        # the observables of a printed step
        dict(name="observe_gas24576", kind="observe", model="DNA2", precision="mixed", layout="gas", n=512, length=24, salt=0.5, tc=25.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["noalloc", "forces", "forces", "md", "md", "pool", "observe"])
    c = dict(kind=kind, model="DNA2", precision="mixed", salt=round(rng.uniform(0.2, 1.0), 3), tc=round(rng.uniform(20.0, 60.0), 2))
    if kind == "noalloc":
        c.update(layout=rng.choice(["gas", "strands"]), salt=round(rng.uniform(0.4, 1.0), 3), length=_log(rng, 8, 60),
                 precision=rng.choice(["mixed", "mixed", "double"]))
        c["n"] = max(1, _log(rng, 16, 4000) // (2 * c["length"]))
        return c
    if kind == "pool":
        c.update(layout="mix", n=rng.randint(2, 12), length=_log(rng, 520, 2048), thermostat="langevin", steps=_log(rng, 64, 320))
        return c
    if kind == "md" and rng.random() < 0.4:
        c.update(layout="hairpins", n=_log(rng, 1, 256), length=0, thermostat=rng.choice(["langevin", "langevin", "john", "no"]),
                 steps=_log(rng, 96, 512))
        return c
    if kind == "forces" and rng.random() < 0.25:
        c.update(model="RNA2", layout="rna", n=_log(rng, 1, 24), length=rng.randint(9, 32), precision=rng.choice(["mixed", "double"]))
        return c
    c["precision"] = rng.choice(["mixed", "mixed", "mixed", "double"])
    c["layout"] = rng.choice(["gas", "bundle", "strands"])
    total = _log(rng, 40, 40000 if c["precision"] == "double" else 160000)
    if c["layout"] == "bundle":
        c["length"] = rng.randint(30, 97)
        c["n"] = max(6, int(math.sqrt(total / (2 * c["length"]))))
        c["ny"] = 2 * max(3, (total // (2 * c["length"] * c["n"])) // 2)
    else:
        c["length"] = min(_log(rng, 8, 97), total)
        c["n"] = max(1, total // (c["length"] * (2 if c["layout"] == "gas" else 1)))
    if kind == "md":
        c.update(thermostat=rng.choice(["langevin", "langevin", "bussi", "john", "no"]), steps=_log(rng, 64, 192))
    return c


# ------------------------------------------------------------------ the systems

def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    return np.stack([np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)], 1),
                     np.stack([2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)], 1),
                     np.stack([2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1)], 1)


def _thermal(s, rng):
    """Thermal displacements of every centre and orientation, and velocities at the system's temperature."""
    n = s.N
    s.pos = s.pos + SIGMA_POS * rng.normal(size=(n, 3))
    v = SIGMA_ROT * rng.normal(size=(n, 3))
    a1, a3 = s.a1 + np.cross(v, s.a1), s.a3 + np.cross(v, s.a3)
    s.a1 = a1 / np.linalg.norm(a1, axis=1, keepdims=True)
    a3 = a3 - s.a1 * (a3 * s.a1).sum(1, keepdims=True)
    s.a3 = a3 / np.linalg.norm(a3, axis=1, keepdims=True)
    s.vel, s.L = math.sqrt(s.T) * rng.normal(size=(n, 3)), math.sqrt(s.T) * rng.normal(size=(n, 3))
    return s


def _assemble(template, strands, centres, rot, rng, box, case):
    """Copies of a template (rows of `strands` strands of equal length, bases of strand 2 pairing with strand 1's) at `centres`."""
    pos0, a10, a30 = template
    m, k = len(pos0), len(centres)
    length = m // strands
    turn = (lambda v: np.einsum("kab,mb->kma", rot, v)) if rot is not None else (lambda v: np.broadcast_to(v, (k, m, 3)))
    seq = rng.integers(0, 4, (k, length))
    bt = seq if strands == 1 else np.concatenate([seq, 3 - seq[:, ::-1]], 1)
    i = np.arange(k * m)
    n3 = np.where(i % length == 0, -1, i - 1)
    n5 = np.where(i % length == length - 1, -1, i + 1)
    s = systems.System(pos=(turn(pos0) + centres[:, None, :]).reshape(-1, 3), a1=turn(a10).reshape(-1, 3).copy(), a3=turn(a30).reshape(-1, 3).copy(),
                       btype=bt.reshape(-1).astype(np.int32), n3=n3.astype(np.int32), n5=n5.astype(np.int32), strand=(i // length).astype(np.int32),
                       box=np.asarray(box, np.float64), T=systems.celsius(case["tc"]), salt=case["salt"], name=case["layout"])
    return _thermal(s, rng)


def _centred_duplex(bp):
    pos, a1, a3 = systems.duplex_geometry(bp, perp=(1.0, 0.0, 0.0))
    return pos - np.array([0.0, 0.0, (bp - 1) * systems.BASE_BASE / 2.0]), a1, a3


def _lattice(n, a):
    side = math.ceil(round(n ** (1.0 / 3.0), 6))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return (g + 0.5) * a, [side * a] * 3


def _gas(n, length, rng, case, strands=2):
    # 1e-3 nucleotides per unit volume, as the plain duplex gas
    t = _centred_duplex(length)
    a = max(20.0, (strands * length / 1e-3) ** (1.0 / 3.0))
    centres, box = _lattice(n, a)
    if strands == 1:
        t = tuple(v[:length] - (v[:length].mean(0) if k == 0 else 0.0) for k, v in enumerate(t))
    return _assemble(t, strands, centres, _rotations(rng, n), rng, box, case)


def _bundle(nx, ny, bp, rng, case):
    dy = 2.6 * math.sqrt(3.0) / 2.0
    lz = max(14.0, bp * systems.BASE_BASE + 2.6)
    j, i = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    centres = np.stack([(i + 0.5 * (j % 2) + 0.25) * 2.6, (j + 0.5) * dy, np.full(i.shape, lz / 2)], -1).reshape(-1, 3)
    return _assemble(_centred_duplex(bp), 2, centres, None, rng, [nx * 2.6, ny * dy, lz], case)


def _systems(case, seed):
    rng = np.random.default_rng([seed, 77])
    lay = case["layout"]
    if lay == "gas":
        return [_gas(case["n"], case["length"], rng, case)]
    if lay == "strands":
        return [_gas(case["n"], case["length"], rng, case, 1)]
    if lay == "bundle":
        return [_bundle(case["n"], case["ny"], case["length"], rng, case)]
    if lay == "hairpins":
        # the sizes are the case's; bases are exchanged (complements stay complements) and each hairpin is turned by the seed
        out = systems.hairpin_set(9, n=case["n"], t_lo=case["tc"], t_hi=case["tc"] + 15.0)
        for s, turn in zip(out, _rotations(rng, len(out))):
            pairs = rng.permutation(2)
            swap = rng.integers(0, 2, 2)
            low = pairs[np.minimum(s.btype, 3 - s.btype)]
            s.btype = np.where((s.btype > 1) ^ (swap[low] == 1), 3 - low, low).astype(np.int32)
            s.pos, s.a1, s.a3 = (s.pos - 15.0) @ turn.T + 15.0, s.a1 @ turn.T, s.a3 @ turn.T
            s.salt = case["salt"]
            _thermal(s, rng)
        return out
    if lay == "rna":
        out = []
        for _ in range(case["n"]):
            g = (np.stack(np.meshgrid(np.arange(4), np.arange(4), indexing="ij"), -1).reshape(-1, 2) + 0.5) * 5.0
            ang = rng.uniform(0.0, 2.0 * math.pi, 16)
            rot = np.zeros((16, 3, 3))
            rot[:, 0, 0] = rot[:, 1, 1] = np.cos(ang)
            rot[:, 1, 0] = np.sin(ang)
            rot[:, 0, 1], rot[:, 2, 2] = -rot[:, 1, 0], 1.0
            out.append(_assemble(systems.rna_duplex_geometry(case["length"]), 2, np.concatenate([g, np.full((16, 1), 10.0)], 1), rot, rng,
                                 [20.0, 20.0, 20.0], case))
        return out
    # a server's jobs: uneven sizes up to `length` nucleotides, the layouts in turn
    out = []
    sizes = np.random.default_rng([case["n"], case["length"]])   # the case's, whatever the seed
    for k in range(case["n"]):
        size = max(40, int(round(math.exp(sizes.uniform(math.log(case["length"] / 8), math.log(case["length"] - 8))))))
        if k % 3 == 0:
            out.append(_gas(max(1, size // 48), 24, rng, case))
        elif k % 3 == 1:
            out.append(_gas(max(1, size // 37), 37, rng, case, 1))
        else:
            n = 6 if size > 420 else 4
            out.append(_bundle(n, n, max(10, size // (2 * n * n)), rng, case))
    return out


def _options(case, seed):
    o = dict(dt=DT, verlet_skin=SKIN, backend_precision=case["precision"], interaction_type=case["model"], thermostat=case.get("thermostat", "no"))
    if o["thermostat"] in ("langevin", "john"):
        o["diff_coeff"] = DIFF
    if o["thermostat"] == "john":
        o["newtonian_steps"] = 7
    if o["thermostat"] == "bussi":
        o.update(newtonian_steps=10, bussi_tau=100)
    return o, [dict(seed=1000 * seed + k) for k in range(case["n"])]


def _job_steps(case):
    return [max(1, case["steps"] * (k + 1) // case["n"]) for k in range(case["n"])]


# ------------------------------------------------------------------ the calls

_streams = {}


def _stream():
    """The caller's stream: one for all states, since calls that share the library's scratch have to follow each other."""
    d = torch.cuda.current_device()
    if d not in _streams:
        _streams[d] = torch.cuda.Stream()
    return _streams[d]


def prepare(case, seed):
    ss = _systems(case, seed)
    opts, per = _options(case, seed)
    st = dict(case=case, systems=ss, opts=opts, per=per)
    kind = case["kind"]
    if kind in ("noalloc", "forces"):
        n = sum(s.N for s in ss)
        pos = np.zeros((n, 4))
        pos[:, :3] = np.concatenate([s.pos for s in ss])
        quat = np.concatenate([backend.quat_from_frame(s.a1, s.a3) for s in ss])
        ft = torch.float64 if case["precision"] == "double" else torch.float32
        st.update(pos=torch.from_numpy(pos).cuda(), quat=torch.from_numpy(quat).cuda(), F=torch.zeros((n, 4), dtype=ft, device="cuda"),
                  T=torch.zeros((n, 4), dtype=ft, device="cuda"), stream=_stream())
        torch.cuda.synchronize()
    if kind == "pool":
        st["pool"] = backend.HIPPool([2048] * case["n"])
    elif kind != "noalloc":
        st["batch"] = backend.HIPBatch(ss, options=per[: len(ss)], **opts)
    return st


def _typed(case, v):
    return v if case["precision"] == "double" else np.asarray(v, np.float32)


def _states(case, states):
    return {k: _typed(case, np.concatenate([s[k] for s in states])) for k in ("pos", "a1", "a3", "vel", "L")}


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind in ("noalloc", "forces"):
        with torch.cuda.stream(st["stream"]):
            st["F"].zero_()
            st["T"].zero_()
        where = (st["pos"].data_ptr(), st["quat"].data_ptr(), st["F"].data_ptr(), st["T"].data_ptr(), st["stream"].cuda_stream)
        if kind == "forces":
            st["batch"].interaction_forces(*where)
        else:
            backend.interaction_forces_noalloc(st["systems"][0], *where, **st["opts"])
        return {"F": st["F"], "T": st["T"]}
    if kind == "md":
        b = st["batch"]
        b.run(case["steps"])
        return _states(case, [b.state(k) for k in range(b.nsys)])
    if kind == "pool":
        p = st["pool"]
        for k, (s, steps) in enumerate(zip(st["systems"], _job_steps(case))):
            p.admit(k, s, steps, **st["opts"], **st["per"][k])
        p.run(case["steps"])
        out = _states(case, [p.state(k) for k in range(case["n"])])
        out["done"] = p.status()["done"]
        for k in range(case["n"]):
            p.release(k)
        return out
    b = st["batch"]
    energies, split, (virial, kinetic), hb = b.energies(), b.energy_split(), b.stress(), b.hb_count()
    F, T, E = b.forces()
    out = dict(energies=energies, split=split, virial=virial, kinetic=kinetic, F=F, T=T, E=E)
    return dict({k: _typed(case, v) for k, v in out.items()}, hb=hb)


def _size(case):
    lay, n = case["layout"], case["n"]
    return {"gas": 2 * n * case["length"], "strands": n * case["length"], "bundle": 2 * n * case.get("ny", 0) * case["length"], "hairpins": 38 * n,
            "rna": 32 * n * case["length"], "mix": int(0.42 * n * case["length"])}[lay]


def work(case):
    """Per evaluation and nucleotide: one bond (~500 operations), half of its close pairs (~200 each) and of its Debye-Hueckel pairs (~30
    each), and in a step the integration (~300).  Bytes: the state in, forces out; a step reads and writes the state."""
    n = _size(case)
    dense = case["layout"] in ("bundle", "rna")
    reach = 1.0 + 1.2 / math.sqrt(case["salt"])          # Debye-Hueckel cut-off, about
    far = min(4.2 * reach ** 3 * (0.8 if dense else 0.12), n)
    evaluation = 500 + 0.5 * (18 if dense else 11) * 200 + 0.5 * far * 30
    wide = 8 if case["precision"] == "double" else 4
    once = n * (64 + 16 + 8 * wide)
    if case["kind"] in ("noalloc", "forces"):
        return {"bytes": once, "flops": n * evaluation}
    if case["kind"] == "observe":
        return {"bytes": n * (104 + 16 + 9 * wide), "flops": n * evaluation}
    steps = case["steps"] if case["kind"] == "md" else sum(_job_steps(case)) / case["n"]
    return {"bytes": n * (steps * 2 * 104 + 15 * wide), "flops": n * steps * (evaluation + 300)}


# ------------------------------------------------------------------ the model in 64 bits

def _f(x):
    return float(np.float32(x))


PI = _f(math.pi)


def _table(rows):
    return {k: tuple(_f(x) for x in v) for k, v in rows.items()}


# (a, b, theta0, theta_s, theta_c) of the angular factors f4
_DNA_F4 = _table({"s4": (1.3, 6.4381, 0, 0.8, 0.961538), "s5": (0.9, 3.89361, 0, 0.95, 1.16959),
                  "h1": (1.5, 4.16038, 0, 0.7, 0.952381), "h2": (1.5, 4.16038, 0, 0.7, 0.952381), "h4": (0.46, 0.133855, PI, 0.7, 3.10559),
                  "h7": (4.0, 17.0526, PI * 0.5, 0.45, 0.555556),
                  "c1": (2.25, 7.00545, PI - _f(2.35), 0.58, 0.766284), "c2": (1.7, 6.2469, 1.0, 0.68, 0.865052),
                  "c4": (1.5, 2.59556, 0, 0.65, 1.02564), "c7": (1.7, 6.2469, 0.875, 0.68, 0.865052),
                  "x1": (2.0, 10.9032, PI - 0.25, 0.65, 0.769231), "x4": (1.3, 6.4381, 0, 0.8, 0.961538), "x5": (0.9, 3.89361, 0, 0.95, 1.16959)})
_RNA_F4 = _table({"s5": (0.9, 3.89361, 0, 0.95, 1.16959), "sB": (1.3, 6.4381, 0, 0.8, 0.961538),
                  "h1": (1.5, 4.16038, 0, 0.7, 0.952381), "h2": (1.5, 4.16038, 0, 0.7, 0.952381), "h4": (0.46, 0.133855, PI, 0.7, 3.10559),
                  "h7": (4.0, 17.0526, PI * 0.5, 0.45, 0.555556),
                  "c1": (2.25, 7.00545, 0.505, 0.58, 0.766284), "c2": (1.7, 6.2469, 1.266, 0.68, 0.865052), "c7": (1.7, 6.2469, 0.309, 0.68, 0.865052),
                  "x1": (2.0, 10.9032, 2.592, 0.65, 0.769231), "x4": (1.3, 6.4381, 0.151, 0.8, 0.961538), "x5": (0.9, 3.89361, 0.685, 0.95, 1.16959)})
# (a, rc, r0, b_low, b_high, r_low, r_high, rc_low, rc_high) of the Morse factors f1: hydrogen bonding, stacking
_DNA_F1 = _table({"h": (8, 0.75, 0.4, -126.243, -7.87708, 0.34, 0.7, 0.276908, 0.783775),
                  "s": (6, 0.9, 0.4, -68.1857, -3.12992, 0.32, 0.75, 0.23239, 0.956)})
_RNA_F1 = _table({"h": (8, 0.75, 0.4, -126.243, -7.87708, 0.34, 0.7, 0.276908, 0.783775),
                  "s": (6, 0.93, 0.43, -68.1857, -3.12992, 0.35, 0.78, 0.26239, 0.986)})
# (k, rc, r0, b_low, b_high, r_low, r_high, rc_low, rc_high) of the harmonic factors f2: cross stacking, coaxial stacking
_DNA_F2 = _table({"c": (47.5, 0.675, 0.575, -0.888889, -0.888889, 0.495, 0.655, 0.45, 0.7),
                  "x": (58.5, 0.6, 0.4, -2.13158, -2.13158, 0.22, 0.58, 0.177778, 0.6222222)})
_RNA_F2 = _table({"c": (59.9626, 0.6, 0.5, -0.888889, -0.888889, 0.42, 0.58, 0.375, 0.625),
                  "x": (80.0, 0.6, 0.5, -0.888889, -0.888889, 0.42, 0.58, 0.375, 0.625)})
# (sigma, r_star, b, rc) of the excluded volumes: back-back, base-base, and the two mixed site pairs
_LJ = _table({"bb": (0.70, 0.675, 892.016223343, 0.711879214356), "aa": (0.33, 0.32, 4119.70450017, 0.335388426126),
              "ab": (0.515, 0.50, 1707.30627298, 0.52329943261)})
_TERMS = ("fene", "bexc", "stck", "exc", "hb", "crst", "cxst", "dh")


def _dot(a, b):
    return (a * b).sum(-1)


def _norm(a):
    return _dot(a, a).sqrt()


def _f1(r, t, eps):
    a, rc, r0, bl, bh, lo, hi, cl, ch = t
    shift = eps * (1 - math.exp(_f(-(np.float32(rc) - np.float32(r0)) * np.float32(a)))) ** 2
    mid = eps * (1 - torch.exp(-(r - r0) * a)) ** 2 - shift
    v = torch.where(r > hi, eps * bh * (r - ch) ** 2, torch.where(r > lo, mid, eps * bl * (r - cl) ** 2))
    return torch.where((r > cl) & (r < ch), v, torch.zeros_like(v))


def _f2(r, t):
    k, rc, r0, bl, bh, lo, hi, cl, ch = t
    v = torch.where(r > hi, k * bh * (r - ch) ** 2, torch.where(r > lo, k / 2 * ((r - r0) ** 2 - (rc - r0) ** 2), k * bl * (r - cl) ** 2))
    return torch.where((r > cl) & (r < ch), v, torch.zeros_like(v))


def _acos(c):
    return torch.acos(c.clamp(-1 + 1e-15, 1 - 1e-15))


def _f4(t, p):
    a, b, t0, ts, tc = p
    d = (t - t0).abs()
    v = torch.where(d > ts, b * (tc - d) ** 2, 1 - a * d ** 2)
    return torch.where(d < tc, v, torch.zeros_like(v))


def _f4both(c, p):
    return _f4(_acos(c), p) + _f4(_acos(-c), p)


def _f5(c):
    a, b, xc, xs = 2.0, _f(10.9032), _f(-0.769231), _f(-0.65)
    v = torch.where(c < xs, b * (xc - c) ** 2, torch.where(c < 0, 1 - a * c ** 2, torch.ones_like(c)))
    return torch.where(c > xc, v, torch.zeros_like(v))


def _lj(r, p):
    s, rs, b, rc = p
    r2 = _dot(r, r)
    rm = r2.sqrt()
    l = (s * s / r2.clamp_min(1e-4)) ** 3
    v = torch.where(rm > rs, 2 * b * (rm - rc) ** 2, 8 * (l * l - l))
    return torch.where(rm < rc, v, torch.zeros_like(v))


class _Exact:
    """Independent systems of one model in 64 bits."""

    def __init__(self, ss, model):
        self.rna = model == "RNA2"
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        put = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=self.dev)  # noqa: E731
        sizes = [s.N for s in ss]
        first = np.concatenate([[0], np.cumsum(sizes)])
        self.sizes, self.first, self.n = sizes, first, int(first[-1])
        self.temps = [float(s.T) for s in ss]
        self.sys = put(np.repeat(np.arange(len(ss)), sizes))
        self.idx = put(np.concatenate([np.arange(m) for m in sizes]))
        self.box = put(np.stack([s.box for s in ss]).astype(np.float64))
        self.bt = put(np.concatenate([s.btype for s in ss]).astype(np.int64))
        n3 = np.concatenate([np.where(s.n3 >= 0, s.n3 + f, -1) for s, f in zip(ss, first)])
        n5 = np.concatenate([np.where(s.n5 >= 0, s.n5 + f, -1) for s, f in zip(ss, first)])
        self.n3, self.n5 = put(n3), put(n5)
        p = np.nonzero(n3 >= 0)[0]
        self.bond = put(p), put(n3[p])
        self.charge = put(np.where((n3 < 0) | (n5 < 0), 0.5, 1.0))
        t = np.array(self.temps)
        salt = np.array([float(np.float32(s.salt)) for s in ss])
        lf, q = (0.3667258, 0.0858) if self.rna else (0.3616455, 0.0543)
        l32 = lf * np.sqrt(t / _f(0.1)) / np.sqrt(salt)
        lam, hi = (l32 if self.rna else lf * np.sqrt(t / 0.1) / np.sqrt(salt)), 3.0 * l32
        b = np.exp(-hi / lam) * q * q * (hi + lam) ** 2 / (4 * hi ** 3 * lam ** 2 * q)
        rc = hi * (q * hi + 3 * q * lam) / (q * (hi + lam))
        self.dh = put(np.stack([lam, hi, b, rc, np.full(len(ss), q)]))
        self.eps_s = put(_f(1.40206) + _f(2.77) * t if self.rna else _f(1.3523) + _f(2.6717) * t)
        arm = math.hypot(0.4, 0.2) if self.rna else math.hypot(0.34, 0.3408)
        self.reach, self.close = float(rc.max()) + 2 * arm, 1.7

    def sites(self, ax):
        a1, a2, a3 = ax
        if self.rna:
            return {"back": _f(-0.4) * a1 + _f(0.2) * a3, "stack": _f(0.34) * a1, "base": _f(0.4) * a1, "s3": _f(0.4) * a1 + _f(0.1) * a2,
                    "s5": _f(0.124906078525) * a1 + _f(-0.00866274917473) * a2,
                    "b3": _f(-0.462510) * a1 + _f(-0.528218) * a2 + _f(0.712089) * a3, "b5": _f(-0.104402) * a1 + _f(-0.841783) * a2 + _f(0.529624) * a3}
        return {"back": _f(-0.34) * a1 + _f(0.3408) * a2, "stack": _f(0.34) * a1, "base": _f(0.4) * a1}

    def image(self, pos, p, q):
        d, box = pos[q] - pos[p], self.box[self.sys[p]]
        return d - box * torch.round(d / box)

    def pairs(self, pos, margin):
        """Unbonded pairs p < q of one system with centres within reach + margin, and which of them are within the close range + margin."""
        got, close, r2 = [], [], (self.reach + margin) ** 2
        for s, m in enumerate(self.sizes):
            f, box = int(self.first[s]), self.box[s]
            x = pos[f: f + m]
            rows = max(1, (1 << 26) // m)
            for a in range(0, m, rows):
                e = min(a + rows, m)
                d2 = torch.zeros((e - a, m - a), dtype=torch.float64, device=self.dev)
                for k in range(3):
                    d = x[None, a:, k] - x[a:e, None, k]
                    d2 += (d - box[k] * torch.round(d / box[k])) ** 2
                i, j = torch.nonzero((d2 < r2).triu_(1), as_tuple=True)
                near = d2[i, j] < (self.close + margin) ** 2
                i, j = i + f + a, j + f + a
                keep = (self.n3[i] != j) & (self.n5[i] != j)
                got.append(torch.stack([i[keep], j[keep]]))
                close.append(near[keep])
        pq, close = torch.cat(got, 1), torch.cat(close)
        return (pq[0], pq[1]), (pq[0][close], pq[1][close])

    def bonded(self, ax, p, q, r):
        F1, F4 = (_RNA_F1, _RNA_F4) if self.rna else (_DNA_F1, _DNA_F4)
        a, b = [v[p] for v in ax], [v[q] for v in ax]
        sp, sq = self.sites(a), self.sites(b)
        rback = r + sq["back"] - sp["back"]
        x = _norm(rback) - _f(0.761070781051 if self.rna else 0.7564)
        out = {"fene": -torch.log(1 - x * x / 0.0625)}
        out["bexc"] = (_lj(r + sq["base"] - sp["base"], _LJ["aa"]) + _lj(r + sq["back"] - sp["base"], _LJ["ab"]) +
                       _lj(r + sq["base"] - sp["back"], _LJ["ab"]))
        rs = r + (sq["s5"] - sp["s3"] if self.rna else sq["stack"] - sp["stack"])
        rm = _norm(rs)
        d = rs / rm[:, None]
        radial = _f1(rm, F1["s"], self.eps_s[self.sys[p]])
        c5, c6 = _dot(a[2], d), -_dot(b[2], d)
        if not self.rna:
            ref = r + _f(-0.4) * (b[0] - a[0])
            ref = ref / _norm(ref)[:, None]
            out["stck"] = (radial * _f4(_acos(_dot(a[2], b[2])), F4["s4"]) * _f4(_acos(-c5), F4["s5"]) * _f4(_acos(c6), F4["s5"]) *
                           _f5(_dot(a[1], ref)) * _f5(_dot(b[1], ref)))
            return out
        u = rback / _norm(rback)[:, None]
        angles = radial * _f4(PI - _acos(c5), F4["s5"]) * _f4(_acos(c6), F4["s5"]) * _f5(_dot(a[1], u))
        phi2 = _f5(_dot(b[1], u))
        backs = _f4(_acos(-_dot(u, sp["b3"])), F4["sB"]) * _f4(_acos(-_dot(u, sq["b5"])), F4["sB"])
        e = angles * phi2 * backs
        # the model's force takes the phi2 derivative without the two backbone angles' factors
        out["stck"] = e + torch.where(e != 0, angles * (1 - backs), torch.zeros_like(e)).detach() * (phi2 - phi2.detach())
        return out

    def near(self, ax, p, q, r):
        F1, F2, F4 = (_RNA_F1, _RNA_F2, _RNA_F4) if self.rna else (_DNA_F1, _DNA_F2, _DNA_F4)
        a, b = [v[p] for v in ax], [v[q] for v in ax]
        sp, sq = self.sites(a), self.sites(b)
        base, back = r + sq["base"] - sp["base"], r + sq["back"] - sp["back"]
        out = {"exc": _lj(base, _LJ["aa"]) + _lj(r + sq["back"] - sp["base"], _LJ["ab"]) + _lj(r + sq["base"] - sp["back"], _LJ["ab"]) +
               _lj(back, _LJ["bb"])}
        rm = _norm(base)
        d = base / rm[:, None]
        t1, t2, t3 = _acos(-_dot(a[0], b[0])), _acos(-_dot(b[0], d)), _acos(_dot(a[0], d))
        c4, c7, c8 = _dot(a[2], b[2]), -_dot(b[2], d), _dot(a[2], d)
        hb = (_f1(rm, F1["h"], _f(0.870439 if self.rna else 1.0678)) * _f4(t1, F4["h1"]) * _f4(t2, F4["h2"]) * _f4(t3, F4["h2"]) *
              _f4(_acos(c4), F4["h4"]) * _f4(_acos(c7), F4["h7"]) * _f4(_acos(c8), F4["h7"]))
        out["hb"] = torch.where(self.bt[p] + self.bt[q] == 3, hb, torch.zeros_like(hb))
        both = (lambda c, k: _f4(_acos(c), k) + _f4(PI - _acos(c), k)) if self.rna else _f4both
        out["crst"] = _f2(rm, F2["c"]) * _f4(t1, F4["c1"]) * _f4(t2, F4["c2"]) * _f4(t3, F4["c2"]) * both(c7, F4["c7"]) * both(c8, F4["c7"])
        if not self.rna:
            out["crst"] = out["crst"] * both(c4, F4["c4"])
        rs = r + sq["stack"] - sp["stack"]
        rm = _norm(rs)
        d = rs / rm[:, None]
        x1 = _f4(t1, F4["x1"])
        if self.rna:
            other = _f4(2 * PI - t1, F4["x1"])
            x1 = x1 + 2 * other.detach() - other   # the sign that the model's force gives the reflected angle
        else:
            pi, quarter = np.float32(PI), np.float32(0.25)
            sb = float(pi - np.float32(0.1) * (pi - (pi - quarter)))
            x1 = x1 + torch.where(t1 >= sb, 20.0 * (t1 - sb) ** 2, torch.zeros_like(t1))
        out["cxst"] = _f2(rm, F2["x"]) * x1 * _f4(_acos(c4), F4["x4"]) * both(_dot(a[2], d), F4["x5"]) * both(-_dot(b[2], d), F4["x5"])
        if self.rna:
            u = back / _norm(back)[:, None]
            out["cxst"] = out["cxst"] * _f5(_dot(d, torch.cross(u, a[0], dim=1))) * _f5(_dot(d, torch.cross(u, b[0], dim=1)))
        return out

    def far(self, ax, p, q, r):
        a, b = [v[p] for v in ax], [v[q] for v in ax]
        rm = _norm(r + self.sites(b)["back"] - self.sites(a)["back"])
        lam, hi, bb, rc, pre = self.dh[:, self.sys[p]]
        v = torch.where(rm < hi, pre * torch.exp(-rm / lam) / rm, bb * (rm - rc) ** 2)
        return {"dh": torch.where(rm < rc, v, torch.zeros_like(v)) * self.charge[p] * self.charge[q]}

    def forces(self, pos, quat, lists):
        """Lab forces, body torques, each particle's energies by term, and the virial: the derivatives of the energy by every pair's
        separation and every particle's rotation."""
        axes = _axes(quat)
        n = self.n
        F, T = torch.zeros((n, 3), dtype=torch.float64, device=self.dev), torch.zeros((n, 3), dtype=torch.float64, device=self.dev)
        share = {k: torch.zeros(n, dtype=torch.float64, device=self.dev) for k in _TERMS}
        virial = torch.zeros((3, 3), dtype=torch.float64, device=self.dev)
        everything, close = lists
        for term, (p, q), chunk in ((self.bonded, self.bond, 1 << 20), (self.near, close, 1 << 21), (self.far, everything, 1 << 23)):
            for a in range(0, len(p), chunk):
                i, j = p[a: a + chunk], q[a: a + chunk]
                r0 = self.image(pos, i, j)
                r = r0.clone().requires_grad_(True)
                turn = torch.zeros((n, 3), dtype=torch.float64, device=self.dev, requires_grad=True)
                ax = [v + torch.cross(turn, v, dim=1) for v in axes]
                e = term(ax, i, j, r)
                gr, gt = torch.autograd.grad(sum(v.sum() for v in e.values()), (r, turn))
                F.index_add_(0, i, gr).index_add_(0, j, -gr)
                T -= gt
                virial -= (r0.t()[:, None, :] * gr.t()[None, :, :]).sum(-1)
                for k, v in e.items():
                    share[k].index_add_(0, i, 0.5 * v.detach()).index_add_(0, j, 0.5 * v.detach())
        body = torch.stack([_dot(v, T) for v in axes], 1)
        return F, body, share, virial


def _axes(q):
    x, y, z, w = q.unbind(1)
    return (torch.stack([x * x - y * y - z * z + w * w, 2 * (x * y + z * w), 2 * (x * z - y * w)], 1),
            torch.stack([2 * (x * y - z * w), -x * x + y * y - z * z + w * w, 2 * (y * z + x * w)], 1),
            torch.stack([2 * (x * z + y * w), 2 * (y * z - x * w), -x * x - y * y + z * z + w * w], 1))


def _turned(q, L):
    """The quaternions after one drift: the rotation of angle dt |L| about L, in the body frame."""
    norm = _norm(L)
    k = torch.where(norm > 0, torch.sin(0.5 * DT * norm) / norm.clamp_min(1e-300), torch.zeros_like(norm))
    bx, by, bz = (L * k[:, None]).unbind(1)
    bw = torch.cos(0.5 * DT * norm)
    x, y, z, w = q.unbind(1)
    out = torch.stack([w * bx + x * bw + y * bz - z * by, w * by - x * bz + y * bw + z * bx, w * bz + x * by - y * bx + z * bw,
                       w * bw - x * bx - y * by - z * bz], 1)
    return out / _norm(out)[:, None]


_M32 = 0xFFFFFFFF


def _philox(c, k):
    """Philox4x32-10 on 64-bit integers (tensors, or Python's own masked to 64 bits)."""
    c0, c1, c2, c3 = c
    k0, k1 = k
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & _M32) ^ c1 ^ k0, p1 & _M32, ((p0 >> 32) & _M32) ^ c3 ^ k1, p0 & _M32
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c0, c1, c2, c3


def _unit(x):
    return (x + 0.5) * 2.0 ** -32


def _gauss(a, b):
    r = (-2.0 * _unit(a).log()).sqrt() if torch.is_tensor(a) else math.sqrt(-2.0 * math.log(_unit(a)))
    t = 2.0 * math.pi * _unit(b)
    return (r * t.cos(), r * t.sin()) if torch.is_tensor(a) else (r * math.cos(t), r * math.sin(t))


class _Noise:
    def __init__(self, ex, seeds):
        self.ex = ex
        lo, hi = [s & _M32 for s in seeds], [((s >> 32) & _M32) ^ 0x6F78444E for s in seeds]
        self.keys = list(zip(lo, hi))
        keys = torch.tensor([lo, hi], dtype=torch.int64, device=ex.dev)
        self.key = keys[0][ex.sys], keys[1][ex.sys]

    def words(self, step, stream):
        z = torch.zeros_like(self.ex.idx)
        return _philox((self.ex.idx, z + step, z, z + stream), self.key)

    def normals(self, step, stream):
        w = self.words(step, stream)
        return torch.stack([*_gauss(w[0].double(), w[1].double()), *_gauss(w[2].double(), w[3].double())], 1)

    def one(self, s, idx, step, stream):
        return _philox((idx, step & _M32, 0, stream), self.keys[s])

    def gamma(self, s, step, stream, a):
        # G. Marsaglia and W. W. Tsang, ACM TOMS 26 (2000)
        d = a - 1.0 / 3.0
        c = 1.0 / math.sqrt(9.0 * d)
        for it in range(1000):
            w = self.one(s, 0xFFFF0000 + it, step, stream)
            x = _gauss(w[0], w[1])[0]
            v = (1.0 + c * x) ** 3
            if v > 0 and math.log(_unit(w[2])) < 0.5 * x * x + d - d * v + d * math.log(v):
                return d * v
        return d

    def chi2(self, s, step, stream, n):
        w = self.one(s, 0xFFFE0000, step, stream)
        extra = _gauss(w[0], w[1])[0] ** 2 if n % 2 else 0.0
        return extra if n <= 1 else 2.0 * self.gamma(s, step, stream, n // 2) + extra


def _trajectory(ex, state, opts, seeds, steps):
    """`steps` velocity-Verlet steps with the thermostat of `opts`."""
    pos, quat, vel, L = state
    noise, th, ns, temps = _Noise(ex, seeds), opts["thermostat"], opts.get("newtonian_steps", 1), ex.temps
    T = torch.tensor(temps, dtype=torch.float64, device=ex.dev)[ex.sys][:, None]
    D = _f(DIFF)
    # pairs that may come into range during the run: a strand end's drift, and in large systems the short runs' smaller one
    lists = ex.pairs(pos, 1.0 + (1.5 * DT * steps if ex.n < 20000 else 0.0))
    F, tau = ex.forces(pos, quat, lists)[:2]
    K = [[0.5 * 3.0 * (n - 1) * t, 0.5 * 3.0 * n * t] for n, t in zip(ex.sizes, temps)]
    for step in range(steps):
        vel, L = vel + F * (0.5 * DT), L + tau * (0.5 * DT)
        pos, quat = pos + vel * DT, _turned(quat, L)
        F, tau = ex.forces(pos, quat, lists)[:2]
        vel, L = vel + F * (0.5 * DT), L + tau * (0.5 * DT)
        if th == "langevin":
            n = torch.cat([noise.normals(step, 0), noise.normals(step, 1)], 1)
            gt, gr = T / D, T / (3.0 * D)
            vel = vel + DT * (-gt * vel + n[:, 0:3] * (2.0 * gt * T / DT).sqrt())
            L = L + DT * (-gr * L + n[:, 3:6] * (2.0 * gr * T / DT).sqrt())
        elif th == "john" and step % ns == 0:
            h = T * ns * _f(DT)
            pt = 2 * h / (h + 2 * D)
            d = h * (1 / pt - 0.5)
            pr = 2 * h / (h + 6 * d)
            u = noise.words(step, 2)
            n0, n1 = noise.normals(step, 3), noise.normals(step, 8)
            vel = torch.where(_unit(u[0].double())[:, None] < pt, n0[:, :3] * T.sqrt(), vel)
            L = torch.where(_unit(u[1].double())[:, None] < pr, n1[:, :3] * T.sqrt(), L)
        elif th == "bussi" and step % ns == 0:
            c = math.exp(-ns / float(opts["bussi_tau"]))
            vel, L = vel.clone(), L.clone()
            for s, (n, t) in enumerate(zip(ex.sizes, temps)):
                own = slice(int(ex.first[s]), int(ex.first[s]) + n)
                vc = vel[own].mean(0)
                now = [0.5 * float((vel[own] ** 2).sum()) - 0.5 * n * float((vc ** 2).sum()), 0.5 * float((L[own] ** 2).sum())]
                for k, dof in enumerate((3 * (n - 1), 3 * n)):
                    w = noise.one(s, 0xFFFD0000, step, 6 + 4 * k)
                    rr, target = _gauss(w[0], w[1])[0], 0.5 * dof * t
                    K[s][k] += ((1 - c) * (target * (noise.chi2(s, step, 7 + 4 * k, dof - 1) + rr * rr) / dof - K[s][k]) +
                                2.0 * rr * math.sqrt(K[s][k] * target / dof * (1 - c) * c))
                vel[own] = vc + (vel[own] - vc) * math.sqrt(K[s][0] / now[0])
                L[own] = L[own] * math.sqrt(K[s][1] / now[1])
    a1, _, a3 = _axes(quat)
    return dict(pos=pos, a1=a1, a3=a3, vel=vel, L=L)


def _start(ex, ss):
    put = lambda v: torch.as_tensor(v, device=ex.dev)  # noqa: E731
    a1, a3 = np.concatenate([s.a1 for s in ss]), np.concatenate([s.a3 for s in ss])
    m = np.stack([a1, np.cross(a3, a1), a3], 2)
    # the eigenvector of the largest eigenvalue of the frame's quaternion form
    k = np.zeros((len(m), 4, 4))
    for i in range(3):
        j, l = (i + 1) % 3, (i + 2) % 3
        k[:, i, i] = m[:, i, i] - m[:, j, j] - m[:, l, l]
        k[:, i, j] = k[:, j, i] = m[:, i, j] + m[:, j, i]
        k[:, i, 3] = k[:, 3, i] = m[:, l, j] - m[:, j, l]
    k[:, 3, 3] = m[:, 0, 0] + m[:, 1, 1] + m[:, 2, 2]
    quat = np.linalg.eigh(k)[1][:, :, 3]
    return put(np.concatenate([s.pos for s in ss])), put(quat), put(np.concatenate([s.vel for s in ss])), put(np.concatenate([s.L for s in ss]))


def exact(case, seed):
    ss = _systems(case, seed)
    opts, per = _options(case, seed)
    seeds = [o["seed"] for o in per]
    kind = case["kind"]
    if kind == "pool":
        got = []
        for s, one, steps in zip(ss, seeds, _job_steps(case)):
            ex = _Exact([s], case["model"])
            got.append(_trajectory(ex, _start(ex, [s]), opts, [one], steps))
        return dict({k: torch.cat([g[k] for g in got]) for k in got[0]}, done=None)
    ex = _Exact(ss, case["model"])
    if kind == "md":
        return _trajectory(ex, _start(ex, ss), opts, seeds, case["steps"])
    pos, quat, vel, L = _start(ex, ss)
    F, T, share, virial = ex.forces(pos, quat, ex.pairs(pos, 0.0))
    E = sum(share.values())
    if kind != "observe":
        return {"F": torch.cat([F, E[:, None]], 1), "T": torch.cat([T, share["hb"][:, None]], 1)}
    six = lambda m: torch.stack([m[0, 0], m[1, 1], m[2, 2], m[0, 1], m[0, 2], m[1, 2]])  # noqa: E731
    energies = torch.stack([E.sum(), share["hb"].sum(), 0.5 * (vel ** 2).sum(), 0.5 * (L ** 2).sum()])[None]
    return dict(energies=energies, split=torch.stack([share[k].sum() for k in _TERMS]), virial=six(virial),
                kinetic=six((vel.t()[:, None, :] * vel.t()[None, :, :]).sum(-1)), F=F, T=T, E=E, hb=None)
