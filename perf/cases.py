"""Performance cases: what a program that uses this framework has it do, through
the public entry points of picard_amd.host and picard_amd.ensemble.

Five kinds of work:

* ``step``      one pass of the main loop (BCinflow on the device, then
                Domain.step), and the potential, the field and the densities
                read back, as a host does that watches or stores every step.
* ``poisson``   the field solve alone: a given charge, every boundary open,
                BCpotentials and CalcEpotential to a tight tolerance.
* ``cycle``     the particle side of the loop in a given field, through the
                single entry points: inflow, push, outflow, wrap, deposit and
                velocity update, and the densities read back.
* ``gridify``   the deposit of particles that the host handed over.
* ``ensemble``  one step of many independent simulations, and their potentials
                and fields read back.

Precision forms: ``fp64`` (the reference's summation orders), ``order_free``
(FP64, fixed-point deposit and FFT face sums) and ``split`` (FP32-split).  The
split form and the ensemble hold offsets, velocities and E in 32 bits, so their
users keep the fields as float32; the FP64 forms' fields stay float64.
"""
from __future__ import annotations

import math
import random

import numpy as np

from picard_amd import _lib, ensemble, host

CELL = 10.0                  # cell edge [m], as in every workload of this repository
EPS0 = 8.854187817e-12
FORMS = {"fp64": dict(precision=_lib.PICARD_FP64),
         "order_free": dict(precision=_lib.PICARD_FP64, order_free=True),
         "split": dict(precision=_lib.PICARD_FP32_SPLIT)}
PARTICLE_BYTES = {"fp64": 68, "order_free": 68, "split": 35}


def listed():
    return [
        # the smallest domain that the tests step: launches and latency
        dict(name="step_16_split", kind="step", form="split", nx=16, ny=16, nz=16, ppc=8,
             flow="x", haser=False),
        # the 32^3 workload (config1), in the form that reproduces the reference bit for bit
        dict(name="step_32_fp64", kind="step", form="fp64", nx=32, ny=32, nz=32, ppc=8,
             flow="x", haser=False),
        # an uneven box, every boundary open, no edge a multiple of anything
        dict(name="step_odd_split", kind="step", form="split", nx=53, ny=38, nz=45, ppc=6,
             flow="xyz", haser=False),
        # a middle-sized run in FP64 whose user does not need the reference's orders
        dict(name="step_64_order_free", kind="step", form="order_free", nx=64, ny=64, nz=64,
             ppc=12, flow="x", haser=False),
        # the same size in the reference's orders, with the Haser source
        dict(name="step_64_fp64_haser", kind="step", form="fp64", nx=64, ny=64, nz=64, ppc=12,
             flow="x", haser=True),
        # the large single-domain workload (config2) at the size that fits a pass of this file
        dict(name="step_160_split_haser", kind="step", form="split", nx=160, ny=160, nz=160,
             ppc=32, flow="x", haser=True),
        # the Poisson workload (config3) at a quarter of its edge
        dict(name="poisson_128_split", kind="poisson", form="split", nx=128, ny=128, nz=128,
             maxerr=1e-10),
        # the same in FP64 on an uneven box with an odd edge
        dict(name="poisson_odd_fp64", kind="poisson", form="fp64", nx=49, ny=72, nz=60,
             maxerr=1e-8),
        # the particle side of the large workload: 1.3e8 particles
        dict(name="cycle_128_split", kind="cycle", form="split", nx=128, ny=128, nz=128, ppc=32,
             flow="x"),
        # the particle side in the reference's orders, y open too
        dict(name="cycle_64_fp64", kind="cycle", form="fp64", nx=64, ny=60, nz=68, ppc=16,
             flow="xy"),
        # particles that a host appended, deposited as the reference would
        dict(name="gridify_host_fp64", kind="gridify", form="fp64", nx=40, ny=33, nz=28,
             particles=600_000, flow="x"),
        # a batch of small simulations, as the job server steps them
        dict(name="ensemble_24", kind="ensemble", sims=24, nmin=16, nmax=64, mix=20261210),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    n = _log_int(rng, lo, hi)
    if rng.random() < 0.5:
        return n, n, n
    return tuple(min(hi, max(8, int(n * rng.uniform(0.75, 1.3)))) for _ in range(3))


def draw(rng: random.Random):
    kind = rng.choice(["step", "step", "step", "poisson", "cycle", "gridify", "ensemble"])
    if kind == "ensemble":
        nmin = rng.randint(16, 24)
        return dict(kind=kind, sims=rng.randint(4, 24), nmin=nmin, nmax=rng.randint(nmin + 8, 64),
                    mix=rng.randint(1, 10 ** 6))
    form = rng.choice(["split", "split", "order_free", "fp64"])
    c = dict(kind=kind, form=form)
    if kind == "step":
        hi = {"split": 120, "order_free": 72, "fp64": 64}[form]
        c["nx"], c["ny"], c["nz"] = _box(rng, 16, hi)
        c["ppc"] = _log_int(rng, 4, 24)
        c["flow"] = rng.choice(["x", "x", "xy", "xyz"])
        c["haser"] = rng.random() < 0.3
    elif kind == "poisson":
        c["nx"], c["ny"], c["nz"] = _box(rng, 24, 110 if form == "split" else 64)
        c["maxerr"] = rng.choice([1e-6, 1e-8, 1e-10])
    elif kind == "cycle":
        c["nx"], c["ny"], c["nz"] = _box(rng, 24, 120 if form == "split" else 64)
        c["ppc"] = _log_int(rng, 4, 28)
        c["flow"] = rng.choice(["x", "x", "xy", "xyz"])
    else:
        c["nx"], c["ny"], c["nz"] = _box(rng, 12, 48)
        c["particles"] = _log_int(rng, 3_000, 600_000)
        c["flow"] = rng.choice(["x", "xy", "xyz"])
    return c


# ---------------------------------------------------------------------------

def _config(case, **kw):
    n = (case["nx"], case["ny"], case["nz"])
    flow = case.get("flow", "xyz")
    base = dict(nx=n[0], ny=n[1], nz=n[2], flow=tuple(d in flow for d in "xyz"),
                gmin=tuple(-0.5 * CELL * v for v in n), gmax=tuple(0.5 * CELL * v for v in n))
    if "ppc" in case:
        base["ppc"] = (0, case["ppc"], 0, 0, 0, 0, 0, 0)
    base.update(kw)
    if case.get("haser"):
        # the source of the large workload, scaled to this box: 2^18 ions a step at 256^3
        src = host.config2(256)
        share = n[0] * n[1] * n[2] / 256.0 ** 3
        base.update(species=3, Qn=tuple(q * share for q in src.Qn), vn=src.vn, nu_i=src.nu_i,
                    nu_d=src.nu_d, Ek=src.Ek)
        cfg = host.Config(**base)
        cfg.rate_scale = host.derive(cfg).dt
        return cfg
    return host.Config(**base)


def _domain(case, cfg, particles=None):
    d = host.derive(cfg)
    if particles is None:
        per_cell = int(d.ppc[:cfg.species].sum())
        particles = int(1.12 * per_cell * cfg.nx * cfg.ny * cfg.nz) + (1 << 18)
        faces = ((cfg.ny + 2) * (cfg.nz + 2) + (cfg.nx + 2) * (cfg.nz + 2) +
                 (cfg.nx + 2) * (cfg.ny + 2))
        particles += 8 * per_cell * faces
        particles += (1 << 20) if case.get("haser") else 0
    return host.Domain(cfg, max_particles=particles, d=d, **FORMS[case["form"]])


def _charge(case, rng):
    """The Poisson workload's charge [C per cell]: 16 Gaussian blobs (sigma 4-20
    cells, amplitudes up to 1e-3 of the plasma's) and the Haser profile, its
    source anywhere in the middle half of the box."""
    n = (case["nx"], case["ny"], case["nz"])
    ax = [CELL * (np.arange(v) + 0.5 - 0.5 * v) for v in n]
    amp = 1e-3 * host.EC * 5.0e6
    rho = np.zeros(n[::-1])
    for _ in range(16):
        sig = rng.uniform(4.0, 20.0) * CELL
        g = [np.exp(-(a - rng.uniform(-0.5, 0.5) * CELL * v) ** 2 / (2 * sig * sig))
             for a, v in zip(ax, n)]
        rho += rng.uniform(-amp, amp) * (g[2][:, None, None] * g[1][None, :, None] * g[0])
    x0, y0, z0 = (rng.uniform(-0.25, 0.25) * CELL * v for v in n)
    r2 = ((ax[2] - z0)[:, None, None] ** 2 + (ax[1] - y0)[None, :, None] ** 2 + (ax[0] - x0) ** 2)
    r2 = np.maximum(r2, (0.25 * CELL) ** 2)
    rho += host.EC * host.HASER_Q_STATED / (4 * math.pi * r2 * 1.0e3) * np.exp(-np.sqrt(r2) / 1.0e6)
    C = np.zeros(tuple(v + 2 for v in n[::-1]))
    C[1:-1, 1:-1, 1:-1] = rho * CELL ** 3
    return C


def _host_particles(case, rng):
    """Electrons and H+ spread over the box, as a host hands them over."""
    n = (case["nx"], case["ny"], case["nz"])
    m = case["particles"]
    rp = np.zeros((m, 8))
    for q in range(3):
        rp[:, q] = (rng.random(m) - 0.5) * CELL * n[q]
    rp[:, 3:6] = rng.normal(size=(m, 3)) * 1.0e6
    sp = rng.integers(1, 3, m).astype(np.int32)
    return rp, sp


def _potential(cfg, rng):
    """A smooth potential of about a volt, periodic in every direction."""
    out = np.zeros((cfg.nz + 2, cfg.ny + 2, cfg.nx + 2))
    for _ in range(6):
        w = 1.0
        for q, v in ((2, cfg.nx), (1, cfg.ny), (0, cfg.nz)):
            ph = 2 * math.pi * (int(rng.integers(1, 5)) * (np.arange(v + 2) - 1) / v + rng.random())
            w = w * np.cos(ph).reshape([-1 if a == q else 1 for a in range(3)])
        out += rng.uniform(-0.5, 0.5) * w
    return out


def _specs(case, seed):
    specs = ensemble.draw_ensemble(case["sims"], seed=case["mix"], nmin=case["nmin"],
                                   nmax=case["nmax"])
    rng = np.random.default_rng(seed)
    for s in specs:
        s.seed = int(rng.integers(1, 2 ** 62))
    return specs


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    key = int(rng.integers(1, 2 ** 62))
    st = dict(case=case, key=key, it=0)
    kind = case["kind"]
    if kind == "ensemble":
        specs = _specs(case, seed)
        ens = ensemble.Ensemble.sized_for(specs, steps_room=24)
        st.update(ens=ens, slots=[ens.add(s) for s in specs])
        return st
    if kind == "poisson":
        cfg = _config(case, maxerr=case["maxerr"])
        dom = _domain(case, cfg, particles=1024)
        dom.calc_distance()
        dom.set_field(_lib.FIELD_C, _charge(case, rng))
    elif kind == "gridify":
        cfg = _config(case)
        dom = _domain(case, cfg, particles=case["particles"])
        dom.append(*_host_particles(case, rng))
    else:
        cfg = _config(case)
        dom = _domain(case, cfg)
        dom.generate_initial(key)
        if kind == "cycle":
            dom.set_field(_lib.FIELD_U, _potential(cfg, rng))
            dom.calc_efield()
            dom.bc_fields()
        else:
            dom.calc_distance()
            if case["haser"]:
                dom.set_production(key)
    dom.synchronize()
    st["dom"] = dom
    return st


def _field(st, which):
    a = st["dom"].field(which)
    return a.astype(np.float32) if st["case"]["form"] == "split" else a


def run(st):
    kind = st["case"]["kind"]
    st["it"] += 1
    if kind == "ensemble":
        ens = st["ens"]
        ens.step()
        return {name: np.concatenate([ens.field(s, w).ravel() for s in st["slots"]]).astype(np.float32)
                for name, w in (("phi", _lib.FIELD_U), ("E", _lib.FIELD_E))}
    dom = st["dom"]
    if kind == "poisson":
        dom.bc_potentials()
        dom.calc_epotential()
        return {"phi": _field(st, _lib.FIELD_U)}
    if kind == "gridify":
        dom.particles_gridify()
        return {"N": _field(st, _lib.FIELD_N), "C": _field(st, _lib.FIELD_C)}
    dom.generate_inflow(st["key"], st["it"])
    if kind == "cycle":
        dom.advance_position()
        n, _ = dom.bc_outflow()
        dom.particles_transfer()
        dom.particles_gridify()
        dom.advance_velocity()
        return {"N": _field(st, _lib.FIELD_N), "C": _field(st, _lib.FIELD_C), "num_local": n}
    s = dom.step()
    return {"phi": _field(st, _lib.FIELD_U), "E": _field(st, _lib.FIELD_E),
            "N": _field(st, _lib.FIELD_N), "num_local": int(s.num_local)}


def work(case):
    """Bytes: the particles read and written once and each grid that is handed
    in or out moved once.  Operations: about 300 a particle for the whole cycle
    (push, weights, deposit, gather, rotation) and 30 for the deposit alone; a
    field solve by transforms along the three edges, the cheapest way known."""
    if case["kind"] == "ensemble":
        b = f = 0.0
        for s in _specs(case, 1):
            p = 2.0 * s.ppc * s.cells
            g = (s.nx + 2.0) * (s.ny + 2) * (s.nz + 2)
            b += 2 * 35 * p + 20 * g
            f += 300 * p + 12 * s.cells * (s.nx + s.ny + s.nz) / 3.0
        return {"bytes": b, "flops": f}
    n = (case["nx"], case["ny"], case["nz"])
    cells = float(n[0] * n[1] * n[2])
    nodes = (n[0] + 2.0) * (n[1] + 2) * (n[2] + 2)
    solve = 4 * cells * sum(n)
    species = 3 if case.get("haser") else 2
    if case["kind"] == "poisson":
        return {"bytes": 16 * nodes, "flops": solve}
    if case["kind"] == "gridify":
        return {"bytes": 28.0 * case["particles"] + 8 * 3 * nodes, "flops": 30.0 * case["particles"]}
    p = 2.0 * case["ppc"] * cells
    pb = 2 * PARTICLE_BYTES[case["form"]] * p
    if case["kind"] == "cycle":
        return {"bytes": pb + 8 * 3 * nodes + 24 * nodes, "flops": 300 * p}
    return {"bytes": pb + 8 * (4 + species) * nodes, "flops": 300 * p + solve}


# ---------------------------------------------------------------------------
# the same in 64 bits with numpy

def _face_sums(C):
    """BCpotentials with every boundary open: the face nodes' Coulomb sums over
    the interior cells, as one linear convolution per plane of charge."""
    q = C[1:-1, 1:-1, 1:-1]
    U = np.zeros_like(C)
    k = 1.0 / (4.0 * math.pi * EPS0)
    for axis in range(3):
        p = np.moveaxis(q, axis, 0)
        m, a, b = p.shape
        L = (2 * a, 2 * b)
        da = np.minimum(np.arange(L[0]), L[0] - np.arange(L[0]))
        db = np.minimum(np.arange(L[1]), L[1] - np.arange(L[1]))
        r2 = (da[:, None] ** 2 + db[None, :] ** 2) * CELL ** 2
        lo = np.zeros((L[0], b + 1), complex)
        hi = np.zeros_like(lo)
        for s in range(m):
            F = np.fft.rfft2(p[s], L)
            lo += F * np.fft.rfft2(1.0 / np.sqrt(r2 + ((s + 1) * CELL) ** 2))
            hi += F * np.fft.rfft2(1.0 / np.sqrt(r2 + ((m - s) * CELL) ** 2))
        V = np.moveaxis(U, axis, 0)
        V[0, 1:-1, 1:-1] = k * np.fft.irfft2(lo, L)[:a, :b]
        V[-1, 1:-1, 1:-1] = k * np.fft.irfft2(hi, L)[:a, :b]
    return U


def _poisson(C):
    """The solution of the seven-point equation with those face values, by sine
    transforms; the solve stops within its tolerance of it."""
    U = _face_sums(C)
    r = -C[1:-1, 1:-1, 1:-1] / (CELL ** 3 * EPS0) * CELL ** 2
    r[0] -= U[0, 1:-1, 1:-1]
    r[-1] -= U[-1, 1:-1, 1:-1]
    r[:, 0] -= U[1:-1, 0, 1:-1]
    r[:, -1] -= U[1:-1, -1, 1:-1]
    r[:, :, 0] -= U[1:-1, 1:-1, 0]
    r[:, :, -1] -= U[1:-1, 1:-1, -1]
    lam, Q = [], []
    for m in r.shape:
        i = np.arange(1, m + 1)
        Q.append(np.sqrt(2.0 / (m + 1)) * np.sin(np.pi * np.outer(i, i) / (m + 1)))
        lam.append(4.0 * np.sin(0.5 * np.pi * i / (m + 1)) ** 2)

    def transform(a):
        for axis in range(3):
            a = np.moveaxis(np.tensordot(Q[axis], a, (1, axis)), 0, axis)
        return a

    h = transform(r) / -(lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :])
    U[1:-1, 1:-1, 1:-1] = transform(h)
    return U


def _fold(N, flow):
    """The guard planes' weights, folded in or exchanged (z, y, x)."""
    for axis, open_ in ((0, flow[2]), (1, flow[1]), (2, flow[0])):
        a = np.moveaxis(N, axis, 0)
        o1, o2, m1, m2 = (a[q].copy() for q in (0, 1, -2, -1))
        if open_:
            a[1], a[-2] = o2 + o1, m1 + m2
            a[0] = a[-1] = 0.0
        else:
            a[0], a[1], a[-2], a[-1] = o1 + m1, o2 + m2, m1 + o1, m2 + o2


def _gridify(case, seed):
    rng = np.random.default_rng(seed)
    rng.integers(1, 2 ** 62)
    rp, sp = _host_particles(case, rng)
    n = (case["nx"], case["ny"], case["nz"])
    X, Y, Z = (v + 2 for v in n)
    xi = [rp[:, q] / CELL + 0.5 * n[q] + 0.5 for q in range(3)]
    lo = [np.floor(v).astype(np.int64) for v in xi]
    f = [v - i for v, i in zip(xi, lo)]
    d = host.derive(_config(case))
    N = np.zeros((Z, Y, X, 2))
    for s in (1, 2):
        at = sp == s
        grid = np.zeros(X * Y * Z)
        for o in range(8):
            b = (o & 1, (o >> 1) & 1, o >> 2)
            w = np.ones(int(at.sum()))
            node = np.zeros(w.size, np.int64)
            for q, stride in ((0, 1), (1, X), (2, X * Y)):
                w = w * (f[q][at] if b[q] else 1.0 - f[q][at])
                node += (lo[q][at] + b[q]) * stride
            grid += np.bincount(node, w, X * Y * Z)
        N[..., s - 1] = grid.reshape(Z, Y, X) * d.n2p[s - 1]
    _fold(N, tuple(c in case["flow"] for c in "xyz"))
    return {"N": N, "C": N[..., 0] * d.charge[0] + N[..., 1] * d.charge[1]}


def exact(case, seed):
    """Whole steps, cycles and ensembles start from the framework's own device
    sources, so nothing outside it holds their inputs."""
    if case["kind"] == "poisson" and case["maxerr"] <= 1e-8:
        rng = np.random.default_rng(seed)
        rng.integers(1, 2 ** 62)
        return {"phi": _poisson(_charge(case, rng))}
    if case["kind"] == "gridify":
        return _gridify(case, seed)
    return None
