"""Timed cases of the force evaluation and the RK12 integration.

Every case is a call that a program of this framework makes: bodies resident
on the GPU are advanced to the next output epoch (or their forces are
evaluated) and the new state is read back.  Three kinds:

* ``accel``      one force evaluation of given bodies: upload, evaluate,
                 download (what an outside integrator calls per stage);
* ``integrate``  ``steps`` RK12 steps of ``systems`` independent systems and a
                 download: one output interval of an ephemeris or an ensemble;
* ``particles``  ``steps`` RK12 steps of massless particles in the field of
                 the star and eight planets, and a download.

Bodies come from the package's seeded generator: ``field9`` (star and eight
point-mass planets), ``small`` (25 bodies, Newtonian + 1PN + J2) and ``full``
(504 bodies with geopotentials, tides, a ring and radiation pressure; more
main-belt asteroids above 504), cut to the most massive ``bodies``.  Each
system of each seed gets its own relative perturbation of 1e-9 of positions
and velocities, as the members of an ensemble do.
"""
import functools
import math
import tempfile

import numpy as np
import torch

from ephemeris_amd import _lib
from ephemeris_amd import generator as gen
from ephemeris_amd.layout import GP_DTYPE, MASS_DTYPE, RING_DTYPE
from ephemeris_amd.particles import ParticleSet
from ephemeris_amd.system import GpuSystems, MSystem

DAY = 86400.0
FLOP_PAIR = 294 + 54             # main force and deformation sums of one ordered pair
FLOP_PARTICLE_STEP = 61223       # 25 stages in the nine-body field, stage combinations included


def _integrate(name, model, bodies, steps, systems=1, bodies_min=0, dt=300.0, order="pool"):
    return {"name": name, "kind": "integrate", "model": model, "bodies": bodies, "bodies_min": bodies_min or bodies,
            "systems": systems, "steps": steps, "dt": dt, "order": order}


def listed():
    return [
        # the shortest call: two daily steps of the star and eight planets
        _integrate("planets_9", "field9", 9, 2, dt=DAY),
        # an output interval of two hours of a small system without models
        _integrate("small_25", "small", 25, 24),
        # the same for a planetary system with every model, single-thread order by its size
        _integrate("full_40", "full", 40, 24),
        # the full system: an output interval of two hours, the plain single-system path
        _integrate("full_504", "full", 504, 24),
        # the full system in the single-thread summation order, asked for by the caller
        _integrate("full_504_serial", "full", 504, 2, order="serial"),
        # one force evaluation of the full system for an outside integrator
        {"name": "accel_504", "kind": "accel", "model": "full", "bodies": 504, "order": "pool"},
        # a system with more asteroids than the full one
        _integrate("full_804", "full", 804, 8),
        # a planetary-system survey: many small systems side by side
        _integrate("survey_256x25", "small", 25, 24, systems=256),
        # ensembles of uneven systems: a served job's size, and the large batch
        _integrate("ensemble_16", "full", 504, 12, systems=16, bodies_min=64),
        _integrate("ensemble_256", "full", 504, 12, systems=256, bodies_min=64),
        # test particles: a served job's size, and the large set
        {"name": "particles_20k", "kind": "particles", "particles": 20000, "steps": 8},
        {"name": "particles_1m", "kind": "particles", "particles": 1000000, "steps": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "single", "accel", "survey", "ensemble", "ensemble", "particles"])
    if kind == "particles":
        return {"kind": "particles", "particles": _log(rng, 100, 900000), "steps": rng.randint(1, 8)}
    if kind == "accel":
        return {"kind": "accel", "model": "full", "bodies": _log(rng, 12, 1000), "order": rng.choice(["pool", "pool", "serial"])}
    if kind == "single":
        n = _log(rng, 3, 1000)
        order = "serial" if n <= 504 and rng.random() < 0.2 else "pool"
        steps = rng.randint(1, 2) if order == "serial" and n > 64 else rng.randint(2, 24 if n <= 504 else 8)
        model, dt = ("small", 300.0) if n <= 25 and rng.random() < 0.5 else ("full", 300.0)
        c = _integrate("", model, n, steps, dt=dt, order=order)
    elif kind == "survey":
        c = _integrate("", rng.choice(["small", "full"]), rng.randint(4, 25), rng.randint(1, 24), systems=_log(rng, 8, 500))
    else:
        lo = rng.randint(50, 300)
        c = _integrate("", "full", rng.randint(lo, 504), rng.randint(2, 12), systems=_log(rng, 2, 200), bodies_min=lo)
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _base(model):
    """Bodies, geopotentials and rings of a generated system, as the loader gives them."""
    spec = {"field9": gen.make_field9, "small": gen.make_small, "full": gen.make_full,
            "large": lambda: gen.add_asteroids(gen.make_full(), 520)}[model]()
    with tempfile.TemporaryDirectory() as d:
        m = MSystem(gen.write_system(spec, d), analyse=False)
        out = (m.masses, *m.models())
        m.close()
    return out


def _bodies(case, seed):
    """(masses, sys_n, gps, rings) of all systems of a case."""
    masses, gps, rings = _base("large" if case["model"] == "full" and case["bodies"] > 504 else case["model"])
    rng = np.random.default_rng(seed)
    lo, hi, count = case.get("bodies_min", case["bodies"]), case["bodies"], case.get("systems", 1)
    sizes = np.random.default_rng([lo, hi, count]).integers(lo, hi + 1, size=count)
    by_mass = np.argsort(-masses["GM"], kind="stable")
    parts, all_gps, all_rings = [], [], []
    n_gp = n_ring = 0
    for n in sizes:
        m = masses[np.sort(by_mass[:n])] if n <= 504 else masses[:n].copy()
        for q in "xyz":
            m[f"r_{q}_hi"] *= 1 + 1e-9 * rng.standard_normal(len(m))
            m[f"v_{q}_hi"] *= 1 + 1e-9 * rng.standard_normal(len(m))
        # each system carries its own copy of the models that its bodies use
        for key, table, used, off in (("gp", gps, all_gps, n_gp), ("ring", rings, all_rings, n_ring)):
            has = m[key] >= 0
            used.append(table[m[key][has]])
            m[key][has] = off + np.arange(has.sum())
        n_gp += len(all_gps[-1])
        n_ring += len(all_rings[-1])
        parts.append(m)
    return (np.concatenate(parts), np.array([len(m) for m in parts], np.int64),
            np.concatenate(all_gps).astype(GP_DTYPE), np.concatenate(all_rings).astype(RING_DTYPE))


def _order(case):
    return _lib.SUMMATION_SERIAL if case["order"] == "serial" else _lib.SUMMATION_POOL


_FIELD9 = {"model": "field9", "bodies": 9, "order": "pool"}


def prepare(case, seed):
    if case["kind"] == "particles":
        r, v = gen.make_particles(case["particles"], seed=seed, field9=gen.make_field9())
        masses, sys_n, gps, rings = _bodies(_FIELD9, seed)
        field = GpuSystems(masses, sys_n, gps, rings)
        field.accel()
        return {"case": case, "set": ParticleSet(field, r, v)}
    masses, sys_n, gps, rings = _bodies(case, seed)
    g = GpuSystems(masses, sys_n, gps, rings)
    if case["kind"] == "integrate":
        g.accel(_order(case))                # the forces at the epoch, which the first stage reads
    return {"case": case, "systems": g, "masses": masses}


# ---- one pass -----------------------------------------------------------------
# groups of consecutive columns of a downloaded body, by their first field
_GROUPS = (("r", "r_x_hi", 6), ("v", "v_x_hi", 6), ("GL", "GL_x_hi", 6), ("s", "s_xx_hi", 18), ("w", "w_x", 3),
           ("GM", "GM", 1), ("exJ2", "exJ2", 1), ("phi", "phi", 1), ("beta2", "beta2", 1), ("naccel", "naccel_x", 3),
           ("daccel", "daccel_x", 3), ("dtorque", "dtorque_x", 3), ("gaccel", "gaccel_x", 3), ("beta", "beta_x", 3),
           ("GI", "GI_xx", 9), ("C_potential", "C_potential_xx", 9), ("Egrad", "Egrad_x", 3),
           ("idaccel", "idaccel_x", 12), ("min_distance", "min_distance", 1), ("max_influence", "max_influence", 1))


def _columns(masses):
    """The body fields of a download as views of shape (bodies, columns)."""
    flat = masses.view(np.float64).reshape(len(masses), -1)
    return {name: flat[:, MASS_DTYPE.fields[first][1] // 8:][:, :width] for name, first, width in _GROUPS}


def run(state):
    case = state["case"]
    if case["kind"] == "particles":
        state["set"].integrate(DAY, case["steps"])
        r, v, extrema = state["set"].download()
        return {"r": r, "v": v, "extrema": extrema}
    g = state["systems"]
    if case["kind"] == "accel":
        g.upload(state["masses"])
        g.accel(_order(case))
    else:
        g.integrate(case["dt"], case["steps"], _order(case))
    masses, t_eph = g.download()
    return {**_columns(masses), "t_eph": t_eph}


# ---- necessary work -----------------------------------------------------------
def work(case):
    if case["kind"] == "particles":
        n = case["particles"]
        return {"bytes": n * 8.0 * 2 * 17, "flops": float(n) * case["steps"] * FLOP_PARTICLE_STEP}
    lo, hi, count = case.get("bodies_min", case["bodies"]), case["bodies"], case.get("systems", 1)
    mean, var = (lo + hi) / 2, ((hi - lo + 1) ** 2 - 1) / 12
    evaluations = 25 * case["steps"] if case["kind"] == "integrate" else 1
    return {"bytes": count * mean * MASS_DTYPE.itemsize * 2.0,
            "flops": count * (mean * mean + var - mean) * FLOP_PAIR * evaluations}


# ---- the same in plain 64-bit torch --------------------------------------------
_C = 299792458.0


def _pull(r, v, GM, C, R2, soft, sources):
    """Acceleration of every body by the bodies `sources` in plain arithmetic:
    (Newton, potential, 1PN, quadrupole figures)."""
    d = r[None, sources] - r[:, None]
    d2 = torch.maximum((d * d).sum(-1), soft[:, None] + soft[None, sources])
    me = torch.zeros_like(d2, dtype=torch.bool)
    me.diagonal().fill_(True)                # a body does not pull itself
    k = torch.where(me, 0.0, 1 / torch.where(me, 1.0, d2))
    i1 = k.sqrt()
    g1 = GM[None, sources] * i1
    g3 = g1 * k
    newton, phi = (g3[..., None] * d).sum(1), -g1.sum(1)
    b = v / _C
    b2 = (b * b).sum(-1)
    bj, nj = b[None, sources], (newton / _C**2)[None, sources]
    rb, db = (d * bj).sum(-1), bj - b[:, None]
    delta = ((4 * phi[:, None] + phi[None, sources]) / _C**2 + b2[:, None] + 2 * b2[None, sources]
             - 4 * (b[:, None] * bj).sum(-1) + ((d * nj).sum(-1) - 3 * rb * rb * k) / 2)
    pn = ((3.5 * g1)[..., None] * nj + (g3 * delta)[..., None] * d + (g3 * (rb - 4 * (d * db).sum(-1)))[..., None] * db).sum(1)

    def field(Cd):                           # of a figure, Cd = C times the offset
        return ((d * Cd).sum(-1) * 5 * k)[..., None] * d - 2 * Cd

    own = torch.einsum("iab,ija->ijb", C, d)   # symmetric figures
    other = torch.einsum("jab,ija->ijb", C[sources], d)
    k5 = (g3 * k)[..., None]
    figures = (k5 * R2[:, None, None] * field(own) + k5 * R2[None, sources, None] * field(other)).sum(1)
    return newton, phi, pn, figures


def _rk4(r, v, dt, pull):
    kr1, kv1 = v, pull(r, v)
    kr2, kv2 = v + dt / 2 * kv1, pull(r + dt / 2 * kr1, v + dt / 2 * kv1)
    kr3, kv3 = v + dt / 2 * kv2, pull(r + dt / 2 * kr2, v + dt / 2 * kv2)
    kr4, kv4 = v + dt * kv3, pull(r + dt * kr3, v + dt * kv3)
    return r + dt / 6 * (kr1 + 2 * kr2 + 2 * kr3 + kr4), v + dt / 6 * (kv1 + 2 * kv2 + 2 * kv3 + kv4)


def exact(case, seed):
    """Positions and velocities after the pass, and the Newtonian and 1PN parts
    of a force evaluation.  The figures (C_potential) are those that the bodies
    were loaded with; what is left out -- the figures' change within the pass,
    J3 and above, the ring, Lense-Thirring and radiation terms -- moves r and v
    by about 1e-8 of their norm or less.  Other outputs have no value here."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind, steps, dt = case["kind"], case.get("steps", 0), case.get("dt", DAY)
    if kind == "integrate" and (case["systems"] * case["bodies"] ** 2 * case["steps"] > 1e8
                                or case["systems"] * case["steps"] > 1000):
        return None                          # over 20 seconds
    masses, sys_n = _bodies(_FIELD9 if kind == "particles" else case, seed)[:2]
    col = _columns(masses)
    arrays = [col["r"][:, ::2], col["v"][:, ::2], masses["GM"], col["C_potential"].reshape(-1, 3, 3), masses["R2"],
              masses["sR2"]]
    ends, sources = np.cumsum(sys_n), slice(None)
    if kind == "particles":                  # massless points after the field's bodies
        points = gen.make_particles(case["particles"], seed=seed, field9=gen.make_field9())
        zeros = [np.zeros((case["particles"], *a.shape[1:])) for a in arrays[2:]]
        arrays = [np.concatenate(pair) for pair in zip(arrays, [*points, *zeros])]
        ends, sources, sys_n = [len(arrays[0])], slice(0, 9), [len(arrays[0])]
    out_r, out_v = [], []
    for end, n in zip(ends, sys_n):
        r, v, *rest = (torch.tensor(np.ascontiguousarray(a[end - n:end]), device=dev) for a in arrays)

        def pull(x, u):
            newton, _, pn, figures = _pull(x, u, *rest, sources)
            return newton + pn + figures

        parts = 8 if kind == "particles" or dt >= DAY else 3
        for _ in range(steps * parts):
            r, v = _rk4(r, v, dt / parts, pull)
        out_r.append(r)
        out_v.append(v)
    r, v = (np.stack([a, np.zeros_like(a)], -1).reshape(-1, 6) for a in (torch.cat(out_r).cpu().numpy(), torch.cat(out_v).cpu().numpy()))
    if kind == "particles":
        return {"r": r[9:], "v": v[9:], "extrema": None}
    out = dict.fromkeys([name for name, _, _ in _GROUPS])
    if kind == "accel":
        newton, phi, pn, _ = (a.cpu().numpy() for a in _pull(out_r[0], out_v[0], *rest, sources))
        return {**out, "phi": phi[:, None], "naccel": newton, "gaccel": pn, "t_eph": None}
    return {**out, "r": r, "v": v, "t_eph": np.array([[dt * steps, 0.0]] * len(sys_n))}
