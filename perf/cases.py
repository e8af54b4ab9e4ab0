"""The engine's workloads as timed cases, each one pass through the public
Python binding (graphical-edmd_amd/edmd_hip.py over include/edmd.h).

What the cases stand for:
  run      a stretch of event-driven dynamics between two outputs: the loop
           advances every system by so many collisions, then the whole state
           is read (positions, velocities, local times, counters, cells).
           One system is what the reference's program simulates, from a few
           hundred disks to 2^20; a batch is an ensemble of replicas; options
           are the reference's: radii that differ, the velocity-rescaling
           thermostat, walls with a field.
  grow     the reference's default start, whole: a system built from random
           centres, its disks grown to their radii, the state read.
  sweep    the prediction of every disk's next collision and crossing, as at
           a start or after an edit of the state, and the predictions read.
  deriv    derivatives of a run: taping, the forward stretch, the adjoint
           and (whole tapes) the tangent pass; with checkpoints the segments
           are recomputed.
  pcf      g(r) of a configuration held by the caller.

Sizes, packing fractions and options are those of bench.py, the tests and
the reference's own command line (2000 disks of radius 1 at phi = 0.7).
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _binding():
    if "edmd_hip" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "edmd_hip", os.path.join(ROOT, "graphical-edmd_amd", "edmd_hip.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["edmd_hip"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["edmd_hip"]


def listed():
    return [
        # the smallest calls: a few hundred disks advanced by one collision
        # per disk between outputs
        _run("single_400", replicas=1, n=400, n_hi=400, phi=0.60, collisions=200),
        # the reference's own headline system: 2000 disks of radius 1
        _run("single_2000", replicas=1, n=2000, n_hi=2000, phi=0.70, rad=1.0, collisions=4000),
        # one large system (bench.py's plain leg)
        _run("single_1048576", replicas=1, n=1 << 20, n_hi=1 << 20, phi=0.80, collisions=30000),
        # the ensemble of bench.py's headline: replicas of uneven size
        _run("ensemble_4096", replicas=4096, n=256, n_hi=2048, phi=0.50, phi_hi=0.75,
             collisions=20000),
        # dense polydisperse replicas under the thermostat (bench.py's dense
        # leg; the rescale comes every 0.1 time units)
        _run("dense_64x65536", replicas=64, n=65536, n_hi=65536, phi=0.70, poly=0.04,
             thermostat=True, collisions=40000),
        # sedimentation in a channel: walls and the field
        _run("channel_256x1000", replicas=256, n=1000, n_hi=1000, phi=0.40, channel=True,
             collisions=2000),
        # growth starts of polydisperse replicas, through GROWSTOP
        {"name": "grow_64x1000", "kind": "grow", "replicas": 64, "n": 1000, "phi": 0.60,
         "poly": 0.1, "vr": 0.2},
        # every disk of the large system predicted again
        {"name": "sweep_1048576", "kind": "sweep", "n": 1 << 20, "phi": 0.70, "poly": 0.0},
        # derivatives of an ensemble (bench.py's adjoint leg), whole tape
        {"name": "deriv_tape_512x400", "kind": "deriv", "replicas": 512, "n": 400, "phi": 0.60,
         "every": 0, "collisions": 4000},
        # the same with checkpoints every 256 events
        {"name": "deriv_ckpt_512x400", "kind": "deriv", "replicas": 512, "n": 400, "phi": 0.60,
         "every": 256, "collisions": 2000},
        # g(r) of a large configuration over a few diameters, and of a small
        # one over half its box
        {"name": "pcf_60000", "kind": "pcf", "n": 60000, "phi": 0.70, "dr": 0.02, "max_r": 10.0},
        {"name": "pcf_2000", "kind": "pcf", "n": 2000, "phi": 0.70, "dr": 0.01, "max_r": 20.0},
    ]


def _run(name, replicas, n, n_hi, phi, collisions, phi_hi=None, rad=0.5, poly=0.0,
         thermostat=False, channel=False):
    c = {"kind": "run", "replicas": replicas, "n": n, "n_hi": n_hi, "phi": phi,
         "phi_hi": phi if phi_hi is None else phi_hi, "rad": rad, "poly": poly,
         "thermostat": thermostat, "channel": channel, "collisions": collisions}
    if name:
        c["name"] = name
    return c


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run"] * 6 + ["grow", "sweep", "deriv", "deriv", "pcf", "pcf"])
    if kind == "run":
        replicas = _log(rng, 1, 4096) if rng.random() < 0.6 else 1
        n = _log(rng, 200, min(1 << 20, (1 << 22) // replicas))
        option = rng.choice(["", "", "", "poly", "thermostat", "channel"])
        if replicas > 1024 and option:
            option = "poly"
        # at most about a quarter of a second: a wavefront advances one system
        # by some 10^5 collisions a second, the whole chip 3 * 10^8
        most = int(0.25 * min(1e5, 2.5e8 / replicas))
        if option == "channel":
            most //= 4
        coll = min(most, max(100, int(n * rng.uniform(0.5, 5.0))))
        if option == "channel":
            return _run(None, replicas, n, n, round(rng.uniform(0.2, 0.45), 3), coll,
                        channel=True)
        poly = 0.04 if option in ("poly", "thermostat") else 0.0
        # cells have sides of 2 and more: radii above 1 need larger ones
        rad = 0.5 if poly else rng.choice([0.5, 0.5, 1.0])
        return _run(None, replicas, n, max(n, int(n * rng.choice([1.0, 1.0, 2.0]))),
                    round(rng.uniform(0.3, 0.7), 3), coll, rad=rad, poly=poly,
                    thermostat=option == "thermostat")
    if kind == "grow":
        n = _log(rng, 200, 3000)
        return {"kind": "grow", "replicas": _log(rng, 1, 128), "n": n,
                "phi": round(rng.uniform(0.4, 0.62), 3), "poly": rng.choice([0.0, 0.1]),
                "vr": round(rng.uniform(0.2, 0.4), 3)}
    if kind == "sweep":
        return {"kind": "sweep", "n": _log(rng, 1000, 1 << 20),
                "phi": round(rng.uniform(0.3, 0.72), 3), "poly": rng.choice([0.0, 0.04])}
    if kind == "deriv":
        return {"kind": "deriv", "replicas": _log(rng, 1, 512), "n": _log(rng, 200, 2000),
                "phi": round(rng.uniform(0.4, 0.7), 3), "every": rng.choice([0, 0, 128, 256]),
                "collisions": _log(rng, 300, 2000)}
    n = _log(rng, 500, 60000)
    half = 0.5 * math.sqrt(n * math.pi * 0.25 / 0.7)
    return {"kind": "pcf", "n": n, "phi": round(rng.uniform(0.4, 0.72), 3),
            "dr": rng.choice([0.01, 0.02, 0.05]),
            "max_r": round(min(half, rng.uniform(3.0, 25.0)), 2)}


# ------------------------------------------------------------------ inputs

def _disks(n, phi, rng, rad=0.5, poly=0.0, jitter=0.0, channel=False):
    """n disks of radius rad (times 1 + poly * a truncated normal) at packing
    fraction phi on a triangular stacking fitted to a square box, velocities
    normal with zero total momentum and E/N = 1; jitter moves each disk by
    that fraction of the free gap; channel keeps them off the walls."""
    L = math.sqrt(math.pi * n * rad * rad / phi)
    best = (0.0, 2)
    guess = math.sqrt(2.0 * n / math.sqrt(3.0))
    for ny in range(max(2, int(0.7 * guess) // 2 * 2), int(1.3 * guess) + 4, 2):
        nx = -(-n // ny)
        dx, dy = L / nx, L / ny
        best = max(best, (min(dx, math.hypot(dx / 2, dy)), ny))
    gap, ny = best
    nx = -(-n // ny)
    k = np.arange(n)
    i, j = k % nx, k // nx
    x = (i + 0.25 + 0.5 * (j % 2)) * (L / nx)
    y = (j + 0.5) * (L / ny)
    r = np.full(n, rad)
    if poly:
        r = rad * (1 + poly * np.clip(rng.standard_normal(n), -2.0, 2.0))
    if channel:
        f = (L - 2.04 * rad) / L
        x, y = 1.02 * rad + x * f, 1.02 * rad + y * f
        gap *= f
    free = gap - 2 * r.max()
    if not free > 0:
        raise ValueError("phi = %g is too dense for %d disks on a fitted lattice" % (phi, n))
    if jitter:
        a, d = rng.uniform(0, 2 * np.pi, n), rng.uniform(0, 0.5 * jitter * free, n)
        x, y = (x + d * np.cos(a)) % L, (y + d * np.sin(a)) % L
    v = rng.standard_normal((2, n))
    v -= v.mean(axis=1, keepdims=True)
    v /= math.sqrt(0.5 * float((v * v).sum()) / n)
    return {"x": x, "y": y, "vx": v[0].copy(), "vy": v[1].copy(), "rad": r, "m": np.ones(n),
            "Lx": L, "Ly": L}


def _random_disks(n, phi, rng, poly):
    """Random centres and target radii of a growth start."""
    r = 0.5 * (1 + poly * np.clip(rng.standard_normal(n), -3.0, 3.0))
    L = math.sqrt(math.pi * float((r * r).sum()) / phi)
    v = rng.standard_normal((2, n)) * math.sqrt(0.05)
    return {"x": rng.uniform(0, L, n), "y": rng.uniform(0, L, n), "vx": v[0].copy(),
            "vy": v[1].copy(), "rad": r, "m": np.ones(n), "Lx": L, "Ly": L}


def _run_inputs(case, seed):
    """Replica sizes spread evenly over n .. n_hi (the golden-ratio sequence:
    the case's own, whatever the seed); densities and velocities by seed."""
    rng = np.random.default_rng(seed)
    R = case["replicas"]
    spread = np.arange(R) * 0.6180339887498949 % 1.0
    ns = case["n"] + (spread * (case["n_hi"] + 1 - case["n"])).astype(int)
    phis = rng.uniform(case["phi"], case["phi_hi"], size=R)
    return [_disks(int(n), float(p), rng, case["rad"], case["poly"], channel=case["channel"])
            for n, p in zip(ns, phis)]


def _melt(case):
    """Collisions per replica that take the lattice apart before the passes."""
    return min(10 * case["n"], 20000)


def _options(case):
    if case.get("thermostat"):
        return dict(noise=2, dtnoise=0.1, temperature=1.0)
    if case.get("channel"):
        return dict(wall_y=1, wall_x=1, res_tan=1.0, add_field=1, field=-0.02)
    return {}


def prepare(case, seed):
    E = _binding()
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "run":
        states = _run_inputs(case, seed)
        opt = _options(case)
        one = case["replicas"] == 1
        h = E.System(states[0], **opt) if one else E.Batch(states, **opt)
        done = _melt(case)
        h.run(max_collisions=done)
        return {"kind": kind, "h": h, "one": one, "done": done, "step": case["collisions"]}
    if kind == "grow":
        states = [_random_disks(case["n"], case["phi"], rng, case["poly"])
                  for _ in range(case["replicas"])]
        return {"kind": kind, "E": E, "states": states, "vr": case["vr"]}
    if kind == "sweep":
        st = _disks(case["n"], case["phi"], rng, poly=case["poly"], jitter=0.9)
        return {"kind": kind, "h": E.System(st)}
    if kind == "deriv":
        states = [_disks(case["n"], case["phi"], rng) for _ in range(case["replicas"])]
        b = E.Batch(states)
        done = 2 * case["n"]
        b.run(max_collisions=done)
        tin = [rng.standard_normal((case["n"], 4)) for _ in states]
        return {"kind": kind, "b": b, "done": done, "step": case["collisions"],
                "every": case["every"], "tin": [t / np.linalg.norm(t) for t in tin]}
    st = _disks(case["n"], case["phi"], rng, jitter=0.9)
    return {"kind": kind, "E": E, "st": st, "dr": case["dr"], "max_r": case["max_r"]}


def _whole(batch):
    parts = [batch.state(k) for k in range(len(batch))]
    return {f: np.concatenate([p[f] for p in parts]) for f in parts[0]}


def run(state):
    kind = state["kind"]
    if kind == "run":
        h = state["h"]
        state["done"] += state["step"]
        h.run(max_collisions=state["done"])
        return h.state() if state["one"] else _whole(h)
    if kind == "grow":
        b = state["E"].Batch(state["states"], vr=state["vr"])
        b.run(tmax=1.0 / state["vr"])
        out = _whole(b)
        b.close()
        return out
    if kind == "sweep":
        h = state["h"]
        h.sweep_predict()
        return h.events()
    if kind == "deriv":
        b, every = state["b"], state["every"]
        b.deriv_begin(checkpoint_every=every, tape_capacity=0 if every else state["step"])
        state["done"] += state["step"]
        b.deriv_run(max_collisions=state["done"])
        out = {"gradient": np.concatenate(b.adjoint(lw=1.0))}
        if not every:
            tan, dw, dtl = b.tangent(state["tin"])
            out.update(tangent=np.concatenate(tan), dw=dw, dt_last=dtl)
        return out
    st = state["st"]
    r, g = state["E"].pcf(st["x"], st["y"], st["Lx"], st["Ly"], state["dr"], state["max_r"])
    return {"r": r, "g": g}


# -------------------------------------------------------------------- work

def work(case):
    """Bytes: the state a pass starts from read once and its outputs written
    once (a disk: position, velocity, local time, radius, mass, counter and
    cell, 64 B).  Operations: per collision the collision time (24) of each
    neighbour of both disks (nine cells of side 2), per pair of g(r) its
    distance and bin (10)."""
    kind, n = case["kind"], case["n"]
    rad = case.get("rad", 0.5)
    near = 9 * 4.0 * case["phi"] / (math.pi * rad * rad)
    if kind == "pcf":
        pairs = 0.5 * n * case["phi"] * (2 * case["max_r"]) ** 2
        return {"bytes": 16.0 * n + 16.0 * case["max_r"] / case["dr"], "flops": 10 * pairs}
    if kind == "sweep":
        return {"bytes": 80.0 * n, "flops": 24 * near * n}
    R = case["replicas"]
    if kind == "grow":
        # about 16 collisions a disk until the radii are reached
        return {"bytes": R * n * 128.0, "flops": R * n * 16.0 * 48 * near}
    disks = R * 0.5 * (n + case.get("n_hi", n))
    flops = R * case["collisions"] * 48.0 * near
    if kind == "deriv":
        again = 2 if case["every"] else 1
        return {"bytes": disks * 128.0 + again * 2.0 * 64 * R * case["collisions"],
                "flops": again * flops}
    return {"bytes": disks * 128.0, "flops": flops}


# ------------------------------------------------------------------- exact

def exact(case, seed):
    """g(r), the predictions and the velocities of one small system after its
    collisions, in plain 64-bit numpy / torch; None where only the engine's
    event order defines the result or a direct evaluation takes too long."""
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "pcf":
        st = _disks(case["n"], case["phi"], rng, jitter=0.9)
        return _exact_pcf(st, case["dr"], case["max_r"], dev)
    if kind == "sweep":
        st = _disks(case["n"], case["phi"], rng, poly=case["poly"], jitter=0.9)
        tc, tx = _exact_sweep(st, dev)
        return {"t_coll": tc, "t_cross": tx, "partner": None, "dir": None, "coll_actual": None}
    if kind == "run" and case["replicas"] == 1 and not (case["channel"] or case["thermostat"]):
        total = _melt(case) + case["collisions"]
        if case["n"] > 3000 or total > 30000:
            return None
        st = _run_inputs(case, seed)[0]
        vx, vy = _exact_velocities(st, total)
        return {"x": None, "y": None, "vx": vx, "vy": vy, "t": None, "coll": None, "cx": None,
                "cy": None}
    return None


def _exact_pcf(st, dr, max_r, dev):
    n, L = len(st["x"]), st["Lx"]
    nb = int(max_r / dr)
    x, y = (torch.tensor(st[k], dtype=torch.float64, device=dev) for k in ("x", "y"))
    hist = torch.zeros(nb, dtype=torch.float64, device=dev)
    step = max(1, (1 << 25) // n)
    for a in range(0, n, step):
        dx = (x[a:a + step, None] - x[None, :]).abs()
        dy = (y[a:a + step, None] - y[None, :]).abs()
        dx = torch.minimum(dx, L - dx)
        dy = torch.minimum(dy, L - dy)
        rr = torch.sqrt(dx * dx + dy * dy)
        rr[torch.arange(len(rr)), torch.arange(a, a + len(rr))] = 2 * max_r
        b = (rr[rr < dr * nb] / dr).long()
        hist += torch.bincount(b[b < nb], minlength=nb)[:nb].double()
    r = (np.arange(nb) + 0.5) * dr
    g = hist.cpu().numpy() / (2 * np.pi * r * dr * (n / (L * L)) * n)
    return {"r": r, "g": g}


def _exact_sweep(st, dev):
    """Per disk, the earliest contact with a disk of its 3 x 3 cells (cells
    of side L / floor(L / 2)) and the time at which it leaves its cell."""
    n, L = len(st["x"]), st["Lx"]
    nc = int(L / 2)
    cs = L / nc
    x, y, vx, vy, r = (torch.tensor(st[k], dtype=torch.float64, device=dev)
                       for k in ("x", "y", "vx", "vy", "rad"))
    cx = (x * (1 / cs)).long().clamp(max=nc - 1)
    cy = (y * (1 / cs)).long().clamp(max=nc - 1)
    cell = cy * nc + cx
    order = torch.argsort(cell, stable=True)
    count = torch.bincount(cell, minlength=nc * nc)
    first = torch.cumsum(count, 0) - count
    best = torch.full((n,), 1e26, dtype=torch.float64, device=dev)
    me = torch.arange(n, device=dev)
    for sy in (-1, 0, 1):
        for sx in (-1, 0, 1):
            c = ((cy + sy) % nc) * nc + (cx + sx) % nc
            for k in range(int(count.max())):
                ok = k < count[c]
                q = order[torch.where(ok, first[c] + k, torch.zeros_like(c))]
                ok &= q != me
                dx, dy = x[q] - x, y[q] - y
                dx = dx - L * torch.round(dx / L)
                dy = dy - L * torch.round(dy / L)
                dvx, dvy = vx[q] - vx, vy[q] - vy
                b = dx * dvx + dy * dvy
                v2 = dvx * dvx + dvy * dvy
                det = b * b - v2 * (dx * dx + dy * dy - 4 * r * r[q])
                ok &= (b <= 0) & (det >= 0)
                t = (-b - torch.sqrt(det.clamp(min=0))) / v2
                best = torch.where(ok & (t < best), t, best)
    ex = torch.where(vx < 0, cx.double() * cs, (cx + 1).double() * cs) - x
    ey = torch.where(vy < 0, cy.double() * cs, (cy + 1).double() * cs) - y
    return best.cpu().numpy(), torch.minimum(ex / vx, ey / vy).cpu().numpy()


def _exact_velocities(st, collisions):
    """Velocities after so many collisions of disks of equal mass: every
    disk's next contact kept, the earliest taken, both disks' contacts (and
    of those that were to meet them) found again over all others."""
    n, L = len(st["x"]), st["Lx"]
    x, y, vx, vy, r = (st[k].copy() for k in ("x", "y", "vx", "vy", "rad"))
    at = np.zeros(n)
    when = np.full(n, np.inf)
    whom = np.zeros(n, dtype=np.int64)

    def look(i, t):
        h = t - at
        dx = (x + h * vx) - (x[i] + h[i] * vx[i])
        dy = (y + h * vy) - (y[i] + h[i] * vy[i])
        dx -= L * np.rint(dx / L)
        dy -= L * np.rint(dy / L)
        dvx, dvy = vx - vx[i], vy - vy[i]
        b = dx * dvx + dy * dvy
        v2 = dvx * dvx + dvy * dvy
        det = b * b - v2 * (dx * dx + dy * dy - 4 * r[i] * r)
        ok = (b < 0) & (det >= 0)
        ok[i] = False
        tt = np.full(n, np.inf)
        tt[ok] = (-b[ok] - np.sqrt(det[ok])) / v2[ok]
        whom[i] = int(np.argmin(tt))
        when[i] = t + tt[whom[i]]
        closer = t + tt < when
        closer[i] = False
        whom[closer] = i
        when[closer] = t + tt[closer]

    for i in range(n):
        look(i, 0.0)
    for _ in range(collisions):
        i = int(np.argmin(when))
        j, t = int(whom[i]), when[i]
        for k in (i, j):
            h = t - at[k]
            x[k] += h * vx[k]
            y[k] += h * vy[k]
            at[k] = t
        dx, dy = x[j] - x[i], y[j] - y[i]
        dx -= L * np.rint(dx / L)
        dy -= L * np.rint(dy / L)
        f = (dx * (vx[j] - vx[i]) + dy * (vy[j] - vy[i])) / (4 * r[i] * r[j])
        vx[i] += f * dx
        vy[i] += f * dy
        vx[j] -= f * dx
        vy[j] -= f * dy
        when[i] = when[j] = np.inf
        lost = np.nonzero((whom == i) | (whom == j))[0]
        for k in lost:
            when[k] = np.inf
        for k in set([i, j, *lost.tolist()]):
            look(int(k), t)
    return vx, vy
