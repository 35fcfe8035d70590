"""Performance cases of the framework: what its users have it do, through its public entry points.

A case is a dict of plain values.  Its ``kind`` names the entry point:

* ``points``   ``Magnet.magnetic_field_at`` / ``magnetic_field_at_points`` on host points (FP64), the
               call of scripts and of field analysis;
* ``field``    ``DeviceModel.field_tensors`` on device points: field maps and field lines;
* ``track``    ``DeviceModel.track_tensors``: RK4 tracking of a resident beam (the headline workload);
* ``replay``   the same pass captured once as a ``TrackGraph`` and replayed;
* ``facade``   ``GPU_ACCELERATOR.track_multi_particle_beamline_for_magnet_with_multi_qs`` on host
               particles, the drop-in call of the reference's scripts;
* ``search``   ``GantryPopulationProblem.run``, one generation of a design search: building the
               designs on the host, tracking them and reducing to the objectives;
* ``adjoint``  ``AdjointTracker.forward`` and ``.backward``: the gradients of a beam size.

``magnet`` names a workload of ``cctpy_amd/workloads.py`` (``cct`` a single CCT, ``section`` the AG-CCT
section, ``population`` many CCT designs, ``gantry`` the whole HUST gantry) and ``parts`` its segments
per winding.  The seed moves the magnet currents by up to 1 % and draws the beam, so that no two seeds
share segments or particles.  Beams have the workloads' widths (1.75 mm, 2 mrad) and a momentum spread
of 2 %, which keeps them inside the bore.  A pass is a stretch of the whole track (the cost of a step does
not depend on how many follow), short enough that a plain FP64 sum of the same steps takes seconds.
"""
import math

import numpy
import torch

from cctpy_amd import adjoint, engine, optim, workloads
from cctpy_amd.cctpy import GPU_ACCELERATOR, P3
from cctpy_amd.magnets import device_parts

MM = 0.001
PAIR_FLOPS = 27  # one field point x segment term: difference, |r|^2, 1/|r|^3, cross product, accumulation
MOST_PAIRS = 1.5e11  # of a drawn case; the largest listed one has 1.9e11

# The tuned design vector around which a design search samples its generations.
TUNED = [3.5302, 5.5552, -42.9943, -19.1617, 94.9830, 75.8091, 80.5371, 87.3605, 81.8937, 95.5016,
         -9613.5385, 10969.1606, 24.0, 24.0, 2.9978, -92.7398, 85.1549, 88.9347, 88.3576, 78.3727, 86.5075,
         95.0290, 9147.5885, -7582.9665, 22.0, 39.0, 32.0]


def listed():
    return [
        # latency of one field value in a script's loop
        {"name": "point_cct", "kind": "points", "magnet": "cct", "parts": 360, "n": 1},
        # the field along the ideal arc of a single CCT, FP32 path
        {"name": "arc_field_f32", "kind": "field", "magnet": "cct", "parts": 360, "n": 1000, "precision": 33},
        # a field map of the AG-CCT section (off-axis points), FP64
        {"name": "map_section_f64", "kind": "field", "magnet": "section", "parts": 720, "n": 5003, "precision": 64},
        # a small beam through a single CCT, where launches count: the whole arc, replayed as a graph
        {"name": "cct_replay_f32", "kind": "replay", "magnet": "cct", "parts": 360, "designs": 1, "particles": 64,
         "steps": 498, "step_mm": 1.0, "s0": 0.1, "precision": 33},
        # the reference's script call: a few host particles through two beamlines, 10 mm steps, FP64
        {"name": "facade_f64", "kind": "facade", "magnet": "gantry", "parts": 120, "designs": 2, "particles": 24,
         "steps": 150, "step_mm": 10.0, "s0": 0.5, "precision": 64},
        # the headline beam through the AG-CCT section on the FP64 path, 10 mm steps
        {"name": "section_track_f64", "kind": "track", "magnet": "section", "parts": 720, "designs": 1,
         "particles": 512, "steps": 64, "step_mm": 10.0, "s0": 0.6, "precision": 64},
        # the headline beam and step on the FP32 path, a stretch inside the windings
        {"name": "section_track_f32", "kind": "track", "magnet": "section", "parts": 720, "designs": 1,
         "particles": 512, "steps": 150, "step_mm": 1.0, "s0": 0.9, "precision": 33},
        # the 64-design population in one launch per stage, FP32 path
        {"name": "population_track_f32", "kind": "track", "magnet": "population", "parts": 0, "designs": 64,
         "particles": 32, "steps": 80, "step_mm": 1.0, "s0": 0.2, "precision": 33},
        # the largest beam and segment set: the whole gantry, FP32 path, steps of 0.5 mm
        {"name": "gantry_track_f32", "kind": "track", "magnet": "gantry", "parts": 720, "designs": 1,
         "particles": 4096, "steps": 12, "step_mm": 0.5, "s0": 1.0, "precision": 33},
        # one generation of the design search: 8 gantries x 80 particles, FP64, 50 mm steps
        {"name": "search_f64", "kind": "search", "designs": 8, "per_plane": 10},
        # gradients of the section's beam size, tape of every step kept
        {"name": "adjoint_section", "kind": "adjoint", "magnet": "section", "parts": 720, "designs": 1,
         "particles": 256, "steps": 40, "step_mm": 1.0, "s0": 0.9, "ckpt": 0},
        # gradients of a population, recomputed from checkpoints
        {"name": "adjoint_population", "kind": "adjoint", "magnet": "population", "parts": 0, "designs": 16,
         "particles": 32, "steps": 30, "step_mm": 1.0, "s0": 0.2, "ckpt": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "field", "field", "replay", "facade", "track", "track", "track", "track", "track",
                       "search", "adjoint", "adjoint"])
    if kind == "points":
        return {"kind": kind, "magnet": rng.choice(["cct", "section", "gantry"]), "parts": rng.choice([60, 120, 360]),
                "n": _log(rng, 1, 2000)}
    if kind == "field":
        return {"kind": kind, "magnet": rng.choice(["cct", "section"]), "parts": rng.choice([360, 720]),
                "n": _log(rng, 16, 20000), "precision": rng.choice([32, 33, 64])}
    if kind == "search":
        return {"kind": kind, "designs": rng.randint(1, 8), "per_plane": rng.randint(3, 10)}
    magnet = {"replay": ["cct"], "facade": ["section", "gantry"], "adjoint": ["section", "population"],
              "track": ["cct", "section", "section", "population", "gantry"]}[kind]
    magnet = rng.choice(magnet)
    c = {"kind": kind, "magnet": magnet,
         "parts": rng.choice([360, 720]) if magnet != "population" else 0,
         "designs": rng.randint(2, 48) if magnet == "population" else 1,
         "particles": _log(rng, 16, 2048) if magnet != "population" else _log(rng, 8, 64),
         "steps": rng.randint(20, 200), "step_mm": rng.choice([0.5, 1.0]),
         "s0": round(rng.uniform({"cct": 0.1, "section": 0.5, "population": 0.15, "gantry": 0.5}[magnet],
                                 {"cct": 0.3, "section": 1.2, "population": 0.3, "gantry": 2.0}[magnet]), 3)}
    if kind == "facade":
        c.update(parts=rng.choice([60, 120, 360]), designs=rng.randint(1, 4), particles=_log(rng, 1, 64),
                 step_mm=rng.choice([5.0, 10.0]), precision=64)
    elif kind == "adjoint":
        c.update(particles=min(c["particles"], 300), steps=rng.randint(8, 40), designs=min(c["designs"], 16),
                 ckpt=rng.choice([0, 8, 20]))
    else:
        c["precision"] = rng.choice([33, 64])
        if c["precision"] == 64:
            c["step_mm"] = rng.choice([1.0, 5.0, 10.0])
            c["steps"] = min(c["steps"], int(600 / c["step_mm"]))
        if kind == "replay":
            c["particles"] = min(c["particles"], 300)
    most = MOST_PAIRS / (4 if kind == "adjoint" else 1)
    each = 4 * c["designs"] * c["particles"] * _segments(c)
    c["steps"] = max(4, min(c["steps"], int(most / each)))
    if each * c["steps"] > most:
        c["particles"] = max(16, int(c["particles"] * most / (each * c["steps"])))
    return c


def _segments(c):
    """Segments of one design of a case (the population's mean)."""
    return {"cct": 64 * c.get("parts", 0), "section": 512 * c.get("parts", 0),
            "gantry": 1332 * c.get("parts", 0), "population": 204800}[c["magnet"]]


# ---------------------------------------------------------------- inputs
def _workload(c, seed):
    """The case's workload with this seed's currents and beam."""
    rng = numpy.random.default_rng(seed)
    if c["magnet"] == "population":
        wl = workloads.population(n_designs=c["designs"], n_particles=1)
    elif c["magnet"] == "cct":
        wl = workloads.single_cct(n_particles=1)
    elif c["magnet"] == "section":
        wl = workloads.agcct_section(n_particles=1, disperse_number_per_winding=c["parts"])
    else:
        wl = workloads.hust_total(n_particles=1)
    designs = []
    for k in range(c.get("designs", 1)):
        ops = []
        for name, kw in wl.designs[k if c["magnet"] == "population" else 0]:
            kw = dict(kw)
            f = 1 + 0.01 * rng.uniform(-1, 1)
            if "current" in kw:
                kw["current"] *= f
            if "currents" in kw:
                kw["currents"] = [f * i for i in kw["currents"]]
            if name == "append_single_cct":
                kw["disperse_number_per_winding"] = c["parts"]
            if name == "hust_total":
                kw.update(part_per_winding=c["parts"], dicct345_current=9664 * f, agcct345_current=-6000 * f,
                          dicct12_current=-9780.7 * f, agcct12_current=9736.8 * f)
            ops.append((name, kw))
        designs.append(ops)
    return [workloads.build_beamline(ops) for ops in designs], rng


def _beam(c, bls, rng):
    """The running particles of each design."""
    if c["kind"] == "facade":  # one beam through every beamline
        coords = workloads.gaussian_beam(rng, c["particles"], 0.02)
        return [workloads.beam_particles(workloads.Beam(coords, c["s0"], 250.0), bls[0])]
    return [workloads.beam_particles(workloads.Beam(workloads.gaussian_beam(rng, c["particles"], 0.02), c["s0"], 250.0),
                                     bl) for bl in bls]


def _arrays(c, beams):
    """(state (P, 6), kq, dt, nsteps) of particles that all take the case's steps."""
    ps = [p for b in beams for p in b]
    state = numpy.array([p.position.to_list() + p.velocity.to_list() for p in ps])
    sd = [engine.rk4_steps(c["steps"] * c["step_mm"] * MM, c["step_mm"] * MM, p.speed) for p in ps]
    return (state, numpy.array([p.e / p.relativistic_mass for p in ps]), numpy.array([d for _, d in sd]),
            numpy.array([n for n, _ in sd], numpy.int64))


def _points(c, bl, rng):
    """Points along the orbit, up to 30 mm off it."""
    s = numpy.linspace(0.0, bl.get_length(), c["n"] + 2)[1:-1]
    off = rng.uniform(-30 * MM, 30 * MM, (c["n"], 3))
    q = [bl.trajectory.point_at(float(x)) for x in s]
    return numpy.array([[p.x, p.y, 0.0] for p in q]) + off


def _generation(c, seed):
    """A design search's generation: the tuned vector with its real variables moved by about 0.5 %."""
    base = numpy.array(TUNED)
    v = base * (1 + 0.005 * numpy.random.default_rng(seed).standard_normal((c["designs"], base.size)))
    whole = numpy.array(optim.VAR_TYPES) == 1
    v[:, whole] = base[whole]
    return v


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = c = case
    if c["kind"] == "search":
        s.problem = optim.GantryPopulationProblem(particle_number_per_plane_per_dp=c["per_plane"])
        s.vars = _generation(c, seed)
        return s
    bls, rng = _workload(c, seed)
    if c["kind"] == "points":
        s.magnet = bls[0]
        s.points = [P3(*row) for row in _points(c, bls[0], rng)]
        return s
    if c["kind"] == "facade":
        s.beamlines, s.particles = bls, _beam(c, bls, rng)[0]
        s.accelerator = GPU_ACCELERATOR(GPU_ACCELERATOR.FLOAT64)
        return s
    if c["kind"] == "adjoint":
        s.state, s.kq, s.dt, s.nsteps = _arrays(c, _beam(c, bls, rng))
        s.npt = [c["particles"]] * len(bls)
        s.tracker = adjoint.AdjointTracker(bls, ckpt_every=c["ckpt"],
                                           ppl=engine.block_shape_for(s.npt, 33))
        return s
    s.model = engine.DeviceModel([device_parts(bl).spec() for bl in bls], fp32=c["precision"] != 64)
    dev = engine.device()

    def up(a):
        return torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)

    if c["kind"] == "field":
        s.points = up(_points(c, bls[0], rng).T)
        s.out = torch.empty_like(s.points)
        s.plan = s.model.plan([c["n"]], engine.block_shape_for([c["n"]], c["precision"]))
        _, s.partial = s.model.workspace(s.plan)
        return s
    state, kq, dt, ns = _arrays(c, _beam(c, bls, rng))
    s.initial, s.kq, s.dt, s.nsteps, s.steps = up(state.T), up(kq), up(dt), up(ns), int(ns.max())
    s.state = s.initial.clone()
    npt = [c["particles"]] * len(bls)
    s.plan = s.model.plan(npt, engine.block_shape_for(npt, c["precision"]))
    s.scratch, s.partial = s.model.workspace(s.plan)
    if c["kind"] == "replay":
        s.graph = engine.TrackGraph(s.model, s.plan, c["precision"], s.state, s.kq, s.dt, s.nsteps, s.steps,
                                    s.scratch, s.partial)
    return s


# ------------------------------------------------------------------ a pass
def _beam_size_seed(final):
    """dJ/d(final states) of J = sqrt(mean |p - mean p|^2), the beam size."""
    d = final[:, :3] - final[:, :3].mean(0)
    seed = 0.0 * final
    seed[:, :3] = d / (len(final) * ((d * d).sum(1).mean()) ** 0.5)
    return seed


def run(s):
    c = s.case
    if c["kind"] == "points":
        if c["n"] == 1:
            return numpy.array(s.magnet.magnetic_field_at(s.points[0]).to_list())
        return numpy.array([b.to_list() for b in s.magnet.magnetic_field_at_points(s.points)])
    if c["kind"] == "field":
        s.model.field_tensors(s.plan, c["precision"], s.points, s.partial, s.out)
        return s.out
    if c["kind"] == "track":
        s.state.copy_(s.initial)
        s.model.track_tensors(s.plan, c["precision"], s.state, s.kq, s.dt, s.nsteps, s.steps, s.scratch, s.partial)
        return s.state
    if c["kind"] == "replay":
        s.state.copy_(s.initial)
        s.graph.replay()
        return s.state
    if c["kind"] == "facade":
        ends = s.accelerator.track_multi_particle_beamline_for_magnet_with_multi_qs(
            s.beamlines, s.particles, c["steps"] * c["step_mm"] * MM, c["step_mm"] * MM)
        return numpy.array([[p.position.to_list() + p.velocity.to_list() for p in row] for row in ends])
    if c["kind"] == "search":
        return s.problem.run(s.vars)
    final = s.tracker.forward(s.state, s.kq, s.dt, s.nsteps, s.npt)
    first, cct, qs = s.tracker.backward(_beam_size_seed(final))
    return {"final": final, "initial_gradient": first, "cct_gradient": cct, "qs_gradient": qs}


def work(case):
    """Pair terms of the Biot-Savart sum (x 27 operations); an adjoint's reverse pass counts two more such
    sums (the field's gradient at the points and at the segments).  Bytes: the segments (two vectors) and the
    points or states once, and what is returned."""
    c = case
    if c["kind"] == "search":
        n, steps, seg = c["designs"] * 8 * c["per_plane"], 274, 64800
        pairs, nbytes = 4.0 * steps * n * seg, c["designs"] * (seg * 48 + 27 * 8 + 88)
    elif c["kind"] in ("points", "field"):
        seg = _segments(c)
        pairs, nbytes = float(c["n"] * seg), seg * 48 + 48 * c["n"]
    else:
        n, seg = c["designs"] * c["particles"], _segments(c)
        pairs, nbytes = 4.0 * c["steps"] * n * seg, c["designs"] * seg * 48 + 96 * n
        if c["kind"] == "adjoint":
            pairs, nbytes = 3 * pairs, nbytes + 96 * n
    return {"bytes": nbytes, "flops": PAIR_FLOPS * pairs}


# ------------------------------------------------------- the same in 64 bits
# From the winding and QS records of the magnets (their shape parameters, placed in the global frame), in plain
# torch: discretised windings, Biot-Savart sum, hard-edge QS fields, RK4, and the reverse of each.
CHUNK = 1 << 23  # point x segment terms at a time


class _Segments:
    def __init__(self, spec, dev):
        kl, m, self.windings = [], [], []
        at = 0
        for rec, n in zip(spec.cct_params, spec.cct_counts):
            if n == 0:
                continue
            r = [float(v) for v in rec]
            o, axes = rec[:3], torch.tensor(rec[3:12].reshape(3, 3), device=dev)
            ksi = r[15] + r[16] * torch.arange(int(n) + 1, dtype=torch.float64, device=dev)
            phi = r[17] * ksi + r[18]
            for j in range(int(r[20])):
                if not (int(r[29]) >> j) & 1:
                    phi = phi + r[21 + j] * torch.sin((j + 1) * ksi)
            t = r[12] / (r[14] - torch.cos(ksi))
            local = torch.stack([t * r[13] * torch.cos(phi), t * r[13] * torch.sin(phi), t * torch.sin(ksi)], 1)
            p = torch.tensor(o, device=dev) + local @ axes
            tangent = torch.stack([-t * r[13] * torch.sin(phi), t * r[13] * torch.cos(phi), 0 * t], 1) @ axes
            kl.append(r[19] * (p[1:] - p[:-1]))
            m.append(0.5 * (p[1:] + p[:-1]))
            self.windings.append((at, int(n), r[19], int(r[20]), ksi, tangent))
            at += int(n)
        self.kl, self.m = torch.cat(kl), torch.cat(m)
        self.qs = [[float(v) for v in q] for q in spec.qs]
        self.uniform = torch.tensor(spec.bconst, device=dev)

    def pieces(self, npoints):
        n = max(1, CHUNK // max(1, npoints))
        return [slice(a, min(a + n, len(self.kl))) for a in range(0, len(self.kl), n)]

    def _offsets(self, p, part):
        m = self.m[part].T.contiguous()
        r = [p[:, c, None] - m[c] for c in range(3)]
        r2 = (r[0] * r[0]).addcmul_(r[1], r[1]).addcmul_(r[2], r[2])
        return r, r2, (r2 * torch.sqrt(r2)).reciprocal_()

    def _in_qs(self, q, p):
        d = p - torch.tensor(q[:3], dtype=torch.float64, device=p.device)
        x, y, z = (d @ torch.tensor(q[k:k + 3], dtype=torch.float64, device=p.device) for k in (3, 6, 9))
        inside = (z >= 0) & (z <= q[12]) & (torch.sqrt(x * x + y * y) <= q[15])
        return x, y, inside.double()

    def field(self, p):
        b = self.uniform.expand(len(p), 3).clone()
        for part in self.pieces(len(p)):
            r, _, w = self._offsets(p, part)
            kl = self.kl[part].T.contiguous()
            for c in range(3):
                i, j = (c + 1) % 3, (c + 2) % 3
                b[:, c] += (kl[i] * r[j]).addcmul_(kl[j], r[i], value=-1).mul_(w).sum(1)
        for q in self.qs:
            x, y, inside = self._in_qs(q, p)
            bx = inside * (q[13] * y + q[14] * x * y)
            by = inside * (q[13] * x + 0.5 * q[14] * (x * x - y * y))
            for c in range(3):
                b[:, c] += q[3 + c] * bx + q[6 + c] * by
        return b

    def reverse(self, p, bb, grad_kl, grad_m, grad_qs):
        """dJ/dp for dJ/dB = bb at p; adds dJ/d(kl, m, QS gradients) to the last three."""
        pb = torch.zeros_like(p)
        for part in self.pieces(3 * len(p)):
            r, r2, w = self._offsets(p, part)
            kl = self.kl[part]
            c = [r[(k + 1) % 3] * bb[:, (k + 2) % 3, None] - r[(k + 2) % 3] * bb[:, (k + 1) % 3, None] for k in range(3)]
            e = (c[0] * kl[:, 0] + c[1] * kl[:, 1] + c[2] * kl[:, 2]) * w  # b . dB of the pair
            e3 = -3 * e / r2
            for k in range(3):
                u = w * (bb[:, (k + 1) % 3, None] * kl[:, (k + 2) % 3] - bb[:, (k + 2) % 3, None] * kl[:, (k + 1) % 3])
                u = u.addcmul_(e3, r[k])
                pb[:, k] += u.sum(1)
                grad_m[part, k] -= u.sum(0)
                grad_kl[part, k] += (w * c[k]).sum(0)
        for n, q in enumerate(self.qs):
            x, y, inside = self._in_qs(q, p)
            bx = inside * (bb @ torch.tensor(q[3:6], dtype=torch.float64, device=p.device))
            by = inside * (bb @ torch.tensor(q[6:9], dtype=torch.float64, device=p.device))
            dx = bx * q[14] * y + by * (q[13] + q[14] * x)
            dy = bx * (q[13] + q[14] * x) - by * q[14] * y
            for k in range(3):
                pb[:, k] += q[3 + k] * dx + q[6 + k] * dy
            grad_qs[n, 0] += (bx * y + by * x).sum()
            grad_qs[n, 1] += (bx * x * y + by * 0.5 * (x * x - y * y)).sum()
        return pb

    def winding_gradients(self, grad_kl, grad_m):
        """Per winding [sum dJ/dkl . kl, dJ/d(first four tilt coefficients)]."""
        out = []
        for at, n, coef, ntilt, ksi, tangent in self.windings:
            gk, gm = grad_kl[at:at + n], grad_m[at:at + n]
            row = [(gk * self.kl[at:at + n]).sum()]
            for j in range(4):
                d = tangent * torch.sin((j + 1) * ksi)[:, None] * (1.0 if j < ntilt else 0.0)
                row.append((gk * coef * (d[1:] - d[:-1])).sum() + (gm * 0.5 * (d[1:] + d[:-1])).sum())
            out.append(torch.stack(row))
        return torch.stack(out)


STAGES = ((1, 0.5), (2, 0.5), (2, 1.0), (1, 0.0))  # weight in the step, and how far ahead the next stage lies


def _rk4(seg, p, v, kq, dt, ns, tape=None):
    """Each particle takes its own number of steps (rounding makes some take one more for the same length)."""
    k, h = kq[:, None], dt[:, None]
    for step in range(int(ns.max())):
        live = (step < ns).double()[:, None]
        sp, sv, q, u = 0.0, 0.0, p, v
        for weight, ahead in STAGES:
            b = seg.field(q)
            a = k * torch.linalg.cross(u, b)
            if tape is not None:
                tape.append((q, u, b))
            sp, sv = sp + weight * u, sv + weight * a
            q, u = p + ahead * h * u, v + ahead * h * a
        p, v = p + live * h / 6 * sp, v + live * h / 6 * sv
    return p, v


def _rk4_reverse(seg, pb, vb, kq, dt, ns, tape, grads):
    k = kq[:, None]
    for step in range(int(ns.max()) - 1, -1, -1):
        h = (dt * (step < ns))[:, None]
        sum_p, sum_v, qb, ub = 0.0, 0.0, 0.0, 0.0  # of the stage ahead
        for stage in (3, 2, 1, 0):
            q, u, b = tape[4 * step + stage]
            weight, ahead = STAGES[stage]
            up = weight * h / 6 * pb + ahead * h * qb  # dJ/d(position slope)
            ab = weight * h / 6 * vb + ahead * h * ub  # dJ/d(velocity slope)
            ub = up + k * torch.linalg.cross(b, ab)
            qb = seg.reverse(q, k * torch.linalg.cross(ab, u), *grads)
            sum_p, sum_v = sum_p + qb, sum_v + ub
        pb, vb = pb + sum_p, vb + sum_v
    return pb, vb


def _tracked(c, specs, state, kq, dt, ns, tapes=None):
    dev = engine.device()
    out, n = [], len(state) // len(specs)
    for d, spec in enumerate(specs):
        rows = slice(d * n, (d + 1) * n)
        t = [torch.tensor(a[rows], device=dev) for a in (state, kq, dt, ns)]
        seg, tape = _Segments(spec, dev), [] if tapes is not None else None
        p, v = _rk4(seg, t[0][:, :3], t[0][:, 3:], *t[1:], tape)
        if tapes is not None:
            tapes.append((seg, *t[1:], tape))
        out.append(torch.cat([p, v], 1))
    return torch.cat(out)


def _objectives(final, problem, designs):
    """The search's 11 objectives of final states (D n, 6): offsets and angles in the frame of the ideal particle
    at the end, in mm and mrad."""
    end, frame = problem.ip_end, problem.ip_end.get_natural_coordinate_system()
    rows = final.reshape(designs, -1, 6)
    rel = rows[..., :3] - numpy.array(end.position.to_list())
    dv = rows[..., 3:] - numpy.array(end.velocity.to_list())
    speed2 = (rows[..., 3:] ** 2).sum(-1)
    ax, ay = (numpy.array(a.to_list()) for a in (frame.XI, frame.YI))
    x, y = rel @ ax / MM, rel @ ay / MM
    xp, yp = ((dv @ a) / numpy.sqrt(speed2 - (dv @ a) ** 2) / MM for a in (ax, ay))
    hx, hy = (numpy.ptp(a.reshape(designs, -1, problem.group), axis=2) / 2 for a in (x, y))
    top = [numpy.abs(a).max(1) for a in (x, xp, y, yp)]
    return numpy.stack(top + [numpy.abs(a.mean(1)) for a in (x, xp, y, yp)]
                       + [numpy.abs(top[0] - top[2]), numpy.ptp(hx, axis=1), numpy.ptp(hy, axis=1)], 1)


def exact(case, seed):
    c = case
    if c["kind"] == "search":
        prob = optim.GantryPopulationProblem(particle_number_per_plane_per_dp=c["per_plane"])
        specs = [device_parts(bl).spec() for bl in prob.beamlines(_generation(c, seed))]
        ps = prob.particles
        sd = [engine.rk4_steps(prob.length, prob.footstep, p.speed) for p in ps]
        one = (numpy.array([p.position.to_list() + p.velocity.to_list() for p in ps]),
               numpy.array([p.e / p.relativistic_mass for p in ps]), numpy.array([d for _, d in sd]))
        one += (numpy.array([n for n, _ in sd]),)
        final = _tracked(c, specs, *(numpy.concatenate([a] * len(specs)) for a in one))
        return _objectives(final.cpu().numpy(), prob, len(specs))
    bls, rng = _workload(c, seed)
    specs = [device_parts(bl).spec() for bl in bls]
    dev = engine.device()
    if c["kind"] in ("points", "field"):
        p = torch.tensor(_points(c, bls[0], rng), device=dev)
        b = _Segments(specs[0], dev).field(p)
        return b.T.contiguous() if c["kind"] == "field" else b[0] if c["n"] == 1 else b
    beams = _beam(c, bls, rng)
    if c["kind"] == "facade":
        beams = beams * len(bls)
    state, kq, dt, ns = _arrays(c, beams)
    if c["kind"] != "adjoint":
        out = _tracked(c, specs, state, kq, dt, ns)
        return out.T.contiguous() if c["kind"] != "facade" else out.reshape(len(bls), -1, 6)
    tapes = []
    final = _tracked(c, specs, state, kq, dt, ns, tapes)
    seed_ = _beam_size_seed(final)
    first, cct, qs, n = [], [], [], c["particles"]
    for d, (seg, k, h, own, tape) in enumerate(tapes):
        grads = (torch.zeros_like(seg.kl), torch.zeros_like(seg.m),
                 torch.zeros((len(seg.qs), 2), dtype=torch.float64, device=dev))
        rows = seed_[d * n:(d + 1) * n]
        pb, vb = _rk4_reverse(seg, rows[:, :3], rows[:, 3:], k, h, own, tape, grads)
        first.append(torch.cat([pb, vb], 1))
        cct.append(seg.winding_gradients(grads[0], grads[1]))
        qs.append(grads[2])
    return {"final": final, "initial_gradient": torch.cat(first), "cct_gradient": torch.cat(cct),
            "qs_gradient": torch.cat(qs)}
