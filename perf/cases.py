"""The work that programs built on this package have it do, as measurable cases.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` builds what a program holds before the call (grids
with their fields, sources and records), ``run(state)`` is one pass through
the public entry points and ``work(case)`` the bytes and operations a pass
cannot do without.  ``exact(case, seed)`` is the same pass in plain torch, in
64 bits.

A case is a dict of plain values.  ``kind`` says which entry points a pass
calls:

* ``steps``: ``update_fields(n)`` on a periodic grid holding a superposition
  of plane waves, with waveform point sources; optionally probes and energy
  records (``records``), and in-run rescaling on FP16 grids (``rescale``);
* ``loop``: the reference driver's loop, n times "set J in the box of cells
  around the centre, then one step", through ``set_current_values`` and
  ``update_fields()``, and the six fields read back to the host at the end;
* ``currents``: the same loop handed over as one call,
  ``update_fields_with_currents``;
* ``device_j``: the device-array loop: J written by the caller's own device
  code on the grid's stream before each step, ``zeroed_currents`` at the end;
* ``pml``: ``update_fields(n)`` of a grid with an absorbing layer;
* ``batch``: many independent grids stepped together.

Fields come back as the grid's device arrays (FP16: stored values, that is
scale times physical value).
"""
from __future__ import annotations

import math

import numpy as np
import torch

torch.cuda.is_available()  # torch's HIP runtime starts before the first grid

from fdtd_method_amd import FDTD, FDTD_PML, Parameters, Precision  # noqa: E402
from fdtd_method_amd.batch import Batch  # noqa: E402

C = 3e10                 # include/Constants.h:6
PI = 3.14159265358       # include/Constants.h:11
PRECISION = {"fp64": Precision.FP64, "fp32": Precision.FP32, "fp16": Precision.FP16}
BYTES = {"fp64": 8, "fp32": 4, "fp16": 2}
SCALE_LOG2 = 12          # FP16: max |stored| below 2**12


def _case(name, kind, precision, Ni, Nj, Nk, steps, dx=1.0, dy=1.0, dz=1.0, sources=1, waves=2,
          records=False, rescale=0, pml=0.0, grids=1, blocking=-1):
    """`blocking`: -1 leaves the grid's own choice, L > 0 asks a batch for strip passes of L steps."""
    return dict(name=name, kind=kind, precision=precision, Ni=Ni, Nj=Nj, Nk=Nk, steps=steps,
                dx=dx, dy=dy, dz=dz, sources=sources, waves=waves, records=records,
                rescale=rescale, pml=pml, grids=grids, blocking=blocking)


def listed():
    return [
        # the reference driver as its tests run it (32^3, 100 steps): every
        # step is a call of its own, so latency and launches are what counts
        _case("loop_fp64_32", "loop", "fp64", 32, 32, 32, 100, sources=0, waves=0),
        # the convergence-test size in a longer run: a wave on 64^3, below
        # the size at which grids step in blocked passes by themselves
        _case("steps_fp64_64", "steps", "fp64", 64, 64, 64, 200, sources=0),
        # a caller's own device code writes J (the Kokkos driver's loop), on
        # a ragged grid
        _case("device_j_fp64_200x151x97", "device_j", "fp64", 200, 151, 97, 20,
              dx=1.0, dy=1.25, dz=0.8, sources=0, waves=0),
        # an ordinary ragged grid, odd along x, a step count no pass length divides
        _case("steps_fp32_251x190x131", "steps", "fp32", 251, 190, 131, 50,
              dx=1.0, dy=0.9, dz=1.1, sources=4),
        # an ordinary run watched through probes and energy records
        _case("records_fp32_256", "steps", "fp32", 256, 256, 256, 40, sources=1, records=True),
        # the reference's benchmark command, sample 512 25, as one call
        _case("currents_fp64_512", "currents", "fp64", 512, 512, 512, 25, sources=0, waves=0),
        # the benchmark grid in 32 bits
        _case("steps_fp32_512", "steps", "fp32", 512, 512, 512, 20),
        # the same in 16-bit storage with in-run rescaling
        _case("steps_fp16_512", "steps", "fp16", 512, 512, 512, 40, rescale=20),
        # the reference driver's absorbing-layer run at an ordinary size
        _case("pml_fp64_128", "pml", "fp64", 128, 128, 128, 25, pml=0.2),
        # the benchmark's absorbing-layer workload
        _case("pml_fp32_512", "pml", "fp32", 512, 512, 512, 10, pml=0.2),
        # a sweep over many independent designs of uneven sizes, 32 to 160 cells a side
        _case("batch_fp32_64", "batch", "fp32", 32, 160, 16, 40, waves=1, grids=64, blocking=4),
        # the largest: the benchmark's anisotropic grid
        _case("steps_fp32_1024x1024x256", "steps", "fp32", 1024, 1024, 256, 24, sources=4),
    ]


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "steps", "loop", "currents", "device_j", "pml",
                       "pml", "batch"])
    precision = rng.choice(["fp64", "fp32", "fp32", "fp16"])
    if kind in ("loop", "currents", "device_j"):
        precision = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "batch":
        n = rng.randint(8, 64)
        lo = 16 * rng.randint(2, 4)
        hi = lo + 16 * rng.randint(2, 6)
        return _case("", "batch", precision, lo, hi, 16, rng.randint(8, 40), waves=1, grids=n,
                     blocking=rng.choice([0, 4]))
    # cells over their logarithm, sides within a factor of a few of each other
    top = {"steps": 2.0e8, "currents": 1.3e8, "pml": 4e7, "device_j": 6e6, "loop": 1e6}[kind]
    cells = math.exp(rng.uniform(math.log(2.5e4), math.log(top)))
    side = cells ** (1.0 / 3.0)
    fx, fy = math.exp(rng.uniform(-0.7, 0.7)), math.exp(rng.uniform(-0.7, 0.7))
    Ni, Nj = max(16, round(side * fx)), max(16, round(side * fy))
    Nk = max(16, round(cells / (Ni * Nj)))
    if rng.random() < 0.5:  # programs also take round sizes
        Ni, Nj, Nk = (max(16, 16 * round(v / 16)) for v in (Ni, Nj, Nk))
    Nk = max(16, min(Nk, int(top) // (Ni * Nj)))
    budget = {"fp64": 4e8, "fp32": 8e8, "fp16": 8e8}[precision] * (0.3 if kind == "pml" else 1.0)
    steps = int(max(1, min(budget / (Ni * Nj * Nk), 120)))
    steps = rng.randint(max(1, steps // 2), steps)
    if kind in ("loop", "device_j"):
        steps = min(steps, 60)
    d = [1.0, 1.0, 1.0] if rng.random() < 0.5 else [round(rng.uniform(0.8, 1.25), 3) for _ in range(3)]
    return _case("", kind, precision, Ni, Nj, Nk, steps, dx=d[0], dy=d[1], dz=d[2],
                 sources=rng.randint(0, 4) if kind in ("steps", "pml") else 0,
                 waves=2 if kind in ("steps", "pml") else 0,
                 records=kind == "steps" and precision == "fp32" and rng.random() < 0.25,
                 rescale=20 if kind == "steps" and precision == "fp16" and rng.random() < 0.5 else 0,
                 pml=rng.choice([0.1, 0.15, 0.2]) if kind == "pml" else 0.0)


# ---------------------------------------------------------------------------
# Inputs, from the seed alone

def _dt(case):
    """Half the stability limit."""
    return 0.5 / (C * math.sqrt(sum(1.0 / case[a] ** 2 for a in ("dx", "dy", "dz"))))


def _shape(case):
    return case["Ni"], case["Nj"], case["Nk"]


def _waves(case, seed):
    """Plane waves with whole wave numbers (add_plane_wave's arguments)."""
    rng = np.random.default_rng([seed, 1])
    out = []
    while len(out) < case["waves"]:
        m = [int(x) for x in rng.integers(-6, 7, 3)]
        if not any(m):
            continue
        out.append((m, float(rng.uniform(0.1, 1.0)), float(rng.uniform(0.0, 2.0 * math.pi)),
                    [float(x) for x in rng.standard_normal(3)]))
    return out


def _sources(case, seed):
    """Gaussian-modulated point currents at cells of the main box."""
    rng = np.random.default_rng([seed, 2])
    dt = _dt(case)
    lo = [int(n * case["pml"]) for n in _shape(case)]
    out = []
    for _ in range(case["sources"]):
        i, j, k = (int(rng.integers(p, n - p)) for n, p in zip(_shape(case), lo))
        out.append(dict(i=i, j=j, k=k, comp=int(rng.integers(3)), kind=1,
                        amp=float(rng.uniform(0.5, 1.5)) * 1e-3 / dt, period=float(rng.uniform(16, 40)) * dt,
                        t0=12 * dt, sigma=10 * dt, phase=float(rng.uniform(0.0, 6.0))))
    return out


def _box(case):
    """The 2x2x2 cells around the centre, where the drivers set J."""
    Ni, Nj, Nk = _shape(case)
    return [i + j * Ni + k * Ni * Nj for k in (Nk // 2 - 1, Nk // 2)
            for j in (Nj // 2 - 1, Nj // 2) for i in (Ni // 2 - 1, Ni // 2)]


def _box_values(case, seed):
    """J of every step: values[step][cell], the same in Jx, Jy and Jz as in the drivers."""
    rng = np.random.default_rng([seed, 3])
    amp, period = rng.uniform(0.5, 1.5, 8) / _dt(case), rng.uniform(8.0, 32.0)
    t = np.arange(1, case["steps"] + 1)
    return np.sin(2.0 * PI * t / period)[:, None] * amp[None, :]


def _probe_cells(case, seed):
    rng = np.random.default_rng([seed, 4])
    return [tuple(int(rng.integers(n)) for n in _shape(case)) + (c,) for c in (0, 1, 2, 3, 4, 5, 2, 2)]


def _batch_cases(case, seed):
    """The grids of a batch: sides from {Ni, Ni + Nk, .., Nj}, one source each."""
    rng = np.random.default_rng([20240, case["grids"], case["Ni"]])  # the sizes are the case's, not the seed's
    sides = np.arange(case["Ni"], case["Nj"] + 1, case["Nk"])
    return [(_case("", "steps", case["precision"], *(int(x) for x in rng.choice(sides, 3)),
                   case["steps"], sources=1, waves=case["waves"]), seed * 1000 + q)
            for q in range(case["grids"])]


# ---------------------------------------------------------------------------
# The program

def _grid(case, seed):
    p = Parameters(*_shape(case), dx=case["dx"], dy=case["dy"], dz=case["dz"])
    if case["kind"] == "pml":
        g = FDTD_PML(p, _dt(case), case["pml"], PRECISION[case["precision"]])
    else:
        g = FDTD(p, _dt(case), PRECISION[case["precision"]])
    for m, amp, phase, pol in _waves(case, seed):
        g.add_plane_wave(m, amp, phase, pol)
    if case["precision"] == "fp16":
        g.autoscale(SCALE_LOG2)
        if case["rescale"]:
            g.set_autoscale_interval(case["rescale"], SCALE_LOG2)
    src = _sources(case, seed)
    if src:
        g.set_point_sources(src)
    return g


def prepare(case, seed):
    if case["kind"] == "batch":
        grids = [_grid(c, s) for c, s in _batch_cases(case, seed)]
        b = Batch(grids)
        if case["blocking"] > 0:
            b.set_time_blocking_strips(case["blocking"])
        return dict(case=case, batch=b, grids=grids)
    g = _grid(case, seed)
    state = dict(case=case, grid=g)
    if case["kind"] in ("loop", "currents", "device_j"):
        values = _box_values(case, seed)
        cells = _box(case)
        if case["kind"] == "device_j":
            Ni, Nj, Nk = _shape(case)
            j = [torch.as_tensor(g.device_field(c), device="cuda").view(Nk, Nj, Ni) for c in (6, 7, 8)]
            state.update(stream=g.torch_stream(), box=[
                x[Nk // 2 - 1:Nk // 2 + 1, Nj // 2 - 1:Nj // 2 + 1, Ni // 2 - 1:Ni // 2 + 1] for x in j],
                values=torch.as_tensor(values, dtype=j[0].dtype, device="cuda").view(-1, 2, 2, 2))
        else:
            index = np.array(cells * 3, dtype=np.int64)
            comp = np.repeat(np.array([6, 7, 8], dtype=np.int32), 8)
            state["writes"] = [(index, comp, np.tile(v, 3)) for v in values]
    if case["records"]:
        g.set_probes(_probe_cells(case, seed), case["steps"])
        g.set_energy_interval(20, case["steps"])
    torch.cuda.synchronize()
    return state


def _device_fields(g):
    return [torch.as_tensor(g.device_field(c), device="cuda") for c in range(6)]


def run(state):
    case = state["case"]
    kind, steps = case["kind"], case["steps"]
    if kind == "batch":
        state["batch"].update_fields(steps)
        fields = [_device_fields(g) for g in state["grids"]]
        out = [torch.cat([f[c] for f in fields]) for c in range(6)]
        torch.cuda.current_stream().synchronize()  # the next steps write the buffers just read
        return out
    g = state["grid"]
    if kind == "loop":
        for index, comp, value in state["writes"]:
            g.set_current_values(index, comp, value)
            g.update_fields()
        g.zeroed_currents()
        return g.fields()
    if kind == "currents":
        g.update_fields_with_currents(state["writes"])
        g.zeroed_currents()
        return _device_fields(g)
    if kind == "device_j":
        with torch.cuda.stream(state["stream"]):
            for s in range(steps):
                for box in state["box"]:
                    box.copy_(state["values"][s])
                g.update_fields()
        g.zeroed_currents()
        return _device_fields(g)
    if case["records"]:
        g.rewind_records()
    g.update_fields(steps)
    if case["records"]:
        probes, (at, sums) = g.read_probes(), g.energy_records()
        return dict(fields=_device_fields(g), probes=probes, sums=sums)
    if case["precision"] == "fp16":
        return dict(fields=_device_fields(g), scales=g.get_scales())
    return _device_fields(g)


# ---------------------------------------------------------------------------
# What a pass cannot do without

def work(case):
    if case["kind"] == "batch":
        parts = [work(c) for c, _ in _batch_cases(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    Ni, Nj, Nk = _shape(case)
    cells = Ni * Nj * Nk
    p = [int(n * case["pml"]) for n in (Ni, Nj, Nk)]
    layer = cells - (Ni - 2 * p[0]) * (Nj - 2 * p[1]) * (Nk - 2 * p[2])
    # E and B, and in the layer the 12 split fields, read and written once a pass
    words = 12 * cells + 24 * layer
    # a step of a cell: E 18 operations, both half steps of B 21 (their curl terms are the same);
    # in the layer 12 splits of 4 and 6 sums
    return {"bytes": float(words * BYTES[case["precision"]]),
            "flops": float(case["steps"] * (39 * (cells - layer) + 54 * layer))}


# ---------------------------------------------------------------------------
# The same passes in 64 bits

def _stored(x, precision, scale):
    """x as a grid of this precision holds it."""
    if precision == "fp64":
        return x
    if precision == "fp32":
        return x.float().double()
    return (x * scale).half().double() / scale


def _target(m):
    """The power of two that puts a maximum of m just below 2**SCALE_LOG2."""
    return 2.0 ** (SCALE_LOG2 - math.frexp(m)[1]) if m > 0 else 1.0


def _initial(case, seed, dev):
    Ni, Nj, Nk = _shape(case)
    f = [torch.zeros(Nk, Nj, Ni, dtype=torch.float64, device=dev) for _ in range(6)]
    at = [(0.5, 0, 0), (0, 0.5, 0), (0, 0, 0.5), (0, 0.5, 0.5), (0.5, 0, 0.5), (0.5, 0.5, 0)]
    axis = [torch.arange(n, dtype=torch.float64, device=dev) for n in (Ni, Nj, Nk)]
    for m, amp, phase, pol in _waves(case, seed):
        k = 2.0 * np.pi * np.array([m[0] / Ni, m[1] / Nj, m[2] / Nk])
        kh = k / np.linalg.norm(k)
        e = np.asarray(pol) - np.dot(pol, kh) * kh
        e = amp * e / np.linalg.norm(e)
        a = list(e) + list(np.cross(kh, e))
        for c in range(6):
            o = at[c]
            ph = ((axis[0] + o[0]) * k[0]).view(1, 1, -1) + ((axis[1] + o[1]) * k[1]).view(1, -1, 1) \
                + ((axis[2] + o[2]) * k[2]).view(-1, 1, 1) + phase
            f[c] = _stored(f[c] + a[c] * torch.cos(ph), case["precision"], 1.0)
    scales = [1.0] * 6
    if case["precision"] == "fp16":
        scales = [_target(float(x.abs().max())) for x in f]
        f = [_stored(x, "fp16", s) for x, s in zip(f, scales)]
    return f, scales


def _waveform(s, t):
    tau = t - s["t0"]
    return s["amp"] * math.sin(2.0 * PI * tau / s["period"] + s["phase"]) \
        * math.exp(-(tau * tau) / (2.0 * s["sigma"] ** 2))


def _currents(case, seed, step):
    """[(component, flat cell, J)] of one step."""
    Ni, Nj, _ = _shape(case)
    dt = _dt(case)
    out = [(s["comp"], s["i"] + s["j"] * Ni + s["k"] * Ni * Nj, _waveform(s, (step + 1) * dt))
           for s in _sources(case, seed)]
    if case["kind"] in ("loop", "currents", "device_j"):
        v = _box_values(case, seed)[step]
        out += [(c, cell, float(x)) for c in range(3) for cell, x in zip(_box(case), v)]
    return out


def _profile(n, percent, d, dt, dev):
    """(decay, coefficient) of the layer along one axis."""
    p = int(n * percent)
    decay, coef = np.ones(n), np.full(n, C * dt / d)
    if p > 0:
        top = -2.5 * math.log(1e-12) / (p * d)
        for i in range(n):
            dist = p - i if i < p else i + 1 + p - n
            if dist > 0:
                s = top * (dist / p) ** 4
                decay[i] = math.exp(-s * dt * C)
                coef[i] = (1.0 - decay[i]) / (s * d)
    return tuple(torch.as_tensor(x, device=dev) for x in (decay, coef))


def _exact_steps(case, seed, dev):
    Ni, Nj, Nk = _shape(case)
    dt = _dt(case)
    f, scales = _initial(case, seed, dev)
    E, B = f[:3], f[3:]
    cx, cy, cz = (C * dt / case[a] for a in ("dx", "dy", "dz"))
    up = lambda x, d: torch.roll(x, -1, d)   # noqa: E731  neighbour +1 (dims: 2 x, 1 y, 0 z)
    dn = lambda x, d: torch.roll(x, 1, d)    # noqa: E731  neighbour -1
    pml = case["kind"] == "pml"
    if pml:
        p = [int(n * case["pml"]) for n in (Ni, Nj, Nk)]
        main = torch.zeros(Nk, Nj, Ni, dtype=torch.bool, device=dev)
        main[p[2]:Nk - p[2], p[1]:Nj - p[1], p[0]:Ni - p[0]] = True
        layer = (~main).double()
        prof = [_profile(n, case["pml"], case[a], dt, dev)
                for n, a in ((Ni, "dx"), (Nj, "dy"), (Nk, "dz"))]
        (ax, sx), (ay, sy), (az, sz) = [tuple(v.view(s) for v in q) for q, s in
                                        zip(prof, ((1, 1, -1), (1, -1, 1), (-1, 1, 1)))]
        S = [torch.zeros_like(E[0]) for _ in range(12)]

    def split(q, decay, term):
        S[q].mul_(decay).add_(term).mul_(layer)

    def half_b():
        curl = (cz * (up(E[1], 0) - E[1]) - cy * (up(E[2], 1) - E[2]),
                cx * (up(E[2], 2) - E[2]) - cz * (up(E[0], 0) - E[0]),
                cy * (up(E[0], 1) - E[0]) - cx * (up(E[1], 2) - E[1]))
        for d in range(3):
            B[d] = torch.where(main, B[d] + 0.5 * curl[d], B[d]) if pml else B[d] + 0.5 * curl[d]

    rows, sums, cells = [], [], _probe_cells(case, seed) if case["records"] else []
    for s in range(case["steps"]):
        if case["rescale"] and s and s % case["rescale"] == 0:
            scales = [_target(float(x.abs().max())) for x in E + B]
        half_b()
        if pml:
            split(6, ay, -sy * (up(E[2], 1) - E[2]))
            split(7, az, sz * (up(E[1], 0) - E[1]))
            split(8, ax, sx * (up(E[2], 2) - E[2]))
            split(9, az, -sz * (up(E[0], 0) - E[0]))
            split(10, ax, -sx * (up(E[1], 2) - E[1]))
            split(11, ay, sy * (up(E[0], 1) - E[0]))
            for d in range(3):
                B[d] = torch.where(main, B[d], S[6 + 2 * d] + S[7 + 2 * d])
        curl = (cy * (B[2] - dn(B[2], 1)) - cz * (B[1] - dn(B[1], 0)),
                cz * (B[0] - dn(B[0], 0)) - cx * (B[2] - dn(B[2], 2)),
                cx * (B[1] - dn(B[1], 2)) - cy * (B[0] - dn(B[0], 1)))
        for d in range(3):
            E[d] = E[d] + curl[d]
        for c, cell, j in _currents(case, seed, s):
            E[c].view(-1)[cell] += -4.0 * PI * dt * j
        if pml:
            split(0, ay, sy * (B[2] - dn(B[2], 1)))
            split(1, az, -sz * (B[1] - dn(B[1], 0)))
            split(2, ax, -sx * (B[2] - dn(B[2], 2)))
            split(3, az, sz * (B[0] - dn(B[0], 0)))
            split(4, ax, sx * (B[1] - dn(B[1], 2)))
            split(5, ay, -sy * (B[0] - dn(B[0], 1)))
            for d in range(3):
                E[d] = torch.where(main, E[d], S[2 * d] + S[2 * d + 1])
        half_b()
        if cells:
            rows.append([float((E + B)[c][k, j, i]) for i, j, k, c in cells])
            if (s + 1) % 20 == 0:
                sums.append([float((x * x).sum()) for x in E + B])
    fields = [x.reshape(-1) * k for x, k in zip(E + B, scales)]
    return fields, scales, rows, sums


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "batch":
        parts = [_exact_steps(c, s, dev)[0] for c, s in _batch_cases(case, seed)]
        return [torch.cat([p[c] for p in parts]) for c in range(6)] if case["precision"] != "fp16" else None
    fields, scales, rows, sums = _exact_steps(case, seed, dev)
    if case["records"]:
        return dict(fields=fields, probes=np.array(rows), sums=np.array(sums).reshape(-1, 6))
    if case["precision"] == "fp16" and case["kind"] == "steps":
        return dict(fields=fields, scales=scales)
    if case["kind"] == "loop":
        return [x.cpu().numpy() for x in fields]
    return fields
