"""The work a user of this framework has it do, as cases that can be timed.

listed()          the cases
draw(rng)         one more case of the same ranges
prepare(case, s)  what a user's program has in hand before the call
run(state)        one pass through the public entry points, and its outputs
work(case)        bytes and operations the pass cannot do without
exact(case, s)    the outputs in 64 bits, from plain torch and numpy

Kinds of case:

  grid     one engine stepped over a grid: sources, absorber, material boxes,
           dispersive spheres, lumped port, recording box -- run_batch from a
           reset state, then what the program reads back
  sweep    several microstrip structures stepped together until a step count
  farfield near-field to far-field transform of a closed box of phasors
  train    one training batch of the ringdown extrapolator
  infer    one inference batch of it
"""
from __future__ import annotations

import math

import numpy as np
import torch

C0 = 299792458.0
EPS0 = 8.854187817e-12
MU0 = 1.256637062e-6
Z0 = 376.730313668

DRUDE = (1e15, 1e13)                          # plasma frequency, collision rate
LORENTZ = (2 * math.pi * 10e9, 1e9, 3.0)      # resonance, damping, delta eps
LORENTZ_EPS = 2.0
FREQS = tuple(np.linspace(1e9, 20e9, 64))     # port spectra
BOX_FREQS = (5e9, 10e9, 15e9)                 # recording box


def listed():
    return [
        # One small microstrip structure on its own: S11 of a port, the
        # engine's smallest grids, where a step is launches and little else.
        _grid("microstrip_small", 72, 60, 32, steps=600, scene="microstrip", absorber="cpml", delta=5e-4),
        # The plain cavity at the size the reference publishes step times for.
        _grid("cavity_100", 100, 100, 100, steps=600, scene="empty", absorber="pec", delta=1e-3),
        # Mur on six faces, the cheap absorber, and a few dielectric boxes.
        _grid("mur_160", 160, 144, 120, steps=400, scene="boxes", boxes=40, absorber="mur", delta=5e-4),
        # An odd mesh: no axis a multiple of four cells.
        _grid("boxes_odd", 151, 133, 117, steps=400, scene="boxes", boxes=60, absorber="cpml", delta=5e-4),
        # Every extension at once: CPML and Mur, port, Drude and Lorentz
        # spheres, port spectra, recording box and its far field.
        _grid("composite_144", 160, 144, 128, steps=480, scene="port_spheres", absorber="cpml_mur", delta=5e-4),
        # Dielectric boxes in an 8-cell CPML, the ordinary production grid.
        _grid("boxes_256", 256, 256, 256, steps=500, scene="boxes", boxes=200, absorber="cpml", delta=5e-4),
        # The same on a grid twice as large with rows longer than one wave.
        _grid("boxes_384", 256, 320, 384, steps=400, scene="boxes", boxes=200, absorber="cpml", delta=5e-4),
        # A parameter sweep: microstrip structures of uneven size together.
        {"name": "sweep_32", "kind": "sweep", "structures": 32, "steps": 400},
        # Two pattern cuts of a small antenna's box.
        {"name": "farfield_cuts", "kind": "farfield", "n1": 62, "n2": 55, "n3": 41, "thetas": 181, "phis": 2,
         "freq": 2.4e9, "delta": 1e-3},
        # The full sphere at one degree on the box of a large grid.
        {"name": "farfield_sphere", "kind": "farfield", "n1": 349, "n2": 349, "n3": 221, "thetas": 181, "phis": 360,
         "freq": 10e9, "delta": 5e-4},
        # Forward and backward of one full training batch.
        {"name": "train_256", "kind": "train", "batch": 256, "samples": 256, "tail": 512, "update": False},
        # Inference over the structures of a checkpoint.
        {"name": "infer_256", "kind": "infer", "batch": 256, "samples": 256, "tail": 512, "tails": True},
    ]


def _grid(name, nx, ny, nz, steps, scene, absorber, delta, boxes=0, mode="physical"):
    return {"name": name, "kind": "grid", "nx": nx, "ny": ny, "nz": nz, "steps": steps, "scene": scene,
            "absorber": absorber, "delta": delta, "boxes": boxes, "mode": mode}


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("grid", "grid", "grid", "grid", "sweep", "farfield", "train", "infer"))
    if kind == "grid":
        scene = rng.choice(("empty", "boxes", "boxes", "microstrip", "port_spheres"))
        if scene == "microstrip":
            n = [rng.randint(60, 220), rng.randint(60, 120), rng.randint(30, 48)]
            absorber = "cpml"
        elif scene == "port_spheres":
            n = [rng.randint(100, 176), rng.randint(100, 176), rng.randint(96, 144)]
            absorber = "cpml_mur"
        else:
            n = [_spread(rng, 40, 320) for _ in range(3)]
            absorber = rng.choice(("pec", "mur", "cpml", "cpml", "cpml"))
        if rng.random() < 0.6:  # most programs mesh with whole vectors along z
            n[2] = max(4, n[2] // 4 * 4)
        cells = n[0] * n[1] * n[2]
        steps = max(100, min(_spread(rng, 200, 800), int(1.2e10 / cells)))
        case = _grid("", *n, steps=steps, scene=scene, absorber=absorber, delta=rng.choice((2.5e-4, 5e-4, 1e-3)),
                     boxes=_spread(rng, 1, 400) if scene == "boxes" else 0,
                     mode=rng.choice(("physical", "physical", "compat")) if scene == "boxes" else "physical")
        del case["name"]
        return case
    if kind == "sweep":
        return {"kind": "sweep", "structures": _spread(rng, 2, 32), "steps": rng.randint(200, 400)}
    if kind == "farfield":
        n = [_spread(rng, 20, 340) for _ in range(3)]
        if rng.random() < 0.4:
            angles = (rng.randint(37, 361), rng.randint(1, 4))
        else:
            angles = (rng.randint(19, 181), rng.randint(24, 360))
        return {"kind": "farfield", "n1": n[0], "n2": n[1], "n3": n[2], "thetas": angles[0], "phis": angles[1],
                "freq": rng.choice((2.4e9, 5e9, 10e9, 15e9)), "delta": 5e-4}
    batch = _spread(rng, 1, 256)
    case = {"kind": kind, "batch": batch, "samples": rng.choice((128, 256, 256)), "tail": _spread(rng, 16, 512)}
    case["update" if kind == "train" else "tails"] = rng.random() < 0.5
    return case


# ------------------------------------------------------------------- scenes
def _scene(case, seed):
    """What stands on the grid: material boxes and conductors in order, the
    source, dispersive cells, the lumped port and the recording box."""
    rng = np.random.default_rng(seed)
    n = (case["nx"], case["ny"], case["nz"])
    s = {"n": n, "delta": case["delta"], "materials": [], "sources": [], "port": None, "spheres": [], "box": None,
         "cpml": None, "mur": None, "mode": case["mode"]}
    fc = 0.03 * C0 / case["delta"]  # about 30 cells a wavelength at the top
    if case["absorber"] in ("cpml", "cpml_mur"):
        # eight layers, fewer where the axis is too short to hold both faces
        s["cpml"] = [min(8, (n[f // 2] - 1) // 2) for f in range(6)]
    if case["absorber"] == "mur":
        s["mur"] = [True] * 6
    if case["absorber"] == "cpml_mur":
        s["cpml"][5] = 0
        s["mur"] = [False] * 5 + [True]
    amp = float(rng.uniform(0.5, 2.0))
    mid = [int(m // 2 + rng.integers(-2, 3)) for m in n]
    if case["scene"] == "microstrip":
        _microstrip(s, rng, n, amp)
    elif case["scene"] == "port_spheres":
        s["port"] = (n[0] // 2, n[0] // 2 + 1, n[1] // 2, n[1] // 2 + 1, n[2] // 2 - 2, n[2] // 2 + 2)
        s["sources"] = [(n[0] // 2, n[1] // 2, k, -amp) for k in range(n[2] // 2 - 2, n[2] // 2 + 2)]
        s["fc"] = 20e9
        lo = 18
        s["box"] = (lo, n[0] - lo, lo, n[1] - lo, lo, n[2] - lo)
        taken = [(np.array([m // 2 for m in n]), 4)]
        while len(s["spheres"]) < 8:
            r = int(rng.integers(4, 9))
            c = np.array([rng.integers(lo + r, m - lo - r) for m in n])
            if all(((c - p) ** 2).sum() > (r + q + 2) ** 2 for p, q in taken):
                taken.append((c, r))
                s["spheres"].append(("drude" if len(s["spheres"]) % 2 else "lorentz", c, r))
    else:
        for _ in range(case["boxes"]):
            side = [int(min(rng.integers(5, 41), m - 2)) for m in n]
            at = [int(rng.integers(1, m - w)) for m, w in zip(n, side)]
            s["materials"].append((float(rng.uniform(1, 10)), float(rng.uniform(0, 0.05)),
                                   (at[0], at[0] + side[0], at[1], at[1] + side[1], at[2], at[2] + side[2])))
        s["sources"] = [(*mid, amp)]
    s.setdefault("fc", fc)
    s["probe"] = (min(mid[0] + 12, n[0] - 1), mid[1], mid[2])
    return s


def _microstrip(s, rng, n, amp):
    """Ground, substrate and a bent trace with a port from ground to trace."""
    g, h, w = 8, int(rng.integers(2, 9)), int(rng.integers(2, 9))
    lo = 14
    s["materials"] = [(None, 0.0, (0, n[0], 0, n[1], g, g + 1)),
                      (float(rng.uniform(2.2, 10.2)), 0.0, (0, n[0], 0, n[1], g + 1, g + 1 + h))]
    top = (n[0] - lo - w, n[1] - lo - w)
    x, y = int(rng.integers(lo, top[0])), int(rng.integers(lo, top[1]))
    i, j = x + w // 2, y + w // 2
    for q in range(int(rng.integers(2, 7))):
        if q % 2 == 0:
            t = int(rng.integers(lo, top[0]))
            s["materials"].append((None, 0.0, (min(x, t), max(x, t) + w, y, y + w, g + 1 + h, g + 2 + h)))
            x = t
        else:
            t = int(rng.integers(lo, top[1]))
            s["materials"].append((None, 0.0, (x, x + w, min(y, t), max(y, t) + w, g + 1 + h, g + 2 + h)))
            y = t
    s["port"] = (i, i + 1, j, j + 1, g + 1, g + 1 + h)
    s["sources"] = [(i, j, k, -amp) for k in range(g + 1, g + 1 + h)]
    s["fc"] = 20e9


def _pulse(s, dt, steps):
    """The Gaussian pulse of the scene (f0 = 0, cutoff fc) at every step."""
    t0, tau = 9.0 / (2 * math.pi * s["fc"]), 3.0 / (2 * math.pi * s["fc"])
    return np.exp(-((np.arange(steps) * dt - t0) / tau) ** 2)


def _sphere_cells(c, r):
    g = np.mgrid[-r:r + 1, -r:r + 1, -r:r + 1].reshape(3, -1).T
    return (g[(g * g).sum(1) <= r * r] + c).astype(np.int64)


def _build(s):
    """Operator, engine and extensions of a scene."""
    from openems_amd import ADE_DRUDE, ADE_LORENTZ, MODE_COMPAT, MODE_PHYSICAL, CpmlBoundaries, HipEngine, Operator

    op = Operator.uniform(*s["n"], s["delta"])
    for eps, sigma, region in s["materials"]:
        if eps is None:
            op.set_pec(region)
        else:
            op.set_material(eps, 1.0, sigma, 0.0, region)
    cells = {"drude": [], "lorentz": []}
    for kind, c, r in s["spheres"]:
        p = _sphere_cells(c, r)
        cells[kind].append(p)
        if kind == "lorentz":
            columns = {}
            for i, j, k in p:
                lo, hi = columns.get((i, j), (k, k))
                columns[i, j] = (min(lo, k), max(hi, k))
            for (i, j), (lo, hi) in columns.items():
                op.set_material(LORENTZ_EPS, 1.0, 0.0, 0.0, (i, i + 1, j, j + 1, lo, hi + 1))
    if s["port"]:
        op.add_lumped_element(2, s["port"], 50.0)
    eng = HipEngine(op)
    x = {}
    if s["cpml"]:
        x["cpml"] = eng.cpml(CpmlBoundaries(layers=s["cpml"],
                                            mode=MODE_PHYSICAL if s["mode"] == "physical" else MODE_COMPAT))
    if s["mur"]:
        x["mur"] = eng.mur(s["mur"])
    if cells["drude"]:
        x["drude"] = eng.ade(ADE_DRUDE, DRUDE, np.concatenate(cells["drude"]), MODE_PHYSICAL)
    if cells["lorentz"]:
        x["lorentz"] = eng.ade(ADE_LORENTZ, LORENTZ, np.concatenate(cells["lorentz"]), MODE_PHYSICAL)
    if s["port"]:
        x["port"] = eng.lumped_port(2, s["port"], FREQS)
    else:
        x["probe"] = eng.field_probe(s["probe"])
    if s["box"]:
        x["box"] = eng.nf2ff_box(s["box"], BOX_FREQS, time_stride=4)
    return op, eng, x


def _angles(thetas, phis):
    """Polar cuts where few planes are asked for, else the whole sphere."""
    if phis <= 4:
        return np.linspace(-np.pi, np.pi, thetas), np.arange(phis) * np.pi / 2
    return np.linspace(0, np.pi, thetas), np.linspace(0, 2 * np.pi, phis + 1)[:-1]


BOX_ANGLES = (91, 120)


def _surfaces(case, seed):
    """Tangential phasors on a box around seeded current elements, as a run
    records them: their fields at the nodes, a little noise on top."""
    rng = np.random.default_rng(seed)
    n, d, k = (case["n1"], case["n2"], case["n3"]), case["delta"], 2 * np.pi * case["freq"] / C0
    axes = [np.arange(m) * d for m in n]
    dev = "cuda"
    src = np.stack([rng.uniform(0.35, 0.65, 4) * m * d for m in n], 1)
    mom = rng.standard_normal((4, 3)) + 1j * rng.standard_normal((4, 3))
    gen = torch.Generator(device=dev).manual_seed(int(seed) & 0x7FFFFFFF)
    faces = []
    for ax in range(3):
        a1, a2 = (ax + 1) % 3, (ax + 2) % 3
        for side in (0, 1):
            pos = axes[ax][-1] if side else 0.0
            p = torch.zeros(n[a1], n[a2], 3, dtype=torch.float64, device=dev)
            p[..., ax] = pos
            p[..., a1] = torch.tensor(axes[a1], device=dev)[:, None]
            p[..., a2] = torch.tensor(axes[a2], device=dev)[None, :]
            E = torch.zeros(n[a1], n[a2], 3, dtype=torch.complex128, device=dev)
            H = torch.zeros_like(E)
            for c, m in zip(src, mom):
                v = p - torch.tensor(c, device=dev)
                r = v.norm(dim=-1, keepdim=True)
                u = (v / r).to(torch.complex128)
                g = torch.exp(-1j * k * r) / (4 * np.pi * r)
                q = torch.tensor(m, device=dev).expand_as(u)
                kr = k * r
                along = u * (u * q).sum(-1, keepdim=True)
                H += 1j * k * g * (1 + 1 / (1j * kr)) * torch.linalg.cross(q, u)
                E += 1j * k * Z0 * g * (along - q + (3 * along - q) * (1 / (1j * kr) + 1 / (1j * kr) ** 2))
            E += 1e-3 * E.abs().mean() * torch.randn(E.shape, dtype=E.dtype, device=dev, generator=gen)
            H += 1e-3 * H.abs().mean() * torch.randn(H.shape, dtype=H.dtype, device=dev, generator=gen)
            faces.append((ax, 1 if side else -1, float(pos), axes[a1], axes[a2],
                          torch.stack([E[..., a1], E[..., a2]]).cpu().numpy(),
                          torch.stack([H[..., a1], H[..., a2]]).cpu().numpy()))
    return faces


def _ringdowns(case, seed):
    """Windows and tails of decaying port signals: a few damped modes each,
    scaled to the window's peak as the training pairs are."""
    rng = np.random.default_rng(seed)
    B, L, T = case["batch"], case["samples"], case["tail"]
    t = np.arange(L + T)
    m = 5
    f, a = rng.uniform(0.005, 0.15, (B, m, 1)), rng.uniform(0.002, 0.03, (B, m, 1))
    x = np.empty((B, 2, L + T))
    for c in range(2):
        w = rng.standard_normal((B, m, 1)) * np.exp(-a * t) * np.cos(2 * np.pi * f * t + rng.uniform(0, 6.28, (B, m, 1)))
        x[:, c] = w.sum(1)
    x /= np.abs(x[..., :L]).max(-1, keepdims=True)
    return x[..., :L].astype(np.float32), x[..., L:].astype(np.float32)


def _dims(case):
    from openems_amd.extrapolator import ExtrapolatorDims

    return ExtrapolatorDims(L0=case["samples"], batch=case["batch"], tail=case["tail"])


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "grid":
        from openems_amd import EngineBatch, ScheduledExcitation

        s = _scene(case, seed)
        op, eng, x = _build(s)
        pulse = _pulse(s, op.dt, case["steps"])
        batch = EngineBatch(num_steps=case["steps"], extensions=list(x.values()), sample_interval=100, track_peak=True,
                            excitations=[ScheduledExcitation((i, j, k), 2, (a * pulse).astype(np.float32))
                                         for i, j, k, a in s["sources"]])
        return {"case": case, "op": op, "eng": eng, "x": x, "batch": batch}
    if kind == "sweep":
        from openems_amd import ScheduledExcitation, Sweep

        sweep, engines, ports, cpmls = Sweep(), [], [], []
        for s in _sweep_scenes(case, seed):
            op, eng, x = _build(s)
            pulse = _pulse(s, op.dt, case["steps"])
            sweep.add(eng, x["cpml"], x["port"],
                      [ScheduledExcitation((i, j, k), 2, (a * pulse).astype(np.float32)) for i, j, k, a in s["sources"]])
            engines.append(eng)
            ports.append(x["port"])
            cpmls.append(x["cpml"])
        return {"case": case, "sweep": sweep, "engines": engines, "ports": ports, "cpmls": cpmls}
    if kind == "farfield":
        from openems_amd import Nf2ff

        nf = Nf2ff(case["freq"])
        for f in _surfaces(case, seed):
            nf.add_surface(*f)
        return {"case": case, "nf": nf, "angles": _angles(case["thetas"], case["phis"])}
    from openems_amd.extrapolator import Extrapolator

    x, target = _ringdowns(case, seed)
    return {"case": case, "net": Extrapolator(_dims(case), seed=int(seed) & 0xFFFF), "x": x, "target": target}


def _sweep_scenes(case, seed):
    rng = np.random.default_rng(seed)
    for q in range(case["structures"]):
        c = {"nx": int(rng.integers(60, 221)), "ny": int(rng.integers(60, 121)),
             "nz": int(rng.integers(30, 49) + 3) // 4 * 4, "delta": 5e-4, "scene": "microstrip", "absorber": "cpml",
             "mode": "physical", "boxes": 0}
        yield _scene(c, 1000003 * int(seed) + q)


# ---------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "grid":
        eng, x = state["eng"], state["x"]
        eng.reset()
        for e in x.values():
            e.reset()
        res = eng.run_batch(state["batch"])
        out = {"energy": res.energy_samples}
        if "port" in x:
            out["spectra"] = x["port"].dft_values()
            out["s11"] = x["port"].s11(50.0)
        else:
            out["probe"] = x["probe"].data()
            out["E"], out["H"] = eng.read_fields()
        if "box" in x:
            angles = _angles(*BOX_ANGLES)
            for q in range(len(BOX_FREQS)):
                far = x["box"].far_field(q, *angles)
                out["far%d" % q] = [far.e_theta, far.e_phi, far.prad]
        return out
    if kind == "sweep":
        for e in state["engines"] + state["ports"] + state["cpmls"]:
            e.reset()
        res = state["sweep"].run(case["steps"])
        return {"energy": np.array([r.final_energy for r in res]), "steps": np.array([r.timesteps_executed for r in res]),
                "spectra": np.stack([p.dft_values() for p in state["ports"]])}
    if kind == "farfield":
        far = state["nf"].calculate(*state["angles"])
        return [far.e_theta, far.e_phi, far.prad, far.dmax]
    net = state["net"]
    if kind == "infer":
        modes, tails = net.forward(state["x"], tails=case["tails"])
        return [modes, tails] if case["tails"] else [modes]
    if case["update"]:
        return [net.train_step(state["x"], state["target"], 1e-3), net.params()]
    return list(net.gradients(state["x"], state["target"]))


# --------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind == "grid":
        return _steps_work((case["nx"], case["ny"], case["nz"]), case["steps"], case["absorber"].startswith("cpml"),
                           case["scene"] != "empty")
    if kind == "sweep":  # the mean structure of the range
        one = _steps_work((140, 90, 40), case["steps"], True, True)
        return {k: v * case["structures"] for k, v in one.items()}
    if kind == "farfield":
        n = (case["n1"], case["n2"], case["n3"])
        nodes = 2 * (n[0] * n[1] + n[1] * n[2] + n[0] * n[2])
        theta, phi = _angles(case["thetas"], case["phis"])
        angles = theta.size * phi.size
        kap = [np.outer(np.sin(theta), np.cos(phi)), np.outer(np.sin(theta), np.sin(phi)),
               np.outer(np.cos(theta), np.ones(phi.size))]
        distinct = [np.unique(np.round(np.abs(v), 12)).size for v in kap]
        flops = 0.0
        for ax in range(3):  # one contraction per distinct cosine, one sum per angle
            p, q = sorted(((ax + 1) % 3, (ax + 2) % 3), key=lambda a: distinct[a])
            flops += 2 * (2.0 * 2 * distinct[p] * 8 * n[q] * n[p] + 8.0 * 4 * angles * n[q] / 4)
        return {"bytes": nodes * 64.0 + angles * 32.0, "flops": flops}
    B, L, T = case["batch"], case["samples"], case["tail"]
    conv = [(L // 2, 2 * 9, 64), (L // 4, 64 * 9, 128), (L // 8, 128 * 9, 128)]
    mac = sum(r * k * c for r, k, c in conv) + (L // 8 * 128) * 384 + 384 * 192
    weights = sum(k * c + c for _, k, c in conv) + (L // 8 * 128) * 384 + 384 + 384 * 192 + 192
    if kind == "infer":
        return {"bytes": 4.0 * (B * 2 * L + weights + B * 192 + (B * 2 * T if case["tails"] else 0)),
                "flops": 2.0 * B * mac + (B * T * 32 * 10.0 if case["tails"] else 0)}
    return {"bytes": 4.0 * (B * 2 * (L + T) + 2 * weights * (3 if case["update"] else 1)),
            "flops": 6.0 * B * mac + B * T * 32 * 30.0}


def _steps_work(n, steps, cpml, boxes):
    """Six field components read and written per cell and step, one byte of
    material, the CPML state of eight layers on each side of each axis."""
    cells = n[0] * n[1] * n[2]
    slab = sum(cells // m * min(16, m - 1) for m in n) if cpml else 0
    return {"bytes": steps * (cells * (49.0 if boxes else 48.0) + slab * 32.0),
            "flops": steps * (cells * 36.0 + slab * 24.0)}


# -------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        cells = case["nx"] * case["ny"] * case["nz"]
        if cells * case["steps"] > 1.4e10:
            return None
        return _exact_grid(_scene(case, seed), case["steps"])
    if kind == "sweep":
        if case["structures"] * case["steps"] > 14000:
            return None
        outs = [_exact_grid(s, case["steps"], check=100) for s in _sweep_scenes(case, seed)]
        return {"energy": np.array([o["energy"][-1][1] + o["energy"][-1][2] for o in outs]), "steps": None,
                "spectra": np.stack([o["spectra"] for o in outs])}
    if kind == "farfield":
        theta, phi = _angles(case["thetas"], case["phis"])
        return list(_exact_far(_surfaces(case, seed), case["freq"], theta, phi))
    return _exact_net(case, seed)


def _exact_grid(s, steps, check=100):
    """The scene stepped in float64: the leapfrog of the curl equations with
    the scene's media, absorbers, dispersive cells and sources."""
    dev, n, d = "cuda", s["n"], s["delta"]
    dt = 0.99 * d / (C0 * math.sqrt(3.0))
    full = lambda v: torch.full(n, v, dtype=torch.float64, device=dev)  # noqa: E731
    eps, sig, pec = full(1.0), full(0.0), torch.zeros(n, dtype=torch.bool, device=dev)
    cells = {"drude": [], "lorentz": []}
    media = list(s["materials"])
    for kind, c, r in s["spheres"]:
        p = _sphere_cells(c, r)
        cells[kind].append(p)
        if kind == "lorentz":
            i, j, k = (torch.tensor(v, device=dev) for v in p.T)
            eps[i, j, k] = LORENTZ_EPS
    for e, g, (i0, i1, j0, j1, k0, k1) in media:
        at = (slice(i0, i1), slice(j0, j1), slice(k0, k1))
        pec[at] = e is None
        if e is not None:
            eps[at], sig[at] = e, g
    loss = sig * dt / (2 * eps * EPS0)
    ca = torch.where(pec, 0.0, (1 - loss) / (1 + loss))
    cb = torch.where(pec, 0.0, dt / (eps * EPS0) / (1 + loss) / d)
    Ca, Cb = [ca, ca, ca], [cb, cb, cb]
    if s["port"]:  # the resistor on the port's z edges
        i0, i1, j0, j1, k0, k1 = s["port"]
        at = (slice(i0, i1), slice(j0, j1), slice(k0, k1))
        extra = d / (50.0 * (i1 - i0) * (j1 - j0) / (k1 - k0) * d * d)
        lz = (sig[at] + extra) * dt / (2 * eps[at] * EPS0)
        Ca[2], Cb[2] = ca.clone(), cb.clone()
        Ca[2][at] = torch.where(pec[at], 0.0, (1 - lz) / (1 + lz))
        Cb[2][at] = torch.where(pec[at], 0.0, dt / (eps[at] * EPS0) / (1 + lz) / d)
    del eps, sig, pec, loss
    db = -dt / (MU0 * d)
    E = [full(0.0) for _ in range(3)]
    H = [full(0.0) for _ in range(3)]
    inner = tuple(slice(1, None) for _ in range(3))

    # CPML: per face the slab and the two recursions' coefficients
    faces = []
    if s["cpml"] and s["mode"] == "physical":
        top = max(s["cpml"])
        smax = -4.0 * math.log(1e-6) / (2 * Z0 * top * d)
        for f, L in enumerate(s["cpml"]):
            ax, low = f // 2, f % 2 == 0
            if not 0 < L < n[ax]:
                continue
            i = np.arange(L)
            de = (L - i if low else i + 1).astype(np.float64)
            shape = [1, 1, 1]
            shape[ax] = L
            size = list(n)
            size[ax] = L
            at = [slice(None)] * 3
            at[ax] = slice(0, L) if low else slice(n[ax] - L, n[ax])
            tabs = []
            for depth in (de, de - 0.5):
                sg = smax * np.clip(depth / L, 0, 1) ** 3
                b = np.exp(-sg / EPS0 * dt)
                a = np.where(sg / EPS0 > 1e-20, 1 - b, 0.0)
                tabs.append([torch.tensor(v.reshape(shape), device=dev) for v in (b, a)])
            psi = [[torch.zeros(size, dtype=torch.float64, device=dev) for _ in range(2)] for _ in range(2)]
            faces.append((ax, tuple(at), tabs, psi))

    def half(h):
        """One half-step: the curls, the media, the CPML terms."""
        F = E if h else H          # the field whose differences are taken
        D = {}
        for c in range(3):
            for ax in range(3):
                if ax == c:
                    continue
                v = torch.zeros(n, dtype=torch.float64, device=dev)
                lo = [slice(None)] * 3
                hi = [slice(None)] * 3
                lo[ax], hi[ax] = slice(0, -1), slice(1, None)
                torch.sub(F[c][tuple(hi)], F[c][tuple(lo)], out=v[tuple(lo if h else hi)])
                D[c, ax] = v
        for c in range(3):
            a1, a2 = (c + 1) % 3, (c + 2) % 3
            curl = D[a2, a1] - D[a1, a2]
            if h:
                H[c].add_(curl, alpha=db)
            else:
                E[c][inner] = Ca[c][inner] * E[c][inner] + Cb[c][inner] * curl[inner]
        for ax, at, tabs, psi in faces:
            a1, a2 = (ax + 1) % 3, (ax + 2) % 3
            b, a = tabs[1 if h else 0]
            # the difference of component a2 along ax drives component a1, and the other way round
            for q, (drive, into, sign) in enumerate(((a2, a1, 1.0), (a1, a2, -1.0))):
                p = psi[1 if h else 0][q]
                p.mul_(b).addcmul_(a.expand_as(p), D[drive, ax][at])
                if h:
                    H[into][at].add_(p, alpha=sign * db)
                else:
                    add = sign * Cb[into][at] * p
                    for z in range(3):  # index-0 planes are not written
                        if at[z].start in (0, None):
                            cut = [slice(None)] * 3
                            cut[z] = slice(0, 1)
                            add[tuple(cut)] = 0.0
                    E[into][at].add_(add)

    # dispersive cells
    ade = []
    for kind in ("drude", "lorentz"):
        if cells[kind]:
            i, j, k = (torch.tensor(v, device=dev) for v in np.concatenate(cells[kind]).T)
            zero = torch.zeros(3, i.numel(), dtype=torch.float64, device=dev)
            ade.append([kind, (i, j, k), torch.stack([Cb[c][i, j, k] for c in range(3)]) * d, zero, zero.clone()])
    # Mur faces in list order: (component, line, shift) along each axis
    mur = []
    for f, on in enumerate(s["mur"] or ()):
        if on:
            ax = f // 2
            line, shift = [slice(None)] * 3, [slice(None)] * 3
            line[ax], shift[ax] = (n[ax] - 1, n[ax] - 2) if f % 2 else (0, 1)
            mur.append(((ax + 1) % 3, (ax + 2) % 3, tuple(line), tuple(shift)))
    cm = (C0 * dt - d) / (C0 * dt + d)
    pulse = torch.tensor(_pulse(s, dt, steps), device=dev)
    amps = [(i, j, k, a) for i, j, k, a in s["sources"]]
    freqs = torch.tensor(FREQS, dtype=torch.float64, device=dev)
    spectra = torch.zeros(len(FREQS), 2, dtype=torch.complex128, device=dev)
    probe = torch.zeros(steps, 6, dtype=torch.float64, device=dev)
    energy = []
    nodes = _box_nodes(s, dev) if s["box"] else None
    for st in range(steps):
        half(True)
        before = [[E[a][sh] - cm * E[a][ln] for a in (p, q)] for p, q, ln, sh in mur]
        old = [torch.stack([E[c][at] for c in range(3)]) for _, at, *_ in ade]
        half(False)
        for rec, en in zip(ade, old):
            kind, at, K, J, P = rec
            e = torch.stack([E[c][at] for c in range(3)])
            if kind == "drude":
                den = 1 + DRUDE[1] * dt / 2
                kj, bj = (1 - DRUDE[1] * dt / 2) / den, EPS0 * DRUDE[0] ** 2 * dt / 2 / den
                new = (e - K / 2 * ((1 + kj) * J + bj * en)) / (1 + K * bj / 2)
                rec[3] = kj * J + bj * (new + en)
            else:
                w0, g, de = LORENTZ
                den = 1 + g * dt / 2
                nxt = ((2 - (w0 * dt) ** 2) * J + (g * dt / 2 - 1) * P + EPS0 * de * (w0 * dt) ** 2 * en) / den
                new = e - K * (nxt - J) / dt
                rec[3], rec[4] = nxt, J
            for c in range(3):
                E[c][at] = new[c]
        for v, (p, q, ln, sh) in zip(before, mur):
            v[0] += cm * E[p][sh]
            v[1] += cm * E[q][sh]
        for v, (p, q, ln, sh) in zip(before, mur):
            E[p][ln] = v[0]
            E[q][ln] = v[1]
        for i, j, k, a in amps:
            E[2][i, j, k] += a * pulse[st]
        if s["port"]:
            i0, _, j0, _, k0, k1 = s["port"]
            mid = k0 + (k1 - k0) // 2
            u = d * E[2][i0, j0, k0:k1].sum() * -1
            cur = d * (H[1][i0, j0, mid] - H[1][i0 - 1, j0, mid] - H[0][i0, j0, mid] + H[0][i0, j0 - 1, mid])
            spectra[:, 0] += u * torch.exp(-2j * math.pi * freqs * ((st + 1) * dt))
            spectra[:, 1] += cur * torch.exp(-2j * math.pi * freqs * ((st + 0.5) * dt))
        else:
            probe[st] = torch.stack([F[c][s["probe"]] for F in (E, H) for c in range(3)])
        if nodes is not None and st % 4 == 0:
            for ax, sign, pos, c1, c2, acc, take in nodes:
                e, h = take(E, H)
                for q, f in enumerate(BOX_FREQS):
                    w = 2 * math.pi * f
                    acc[q][0] += e * complex(math.cos(w * (st + 1) * dt), -math.sin(w * (st + 1) * dt))
                    acc[q][1] += h * complex(math.cos(w * (st + 0.5) * dt), -math.sin(w * (st + 0.5) * dt))
        if st % check == 0:
            energy.append((float(st), float(sum((v * v).sum() for v in E)), float(sum((v * v).sum() for v in H))))
    out = {"energy": np.array(energy)}
    if s["port"]:
        spectra *= 2 * dt
        out["spectra"] = spectra.cpu().numpy()
        inc = 0.5 * (spectra[:, 0] + 50.0 * spectra[:, 1])
        out["s11"] = ((spectra[:, 0] - inc) / inc).cpu().numpy()
    else:
        out["probe"] = probe.cpu().numpy()
        out["E"] = torch.stack(E).cpu().numpy()
        out["H"] = torch.stack(H).cpu().numpy()
    if nodes is not None:
        theta, phi = _angles(*BOX_ANGLES)
        for q, f in enumerate(BOX_FREQS):
            far = _exact_far([(ax, sign, pos, c1, c2, 8 * dt * acc[q][0], 8 * dt * acc[q][1])
                              for ax, sign, pos, c1, c2, acc, _ in nodes], f, theta, phi)
            out["far%d" % q] = list(far[:3])
    return out


def _box_nodes(s, dev):
    """Per face of the recording box: its sums and a function that takes the
    tangential fields at its nodes (E from the two edges that meet there, H
    from the four faces around it)."""
    lo, hi, d = s["box"][0::2], s["box"][1::2], s["delta"]
    out = []
    for ax in range(3):
        a1, a2 = (ax + 1) % 3, (ax + 2) % 3
        for side in (0, 1):
            at = hi[ax] if side else lo[ax]

            def pick(v, back, ax=ax, a1=a1, a2=a2, at=at):
                ix = [None] * 3
                ix[ax] = at - back[ax]
                for a in (a1, a2):
                    ix[a] = slice(lo[a] - back[a], hi[a] + 1 - back[a])
                w = v[tuple(ix)]
                return w if a1 < a2 else w.transpose(0, 1)

            def take(E, H, ax=ax, a1=a1, a2=a2, pick=pick):
                unit = lambda *a: [1 if q in a else 0 for q in range(3)]  # noqa: E731
                e = torch.stack([0.5 * (pick(E[c], unit(c)) + pick(E[c], unit())) for c in (a1, a2)])
                h = torch.stack([0.25 * (pick(H[c], unit(ax, o)) + pick(H[c], unit(ax)) + pick(H[c], unit(o))
                                         + pick(H[c], unit())) for c, o in ((a1, a2), (a2, a1))])
                return e, h

            shape = (2, hi[a1] - lo[a1] + 1, hi[a2] - lo[a2] + 1)
            acc = [[torch.zeros(shape, dtype=torch.complex128, device=dev) for _ in range(2)] for _ in BOX_FREQS]
            out.append((ax, 1 if side else -1, at * d, np.arange(lo[a1], hi[a1] + 1) * d,
                        np.arange(lo[a2], hi[a2] + 1) * d, acc, take))
    return out


def _exact_far(faces, freq, theta, phi):
    """Radiation integrals of the equivalent surface currents at 1 m."""
    dev = "cuda"
    k = 2 * math.pi * freq / C0
    th, ph = (v.reshape(-1) for v in np.meshgrid(theta, phi, indexing="ij"))
    kap = [torch.tensor(v, device=dev) for v in (np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th))]
    N = torch.zeros(3, th.size, dtype=torch.complex128, device=dev)
    M = torch.zeros_like(N)
    prad = 0.0

    def weights(c):
        w = np.zeros(len(c))
        w[:-1] += np.diff(c) / 2
        w[1:] += np.diff(c) / 2
        return torch.tensor(w, dtype=torch.complex128, device=dev)

    for ax, sign, pos, c1, c2, e, h in faces:
        a1, a2 = (ax + 1) % 3, (ax + 2) % 3
        e, h = (torch.as_tensor(v, device=dev) for v in (e, h))
        w1, w2 = weights(c1), weights(c2)
        cur = torch.stack([-sign * h[1], sign * h[0], sign * e[1], -sign * e[0]]) * w1[:, None] * w2
        prad += 0.5 * sign * float(((e[0] * h[1].conj() - e[1] * h[0].conj()) * w1[:, None] * w2).sum().real)
        x1, x2 = torch.tensor(c1, device=dev), torch.tensor(c2, device=dev)
        right = cur.permute(1, 0, 2).reshape(len(c1), -1).contiguous()
        for b in range(0, th.size, 4096):
            at = slice(b, min(b + 4096, th.size))
            p1 = torch.exp(1j * k * kap[a1][at, None] * x1)
            p2 = torch.exp(1j * k * kap[a2][at, None] * x2)
            v = ((p1 @ right).reshape(-1, 4, len(c2)) * p2[:, None]).sum(-1) * torch.exp(1j * k * kap[ax][at] * pos)[:, None]
            N[a1, at] += v[:, 0]
            N[a2, at] += v[:, 1]
            M[a1, at] += v[:, 2]
            M[a2, at] += v[:, 3]
    st, ct, sp, cp = (torch.tensor(f(v), device=dev) for v in (th, ph) for f in (np.sin, np.cos))
    along_t = lambda v: v[0] * ct * cp + v[1] * ct * sp - v[2] * st  # noqa: E731
    along_p = lambda v: -v[0] * sp + v[1] * cp                       # noqa: E731
    fac = 1j * k * np.exp(-1j * k) / (4 * math.pi)
    et = -fac * (along_p(M) + Z0 * along_t(N))
    ep = fac * (along_t(M) - Z0 * along_p(N))
    shape = (len(theta), len(phi))
    top = float(((et.abs() ** 2 + ep.abs() ** 2) / (2 * Z0)).max())
    return et.reshape(shape).cpu().numpy(), ep.reshape(shape).cpu().numpy(), prad, 4 * math.pi * top / prad if prad > 0 else 0.0


def _exact_net(case, seed):
    """The network in float64 from the weights the program starts with."""
    from openems_amd.extrapolator import Extrapolator, unpack

    dims, dev = _dims(case), "cuda"
    flat = Extrapolator(dims, seed=int(seed) & 0xFFFF).params()
    w = {q: torch.tensor(v, dtype=torch.float64, device=dev).requires_grad_() for q, v in unpack(flat, dims).items()}
    x, target = (torch.tensor(v, dtype=torch.float64, device=dev) for v in _ringdowns(case, seed))
    gelu = lambda v: 0.5 * v * (1 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))  # noqa: E731

    def conv(v, weight, bias):  # kernel 9, stride 2, 4 zeros before the first sample
        rows = torch.nn.functional.pad(v, (4, 4)).unfold(2, 9, 2)[:, :, :v.shape[2] // 2]
        flat_rows = rows.permute(0, 2, 1, 3).reshape(-1, weight.shape[1] * 9)
        return (flat_rows @ weight.reshape(weight.shape[0], -1).t() + bias).reshape(v.shape[0], -1, weight.shape[0]).transpose(1, 2)

    v = x
    for q in "123":
        v = gelu(conv(v, w["W" + q], w["b" + q]))
    v = gelu(v.transpose(1, 2).reshape(v.shape[0], -1) @ w["W4"].t() + w["b4"])
    modes = v @ w["W5"].t() + w["b5"]
    p = modes.reshape(-1, dims.modes, 6, 1)
    t = torch.arange(case["tail"], dtype=torch.float64, device=dev)
    size = torch.exp(-0.05 * torch.nn.functional.softplus(p[:, :, 0]) * t)
    angle = 2 * math.pi * 0.5 * torch.sigmoid(p[:, :, 1]) * t
    zr, zi = size * torch.cos(angle), size * torch.sin(angle)
    tails = torch.stack([(p[:, :, 2 + 2 * c] * zr - p[:, :, 3 + 2 * c] * zi).sum(1) for c in range(2)], 1)
    if case["kind"] == "infer":
        out = [modes, tails] if case["tails"] else [modes]
        return [v.detach().cpu().numpy() for v in out]
    loss = ((tails - target) ** 2).mean()
    loss.backward()
    order = ["W1", "b1", "W2", "b2", "W3", "b3", "W4", "b4", "W5", "b5"]
    g = torch.cat([w[q].grad.reshape(-1) for q in order])
    if case["update"]:  # the first Adam step
        new = torch.cat([w[q].detach().reshape(-1) for q in order]) - 1e-3 * g / (g.abs() + 1e-8)
        return [float(loss), new.cpu().numpy()]
    return [float(loss), g.cpu().numpy()]
