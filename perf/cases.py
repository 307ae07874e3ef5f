"""The time-stepping work that users of this package run, as cases that can be timed and checked one by one.

One pass of a stepping case is one DFT chunk (``dft_stride`` time steps and one sample of every monitor) through
the runner that the drivers use (``Engine.make_runner`` / ``Batch.make_runner`` with graphs), resumed mid-run:
the fields hold a pulse in flight over the whole grid. One pass of an adjoint case is a forward run and the
gradient of a mode-power objective through ``monitor_spectra`` / ``batched_monitor_spectra``.

Kinds:
  box      one real grid with a CPML on every face, dielectric spheres, optional D-form (Drude-Lorentz) nodes,
           a point dipole and a DFT plane, at the launch tiling the solve-level drivers choose
  sphere   the plain gold sphere of the scattering path: conformal vertex tensor, table-fed plane wave, flux boxes
  bloch    one oblique run over a periodic metasurface cell: complex64 fields, Bloch plane source
  sweep    several such runs (normal incidence among them: real fields, 1D-fed plane wave) as one Batch
  adjoint  dL/drho of one waveguide scene, stored tape
  designs  the same for several uneven scenes with a silver cube each, batched, checkpoint recompute

``exact`` restates the update in float64 torch: Yee curls, CPML, pure D-form poles, Bloch ghosts, dipole, mode and
Bloch plane sources, DFT monitors; gradients by torch autograd through the restated steps.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from lightsmith_amd.fdtd import (DFTMonitor, DispersiveGroup, Engine, Medium, PMLSpec, PointDipole, Pole,
                                 workloads)
from lightsmith_amd.fdtd.adjoint import BatchedAdjoint, batched_monitor_spectra, monitor_spectra
from lightsmith_amd.fdtd.batch import Batch
from lightsmith_amd.fdtd.engine import filling_tiling

DEV = "cuda:0"
DX = 2.0  # nm, the cell of the box cases
DT = 0.95 * DX / math.sqrt(3.0)
HBARC = 197.3269804  # eV nm
# gold (Drude + 2 Lorentz) and one ultraviolet pole: (sigma, omega0, gamma) in 1/nm^2, 1/nm, 1/nm; eps_inf 1.53
_POLES_EV = [(8.55 ** 2, 0.0, 0.0735), (0.94 * 2.88 ** 2, 2.88, 0.74), (1.36 * 3.90 ** 2, 3.90, 1.25),
             (0.60 * 8.00 ** 2, 8.00, 2.50)]
EPS_INF = 1.53


# --- the cases ------------------------------------------------------------------------------------------

def listed():
    return [
        # the smallest calls: a quick look at a nanoantenna on a tiny grid, bound by launches and latency
        _box("box_tiny", 40, 36, 32, pml=6, poles=3, disp="scattered", stride=10),
        # an ordinary particle solve: gold sphere in water, 97^3 nodes, 81-wavelength flux boxes, vertex tensor
        {"name": "sphere_gold", "kind": "sphere", "radius": 40.0, "dx": 2.0, "num": 81},
        # a smoothed (subpixel) dielectric scene on a ragged grid: dense coefficients, kappa-graded CPML
        _box("box_dense_ragged", 131, 117, 150, pml=12, poles=0, disp="none", stride=50, dense=True, kappa=3.0),
        # a metal body (one Drude pole) in a medium-sized grid
        _box("box_drude_body", 192, 160, 128, pml=10, poles=1, disp="body", stride=50),
        # a long waveguide-like domain of smoothed dielectric
        _box("box_wide", 514, 96, 80, pml=12, poles=0, disp="none", stride=50, dense=True),
        # a large ragged grid with a two-pole metal body and staircase dielectrics
        _box("box_large_ragged", 255, 257, 250, pml=12, poles=2, disp="body", stride=50),
        # the throughput configuration: 320^3, 10 % three-pole nodes scattered over the interior
        _box("box_throughput", 320, 320, 320, pml=16, poles=3, disp="scattered", stride=50),
        # one oblique run of a metasurface sweep stepped alone
        {"name": "bloch_cell", "kind": "bloch", "lo": 58, "hi": 78, "nz": 256, "angles": 3, "stride": 33, "cells": 5},
        # a metasurface sweep: 12 uneven cells, 3 of them at normal incidence, stepped as one batch
        {"name": "sweep_12", "kind": "sweep", "n": 12, "lo": 48, "hi": 96, "nz": 256, "angles": 4, "stride": 33,
         "cells": 2},
        # inverse design of a waveguide element: forward and gradient with the stored tape
        {"name": "adjoint_waveguide", "kind": "adjoint", "nx": 256, "ny": 192, "nz": 96, "design": 80, "pml": 16,
         "steps": 800},
        # several designs at once, each with a silver cube, checkpoint recompute
        {"name": "designs_4", "kind": "designs", "n": 4, "steps": 300, "cells": 6},
    ]


def _box(name, nx, ny, nz, pml, poles, disp, stride, dense=False, kappa=1.0):
    return {"name": name, "kind": "box", "nx": nx, "ny": ny, "nz": nz, "pml": pml, "poles": poles, "disp": disp,
            "dense": dense, "kappa": kappa, "stride": stride}


def draw(rng: random.Random):
    kind = rng.choice(["box"] * 6 + ["bloch", "sweep", "adjoint", "sphere"])
    if kind == "box":
        cells = math.exp(rng.uniform(math.log(4e4), math.log(2.4e7)))
        f = [math.exp(rng.uniform(-0.4, 0.4)) for _ in range(3)]
        s = (cells / (f[0] * f[1] * f[2])) ** (1 / 3)
        n = [max(30, int(round(s * v))) + rng.randint(0, 3) for v in f]
        poles = rng.choice([0, 0, 1, 2, 3, 4])
        pml = rng.randint(6, max(6, min(16, min(n) // 5)))
        return {"kind": "box", "nx": n[0], "ny": n[1], "nz": n[2], "pml": pml, "poles": poles,
                "disp": "none" if poles == 0 else rng.choice(["scattered", "body"]), "dense": rng.random() < 0.5,
                "kappa": rng.choice([1.0, 3.0]), "stride": rng.randint(10, 60)}
    if kind == "bloch":
        lo = rng.randint(34, 90)
        return {"kind": "bloch", "lo": lo, "hi": lo + rng.randint(0, 20), "nz": rng.randint(200, 300),
                "angles": rng.randint(2, 6), "stride": rng.randint(20, 50), "cells": rng.randint(0, 999)}
    if kind == "sweep":
        lo = rng.randint(40, 70)
        return {"kind": "sweep", "n": rng.randint(3, 12), "lo": lo, "hi": lo + rng.randint(1, 26),
                "nz": rng.randint(200, 260), "angles": rng.randint(2, 4), "stride": rng.randint(20, 40),
                "cells": rng.randint(0, 999)}
    if kind == "adjoint":
        return {"kind": "adjoint", "nx": rng.randint(110, 240), "ny": rng.randint(96, 180), "nz": rng.randint(72, 100),
                "design": rng.randint(20, 30), "pml": rng.randint(8, 14), "steps": 25 * rng.randint(20, 32)}
    return {"kind": "sphere", "radius": float(rng.randint(20, 60)), "dx": rng.choice([2.0, 2.5, 3.0]),
            "num": rng.randint(21, 81)}


# --- inputs shared by prepare() and exact() -------------------------------------------------------------

def _medium(poles):
    return EPS_INF, [(s / HBARC ** 2, w / HBARC, g / HBARC) for s, w, g in _POLES_EV[:poles]]


def _flat(c, i, j, k, shape):
    return ((np.asarray(c) * shape[0] + i) * shape[1] + j) * shape[2] + k


def _plane(shape, pml, kz):
    """(e, h1, h2) reference indices of E_x, E_y and the face-averaged H_y, H_x on node plane kz."""
    i, j = (a.ravel() for a in np.meshgrid(np.arange(pml, shape[0] - pml), np.arange(pml, shape[1] - pml),
                                           indexing="ij"))
    e = np.concatenate([_flat(0, i, j, kz, shape), _flat(1, i, j, kz, shape)])
    h1 = np.concatenate([_flat(1, i, j, kz - 1, shape), _flat(0, i, j, kz - 1, shape)])
    h2 = np.concatenate([_flat(1, i, j, kz, shape), _flat(0, i, j, kz, shape)])
    return e, h1, h2


def _box_inputs(case, seed):
    """Permittivity, D-form nodes, dipole and monitor of a box case (host arrays, as a user's program has them)."""
    shape = (case["nx"], case["ny"], case["nz"])
    pml, rng = case["pml"], np.random.default_rng(seed)
    small = min(shape)
    inv = np.ones((3,) + shape)
    r_hi = max(3.0, small / 16)
    for _ in range(200 if small >= 250 else 40):
        r = rng.uniform(max(1.5, r_hi / 5), r_hi)
        ctr = np.array([rng.uniform(pml + r, n - 1 - pml - r) if n - 1 - 2 * pml > 2 * r else n / 2 for n in shape])
        e = rng.uniform(1.5, 12.0)
        lo = np.maximum(np.floor(ctr - r - 1).astype(int), 0)
        hi = np.minimum(np.ceil(ctr + r + 2).astype(int), shape)
        for c in range(3):
            ax = [np.arange(lo[a], hi[a]) + (0.5 if a == c else 0.0) - ctr[a] for a in range(3)]
            d = np.sqrt(ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2)
            sub = inv[c, lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]]
            if case["dense"]:  # volume-averaged at the surface
                f = np.clip(r - d + 0.5, 0.0, 1.0)
                np.copyto(sub, 1.0 / (1.0 + f * (e - 1.0)), where=f > 0)
            else:
                np.copyto(sub, 1.0 / e, where=d <= r)
    idx = np.zeros(0, np.int64)
    if case["disp"] == "scattered":  # 10 % of the cells inside the CPML, all three components
        inner = tuple(n - 2 * pml for n in shape)
        cells = np.flatnonzero(rng.random(inner, dtype=np.float32) < 0.1)
        i, j, k = np.unravel_index(cells, inner)
        cell = ((i + pml) * shape[1] + j + pml) * shape[2] + k + pml
        idx = np.concatenate([c * int(np.prod(shape)) + cell for c in range(3)])
    elif case["disp"] == "body":  # a metal sphere in the middle
        r = 0.5 * (small - 2 * pml) * 0.7
        for c in range(3):
            ax = [np.arange(n) + (0.5 if a == c else 0.0) - n / 2 for a, n in enumerate(shape)]
            inside = ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2 <= r * r
            idx = np.concatenate([idx, c * inside.size + np.flatnonzero(inside)])
    inv.reshape(-1)[idx] = 1.0
    omega_c = 2 * np.pi / 120.0
    pos = np.array([n * DX * f for n, f in zip(shape, (0.3, 0.55, 0.5))]) + 0.3
    return {"shape": shape, "inv_eps": inv, "idx": idx, "pos": pos,
            "omega_c": omega_c, "omega_half": 0.15 * omega_c, "omega": 2 * np.pi / np.linspace(90.0, 160.0, 16),
            "plane": _plane(shape, pml, shape[2] // 2 + max(1, shape[2] // 10))}


def _pulse(shape, seed, periodic=(False, False, False), bloch=None, spacing=(1.0, 1.0, 1.0)):
    """(E, H) float32 / complex64 tensors (3, n0, n1, n2) of a smooth field over the whole grid: a few standing
    waves per component, falling to zero towards non-periodic faces, (Bloch-)periodic along periodic axes."""
    rng = np.random.default_rng([seed, 77])
    cx = bloch is not None
    out = []
    for _ in range(2):
        comps = []
        for _c in range(3):
            acc = 0.0
            for _m in range(3):
                fac = []
                for a in range(3):
                    n = shape[a]
                    x = np.arange(n, dtype=float)
                    if periodic[a]:
                        m = int(rng.integers(0, 4))
                        v = np.cos(2 * np.pi * m * (x - 1) / (n - 2) + rng.uniform(0, 6.28)) + 0j
                        if cx:
                            v = v * np.exp(1j * bloch[a] * (x - 1) * spacing[a])
                        v[[0, -1]] = 0.0
                    else:
                        v = np.sin(2 * np.pi * x / rng.uniform(9.0, 40.0) + rng.uniform(0, 6.28)) \
                            * np.sin(np.pi * x / (n - 1)) ** 2 + 0j
                        v[[0, -1]] = 0.0
                    v = v * (rng.standard_normal() + (1j * rng.standard_normal() if cx else 0.0) if a == 0 else 1.0)
                    fac.append(torch.as_tensor(v if cx else v.real, device=DEV))
                acc = acc + fac[0][:, None, None] * fac[1][None, :, None] * fac[2][None, None, :]
            comps.append(acc.to(torch.complex64 if cx else torch.float32))
        out.append(torch.stack(comps))
    return out


def _run_scene(case, seed):
    """The runs of a bloch or sweep case: cell sizes from the case, pillar pattern from the seed."""
    n = case["n"] if case["kind"] == "sweep" else 2
    runs = workloads.oblique_sweep_scene(n_inst=n, nz=case["nz"], size_lo=case["lo"], size_hi=case["hi"],
                                         seed=case["cells"], pattern_seed=seed, n_angles=case["angles"],
                                         n_wl=1)
    return runs if case["kind"] == "sweep" else runs[1:]


def _design_scenes(case, seed):
    """Adjoint scenes with a pulse short enough to cross the design region within the run; rho from the seed."""
    if case["kind"] == "adjoint":
        d = case["design"]
        scenes = [workloads.adjoint_scene(shape=(case["nx"], case["ny"], case["nz"]), design=(d, d, 11),
                                          pml=case["pml"], n_steps=case["steps"])]
    else:
        scenes = workloads.batched_adjoint_scenes(n_inst=case["n"], seed=case["cells"], n_steps=case["steps"])
    rng = np.random.default_rng([seed, 5])
    for sc in scenes:
        t = (np.arange(case["steps"] + 2) + 0.5) * sc["dt"]
        w, tau, t0 = float(sc["omega"][0]), 24 * sc["dt"], 70 * sc["dt"]
        sc["t_src"] = (np.exp(-((t - t0) / tau) ** 2) * np.cos(w * (t - t0)))[:, None]
        sc["rho"] = rng.uniform(0.0, 1.0, size=sc["rho"].shape)
        if case["kind"] == "designs":  # watch the plane just behind the design region: a 300-step run reaches it
            n0, n1, _ = sc["shape"]
            back = (n0 - case_pml(case) - 14) - (sc["hi"][0] + 2)
            src = sc["lo"][0] - 6 - (case_pml(case) + 14)
            step = n1 * sc["shape"][2]
            for key in ("e_mon", "h1", "h2"):
                sc[key] = sc[key] - back * step
            sc["e_src"] = sc["e_src"] + src * step
    return scenes


def case_pml(case):
    return case.get("pml", 12)


# --- prepare and run ------------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "box":
        b = _box_inputs(case, seed)
        eps_inf, poles = _medium(case["poles"])
        med = Medium(eps_inf, tuple(Pole(*p) for p in poles))
        groups = [DispersiveGroup(idx=b["idx"], media=[med], frac=np.ones((1, len(b["idx"]))), w=None)] \
            if len(b["idx"]) else []
        src = PointDipole(shape=b["shape"], origin=np.zeros(3), dx=DX, dt=DT, pos=b["pos"], pdir=(0.0, 0.0, 1.0),
                          inv_eps=b["inv_eps"], omega_c=b["omega_c"], omega_half=b["omega_half"], max_steps=20000)
        mon = DFTMonitor(b["omega"], *b["plane"], energy=1)
        pml = PMLSpec(cells=((case["pml"],) * 2,) * 3, kappa_max=case["kappa"], alpha_max=0.002, eps_ref=1.0)
        eng = Engine(DEV, shape=b["shape"], dx=DX, dt=DT, single=True, inv_eps=b["inv_eps"], groups=groups, pml=pml,
                     sources=[src], monitors=[mon], dft_stride=case["stride"])
        eng.set_tiling(*filling_tiling([eng.shape]))
        _fill(eng, _pulse(b["shape"], seed))
        return {"run": eng.make_runner(True)[0], "engines": [eng]}
    if kind == "sphere":
        _, _, scene = workloads.au_sphere_scene(DEV, num_wavelengths=case["num"], spacing_nm=case["dx"]) \
            if case["radius"] == 40.0 else _other_sphere(case)
        eng = scene.engine(DEV)
        _fill(eng, _pulse(eng.shape, seed))
        return {"run": eng.make_runner(True)[0], "engines": [eng]}
    if kind in ("bloch", "sweep"):
        engines = []
        for q, r in enumerate(_run_scene(case, seed)):
            eng = workloads.oblique_engine(r, DEV, max_steps=20000, stride=case["stride"])
            eng.set_tiling(*filling_tiling([eng.shape]))
            _fill(eng, _pulse(eng.shape, seed + 1000 * q, eng.periodic, eng.bloch if eng.complex else None, eng.spacing))
            engines.append(eng)
        if kind == "bloch":
            return {"run": engines[0].make_runner(True)[0], "engines": engines}
        batch = Batch(engines, schedule=filling_tiling([e.shape for e in engines]) + (0,))
        return {"run": batch.make_runner(True)[0], "engines": engines, "batch": batch}
    scenes = _design_scenes(case, seed)
    probs = [workloads.adjoint_problem(sc, DEV, **({} if kind == "adjoint" else {"tape_budget": 0})) for sc in scenes]
    state = {"probs": probs, "rho": [torch.as_tensor(sc["rho"], device=DEV) for sc in scenes],
             "w": [torch.as_tensor(sc["w"], device=DEV) for sc in scenes]}
    if kind == "designs":
        state["batch"] = BatchedAdjoint(probs)
    return state


def _other_sphere(case):
    """The gold sphere scene at another radius."""
    from lightsmith_amd.fdtd import scattering
    from lightsmith_amd.problem import FDTDOptions, Sphere, options_for
    sim = workloads.au_sphere_sim(num_wavelengths=case["num"], spacing_nm=case["dx"])
    sim.particles[0].shape = Sphere(radius_nm=case["radius"])
    opts = FDTDOptions.model_validate(options_for(sim, "lightsmith-fdtd", "fdtd"))
    return sim, opts, scattering.setup(sim, opts, DEV)


def _fill(eng, fields):
    eng.E.copy_(fields[0])
    eng.H.copy_(fields[1])


def run(state):
    if "probs" in state:
        rhos = [r.detach().clone().requires_grad_(True) for r in state["rho"]]
        accs = batched_monitor_spectra(rhos, state["batch"]) if "batch" in state else \
            [monitor_spectra(rhos[0], state["probs"][0])]
        loss = sum(workloads.mode_power(a[0], w) for a, w in zip(accs, state["w"]))
        loss.backward()
        return [{"acc_e": a[0].detach(), "acc_h": a[1].detach(), "grad": r.grad} for a, r in zip(accs, rhos)]
    state["run"]()
    return [{"E": e.E, "H": e.H, "acc_e": e.monitors[0].acc_e, "acc_h": e.monitors[0].acc_h, "energy": e.energy}
            for e in state["engines"]]


# --- work ---------------------------------------------------------------------------------------------------

def _grid_work(shape, s, mat, psi_axes, pml, n_ade, poles):
    """(bytes, flops) of one time step: E and H read and written once, coefficients, CPML psi (two components and
    both fields per axis) and pole pairs read and written."""
    N = int(np.prod(shape))
    psi = sum(2 * 2 * 2 * pml * (N // shape[a]) for a in psi_axes)
    return N * (12 * s + mat) + psi * 2 * s + n_ade * 2 * poles * 2 * s, \
        (N * 36.0 + psi * 5.0 + n_ade * poles * 8.0) * (2 if s == 8 else 1)


def work(case):
    kind = case["kind"]
    if kind == "box":
        shape = (case["nx"], case["ny"], case["nz"])
        inner = [n - 2 * case["pml"] for n in shape]
        n_ade = {"none": 0.0, "scattered": 0.3 * inner[0] * inner[1] * inner[2],
                 "body": 4 * math.pi * (0.35 * min(inner)) ** 3}[case["disp"]]
        b, f = _grid_work(shape, 4, 12 if case["dense"] else 4, (0, 1, 2), case["pml"], n_ade, case["poles"])
        pts = 2 * inner[0] * inner[1]
        return {"bytes": b * case["stride"] + pts * 2 * 16 * 16.0, "flops": f * case["stride"] + pts * 2 * 16 * 8.0}
    if kind == "sphere":
        n = 2 * (math.ceil(case["radius"] / case["dx"]) + 1 + 2 * max(4, math.ceil(12.0 / case["dx"])) + 15) + 1
        steps = 107 * 2.0 / case["dx"]
        n_ade = 4 * math.pi * (case["radius"] / case["dx"]) ** 3
        b, f = _grid_work((n, n, n), 4, 4, (0, 1, 2), 12, n_ade, 3)
        pts = 2 * 12 * (n - 54) ** 2
        return {"bytes": b * steps + pts * 2 * 16.0 * case["num"], "flops": f * steps + pts * 8.0 * case["num"]}
    if kind in ("bloch", "sweep"):
        rng = np.random.default_rng(case["cells"])
        n = case["n"] if kind == "sweep" else 2
        sizes = [rng.integers(case["lo"], case["hi"] + 1, size=2) for _ in range(n)]
        tot = [0.0, 0.0]
        for q, (a, b) in enumerate(sizes):
            if kind == "bloch" and q == 0:
                continue
            real = q % case["angles"] == 0
            w = _grid_work((int(a) + 2, int(b) + 2, case["nz"]), 4 if real else 8, 4, (2,), 16, 0, 0)
            tot = [tot[0] + w[0] * case["stride"], tot[1] + w[1] * case["stride"]]
        return {"bytes": tot[0], "flops": tot[1]}
    if kind == "adjoint":
        shapes, d, pml = [(case["nx"], case["ny"], case["nz"])], case["design"], case["pml"]
        runs = 2
    else:
        rng, shapes, d, pml, runs = np.random.default_rng(case["cells"]), [], 40, 12, 3
        for _ in range(case["n"]):
            shapes.append((int(rng.integers(128, 257)), int(rng.integers(96, 193)), int(rng.integers(64, 97))))
            rng.integers(1 << 30)
    tot = [0.0, 0.0]
    for sh in shapes:
        b, f = _grid_work(sh, 4, 12, (0, 1, 2), pml, 0, 0)
        tape = 2 * 4 * 3 * d * d * 11
        tot = [tot[0] + (runs * b + tape) * case["steps"], tot[1] + runs * f * case["steps"]]
    return {"bytes": tot[0], "flops": tot[1]}


# --- the same in float64 --------------------------------------------------------------------------------

def _cpml(cells, shape, spacing, dt, a, half, kappa, alpha, eps_ref, eps_high):
    """(b, c, 1/kappa) per node along axis a for E (half = 0) or H (half = 0.5): cubic grading, CFS alpha."""
    lo, hi = cells[a]
    n, h = shape[a], spacing[a]
    u = np.arange(n) + half
    r_lo = np.clip((lo - u) / lo, 0, 1) if lo else np.zeros(n)
    r_hi = np.clip((u - (n - 1 - hi)) / hi, 0, 1) if hi else np.zeros(n)
    rho = np.maximum(r_lo, r_hi)
    smax = np.where(r_lo >= r_hi, 3.2 / (math.sqrt(eps_ref) * h), 3.2 / (math.sqrt(eps_high or eps_ref) * h))
    sig, kap, alp = smax * rho ** 3, 1 + (kappa - 1) * rho ** 3, alpha * (1 - rho) * (rho > 0)
    b = np.exp(-(sig / kap + alp) * dt)
    den = sig * kap + kap ** 2 * alp
    c = np.where(sig > 0, sig * (b - 1) / np.where(den > 0, den, 1), 0.0)
    inside = (u <= lo) | (u >= n - 2 - hi + half) if (lo or hi) else np.zeros(n, bool)
    return np.where(inside, b, 1.0), np.where(inside, c, 0.0), np.where(inside, 1 / kap, 1.0)


class _Exact:
    """One grid in float64 (complex128 under a Bloch phase), reference layout (3, n0, n1, n2)."""

    def __init__(self, shape, spacing, dt, inv_eps, cells, kappa, alpha, eps_ref, eps_high=None, bloch=None,
                 periodic=(False, False, False), idx=None, eps_inf=1.0, poles=()):
        self.shape, self.dt, self.per = shape, dt, periodic
        self.s = [1.0 / d for d in spacing]
        self.dtype = torch.complex128 if bloch is not None else torch.float64
        self.ph = [complex(np.exp(1j * bloch[a] * (shape[a] - 2) * spacing[a])) if bloch is not None else 1.0
                   for a in range(3)]
        self.mask = []
        for h in range(2):
            per_c = []
            for c in range(3):
                m = torch.ones(shape, dtype=torch.float64, device=DEV)
                for a in range(3):
                    v = np.ones(shape[a])
                    if periodic[a]:
                        v[[0, -1]] = 0
                    elif h == 0:
                        v[-1] = 0
                        if a != c:
                            v[0] = 0
                    elif a != c:
                        v[-1] = 0
                    m = m * self._along(v, a)
                per_c.append(m)
            self.mask.append(per_c)
        self.set_inv_eps(torch.as_tensor(inv_eps, device=DEV, dtype=torch.float64))
        self.prof = {}
        for h in range(2):
            for a in range(3):
                if any(cells[a]):
                    b, c, ik = _cpml(cells, shape, spacing, dt, a, 0.5 * h, kappa, alpha, eps_ref, eps_high)
                    self.prof[h, a] = (self._along(b, a), self._along(c, a),
                                       self._along(ik, a) if kappa > 1 else None)
        self.idx = torch.as_tensor(idx, device=DEV) if idx is not None and len(idx) else None
        self.eps_inf = eps_inf
        self.coef = []
        for s, w0, g in poles:
            den = 1 + g * dt / 2
            self.coef.append(((2 - w0 ** 2 * dt ** 2) / den, -(1 - g * dt / 2) / den, s * dt ** 2 / den))

    def set_inv_eps(self, inv):
        self.cb = [self.dt * inv[c] * self.mask[0][c] for c in range(3)]

    def _along(self, v, a):
        return torch.as_tensor(v, device=DEV, dtype=torch.float64).reshape([-1 if q == a else 1 for q in range(3)])

    def start(self, E=None, H=None):
        z = lambda: torch.zeros((3,) + tuple(self.shape), dtype=self.dtype, device=DEV)  # noqa: E731
        st = {"E": z() if E is None else E.to(self.dtype), "H": z() if H is None else H.to(self.dtype)}
        for h, a in self.prof:
            for c in range(3):
                if c != a:
                    st["psi", h, a, c] = torch.zeros(self.shape, dtype=self.dtype, device=DEV)
        if self.idx is not None:
            for p in range(len(self.coef)):
                st["P", p] = torch.zeros(len(self.idx), dtype=self.dtype, device=DEV)
                st["Q", p] = torch.zeros(len(self.idx), dtype=self.dtype, device=DEV)
        return st

    def _diff(self, F, a, fwd):
        n = self.shape[a]
        if self.per[a]:
            F = torch.cat([F.narrow(a, 0, n - 1), F.narrow(a, 1, 1) * self.ph[a]], a) if fwd else \
                torch.cat([F.narrow(a, n - 2, 1) * np.conj(self.ph[a]), F.narrow(a, 1, n - 1)], a)
        d = (F.narrow(a, 1, n - 1) - F.narrow(a, 0, n - 1)) * self.s[a]
        z = torch.zeros_like(F.narrow(a, 0, 1))
        return torch.cat([d, z] if fwd else [z, d], a)

    def _curl(self, st, F, h, c):
        """Component c of curl F with its CPML terms; F = E for the H update (h = 1), H for the E update."""
        d1, d2 = (c + 1) % 3, (c + 2) % 3
        out = 0.0
        for a, g, sign in ((d1, d2, 1.0), (d2, d1, -1.0)):
            d = self._diff(F[g], a, h == 1)
            if (h, a) in self.prof:
                b, cc, ik = self.prof[h, a]
                psi = st["psi", h, a, c] = b * st["psi", h, a, c] + cc * d
                d = (d if ik is None else d * ik) + psi
            out = out + sign * d
        return out

    def half_h(self, st):
        st["H"] = torch.stack([st["H"][c] - self.dt * self.mask[1][c] * self._curl(st, st["E"], 1, c)
                               for c in range(3)])

    def half_e(self, st):
        dE = torch.stack([self.cb[c] * self._curl(st, st["H"], 0, c) for c in range(3)])
        if self.idx is not None:
            flat = dE.reshape(-1)
            eo, dp = st["E"].reshape(-1)[self.idx], 0.0
            for p, (c1, c2, c3) in enumerate(self.coef):
                pn = c1 * st["P", p] + c2 * st["Q", p] + c3 * eo
                dp = dp + (pn - st["P", p])
                st["Q", p], st["P", p] = st["P", p], pn
            dE = flat.index_copy(0, self.idx, (flat[self.idx] - dp) / self.eps_inf).reshape(dE.shape)
        st["E"] = st["E"] + dE

    @staticmethod
    def add(F, idx, v):
        return F.reshape(-1).index_add(0, idx, v.to(F.dtype)).reshape(F.shape)


class _Dft:
    def __init__(self, omega, e, h1, h2):
        self.om = torch.as_tensor(np.asarray(omega, float), device=DEV)
        self.i = [torch.as_tensor(v, device=DEV) for v in (e, h1, h2)]
        self.e = self.h = 0.0

    def sample(self, st, n, dt):
        E, H = st["E"].reshape(-1)[self.i[0]], 0.5 * (st["H"].reshape(-1)[self.i[1]] + st["H"].reshape(-1)[self.i[2]])
        self.e = self.e + torch.exp(1j * self.om * n * dt)[:, None] * E[None, :]
        self.h = self.h + torch.exp(1j * self.om * (n - 0.5) * dt)[:, None] * H[None, :]
        self.energy = float(E.abs().square().sum() + H.abs().square().sum())


def _ghosts(F, shape, per):
    """Ghost planes are not part of the stored state: they stay as the state holds them (zero)."""
    for a in range(3):
        if per[a]:
            F.narrow(a + 1, 0, 1).zero_()
            F.narrow(a + 1, shape[a] - 1, 1).zero_()
    return F


def exact(case, seed):
    kind = case["kind"]
    if kind == "sphere":  # its vertex tensor and source tables are this package's own set-up: no value beside it
        return None
    if kind == "box":
        return [_exact_box(case, seed)]
    if kind in ("bloch", "sweep"):
        return [None if r["theta"] == 0.0 else _exact_bloch(case, r, seed + 1000 * q)
                for q, r in enumerate(_run_scene(case, seed))]
    return [_exact_gradient(sc, case) for sc in _design_scenes(case, seed)]


def _exact_box(case, seed):
    b = _box_inputs(case, seed)
    eps_inf, poles = _medium(case["poles"])
    shape, p = b["shape"], case["pml"]
    ref = _Exact(shape, (DX,) * 3, DT, b["inv_eps"], ((p, p),) * 3, case["kappa"], 0.002, 1.0, idx=b["idx"],
                 eps_inf=eps_inf, poles=poles)
    f = b["pos"] / DX - np.array([0.0, 0.0, 0.5])
    base = np.floor(f).astype(int)
    idx, wt = [], []
    hit = set(b["idx"][np.isin(b["idx"], [int(_flat(2, *(base + np.array([(q >> a) & 1 for a in range(3)])), shape))
                                            for q in range(8)])].tolist())
    for q in range(8):
        bits = np.array([(q >> a) & 1 for a in range(3)])
        i = int(_flat(2, *(base + bits), shape))
        idx.append(i)
        wt.append(float(np.prod(np.where(bits, f - base, 1 - (f - base)))) * b["inv_eps"].reshape(-1)[i] /
                  (eps_inf if i in hit else 1.0))
    idx, wt = torch.as_tensor(idx, device=DEV), torch.as_tensor(wt, device=DEV, dtype=torch.float64)
    tau = 2.0 / b["omega_half"]
    t = np.arange(case["stride"] + 1) * DT - 5.0 * tau
    wave = np.diff(np.exp(-(t / tau) ** 2) * np.sin(b["omega_c"] * t)) / (b["omega_c"] * DT)
    st = ref.start(*_pulse(shape, seed))
    for n in range(case["stride"]):
        ref.half_h(st)
        ref.half_e(st)
        st["E"] = ref.add(st["E"], idx, -DT * wt * wave[n])
    d = _Dft(b["omega"], *b["plane"])
    d.sample(st, case["stride"], DT)
    return {"E": st["E"], "H": st["H"], "acc_e": d.e, "acc_h": d.h, "energy": np.array([d.energy, 0.0])}


def _exact_bloch(case, r, seed):
    """One oblique run: the cell and the column (one real cell in x and y) that feeds its plane source."""
    shape, d, dt = r["shape"], r["spacing"], r["dt"]
    per, bloch = (True, True, False), (r["kpar"][0], r["kpar"][1], 0.0)
    cells = ((0, 0), (0, 0), (r["pml"], r["pml"]))
    alpha = 0.05 * 2 * np.pi / r["wavelength"]
    ref = _Exact(shape, d, dt, r["inv_eps"], cells, 1.0, alpha, 1.0, r["eps_sub"], bloch, per)
    cs = (3, 3, shape[2])
    col = _Exact(cs, d, dt, np.ones((3,) + cs), cells, 1.0, alpha, 1.0, None, bloch, per)
    K = np.array([2 * np.sin(r["kpar"][a] * d[a] / 2) / d[a] for a in (0, 1)])
    u = K / np.linalg.norm(K)
    a = np.array([-u[1], u[0]]) if r["pol"] == "s" else u
    amp = [complex(a[q] * np.exp(0.5j * r["kpar"][q] * d[q])) for q in (0, 1)]
    i, j = np.meshgrid(np.arange(1, shape[0] - 1), np.arange(1, shape[1] - 1), indexing="ij")
    ph = torch.as_tensor(np.exp(1j * (bloch[0] * (i - 1) * d[0] + bloch[1] * (j - 1) * d[1])), device=DEV)
    tau = 2.0 / r["omega_half"]
    k = r["k_src"]
    inner = (slice(1, shape[0] - 1), slice(1, shape[1] - 1))
    st = ref.start(*_pulse(shape, seed, per, bloch, d))
    sc = col.start()
    for n in range(case["stride"]):
        ref.half_h(st)
        H = st["H"].clone()
        H[(0,) + inner + (k - 1,)] -= dt / d[2] * ph * sc["E"][1, 1, 1, k]
        H[(1,) + inner + (k - 1,)] += dt / d[2] * ph * sc["E"][0, 1, 1, k]
        st["H"] = H
        col.half_h(sc)
        ref.half_e(st)
        E = st["E"].clone()
        E[(0,) + inner + (k,)] += dt / d[2] * ph * sc["H"][1, 1, 1, k - 1]
        E[(1,) + inner + (k,)] -= dt / d[2] * ph * sc["H"][0, 1, 1, k - 1]
        st["E"] = E
        col.half_e(sc)
        t = (n + 1) * dt - 3.5 * tau
        w = math.exp(-(t / tau) ** 2) * math.sin(r["omega"] * t)
        for q in (0, 1):
            sc["E"][q, 1, 1, k - 1] += amp[q] * w
    nx, ny = r["n_cells"]
    gi, gj = (v.ravel() for v in np.meshgrid(np.arange(1, nx + 1), np.arange(1, ny + 1), indexing="ij"))
    dfts = []
    for kz in (r["k_r"], r["k_t"]):  # the transmission plane's energy joins the reflection plane's
        pts = [np.concatenate([_flat(c, gi, gj, q, shape) for c in cc]) for cc, q in
               (((0, 1), kz), ((1, 0), kz - 1), ((1, 0), kz))]
        dfts.append(_Dft([r["omega"]], *pts))
        dfts[-1].sample(st, case["stride"], dt)
    return {"E": _ghosts(st["E"], shape, per), "H": _ghosts(st["H"], shape, per), "acc_e": dfts[0].e,
            "acc_h": dfts[0].h, "energy": np.array([dfts[0].energy + dfts[1].energy, 0.0])}


def _exact_gradient(sc, case):
    """Spectra and dL/drho of one scene by torch autograd through the float64 steps, segment by segment."""
    from torch.utils.checkpoint import checkpoint
    shape, p = sc["shape"], case_pml(case)
    groups = sc.get("groups", ())
    idx = groups[0].idx if groups else None
    med = groups[0].media[0] if groups else None
    ref = _Exact(shape, (sc["dx"],) * 3, sc["dt"], sc["inv_eps"], ((p, p),) * 3, 1.0, 0.05 * float(sc["omega"][0]),
                 sc["eps_lo"], idx=idx, eps_inf=med.eps_inf if med else 1.0,
                 poles=[(q.sigma, q.omega0, q.gamma) for q in med.poles] if med else ())
    rho = torch.as_tensor(sc["rho"], device=DEV).requires_grad_(True)
    box = tuple(slice(l, h) for l, h in zip(sc["lo"], sc["hi"]))
    inv = torch.as_tensor(sc["inv_eps"], device=DEV)
    flat = torch.arange(int(np.prod(shape)), device=DEV).reshape(shape)[box].reshape(-1)
    one = 1.0 / (sc["eps_lo"] + rho.reshape(-1) * (sc["eps_hi"] - sc["eps_lo"]))
    ref.set_inv_eps([inv[c].reshape(-1).index_copy(0, flat, one).reshape(shape) for c in range(3)])
    src, m = torch.as_tensor(sc["e_src"], device=DEV), torch.as_tensor(sc["m_src"][:, 0], device=DEV)
    om = float(sc["omega"][0])
    mon = [torch.as_tensor(sc[q], device=DEV) for q in ("e_mon", "h1", "h2")]
    st = ref.start()
    keys = sorted(st, key=str)
    ne = len(sc["e_mon"])
    acc = [torch.zeros(ne, dtype=torch.complex128, device=DEV) for _ in range(2)]

    def segment(n0, n1, cb0, cb1, cb2, ae, ah, *vals):
        ref.cb = [cb0, cb1, cb2]
        s = dict(zip(keys, vals))
        for n in range(n0, n1):
            ref.half_h(s)
            ref.half_e(s)
            s["E"] = ref.add(s["E"], src, m * float(sc["t_src"][n, 0]))
        e = s["E"].reshape(-1)[mon[0]]
        h = 0.5 * (s["H"].reshape(-1)[mon[1]] + s["H"].reshape(-1)[mon[2]])
        ae = ae + complex(np.exp(1j * om * n1 * sc["dt"])) * e
        ah = ah + complex(np.exp(1j * om * (n1 - 0.5) * sc["dt"])) * h
        return (ae, ah) + tuple(s[q] for q in keys)

    vals, cb = tuple(st[q] for q in keys), list(ref.cb)
    for n0 in range(0, case["steps"], sc["stride"]):
        out = checkpoint(segment, n0, n0 + sc["stride"], *cb, *acc, *vals, use_reentrant=False)
        acc, vals = out[:2], out[2:]
    loss = (torch.as_tensor(sc["w"], device=DEV) * acc[0]).sum().abs() ** 2
    loss.backward()
    return {"acc_e": acc[0].detach()[None], "acc_h": acc[1].detach()[None], "grad": rho.grad}
