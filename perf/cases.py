"""Timed cases of the framework's public entry points (gi_amd).

What a user of this framework has it do, at the sizes it is used at:

force       one drop-in force evaluation (gi_force_collision) of an impact,
            the call that replaces the reference's force kernel in its own
            step loop; from a couple of thousand particles to the roofline
            impact of 262,144
steps       a short run of the native stepper (gi_impact_steps) from an
            initial state: force, move and their launches as a loop sees them
separate    the generator's settling steps (gi_separate_steps): two bodies
            that do not interact, damped
ensemble    the batched engine (Ensemble.steps) on impacts of uneven size, the
            parameter sweep and the mix that the request loop keeps resident
recenter    the reference's float recentring (gi_recenter_float)
earth_moon  the final analysis (gi_find_earth_moon) with its group table

States are seeded impacts on jittered lattices (make_impact).  "hot" adds
thermal velocities, so that contact pairs both approach and recede, as they do
once the bodies have met; "debris" throws that share of the silicate outwards
to many body radii, as it is late in a run.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "giant-impact_amd"))

import gi_amd as gi  # noqa: E402

DEV = "cuda"
MASS_FE = 7.850 / 3.320  # iron element over silicate element (equal volumes)


def listed() -> list:
    return [
        # The small configuration of the plain method: 1,536 + 512 particles,
        # one call of the reference's loop.
        dict(name="force_2k", kind="force", n=2048, frac=0.25, hot=0.0, debris=0.0),
        # An impact of the parameter sweep run alone, odd size, bodies in motion.
        dict(name="force_13k", kind="force", n=13255, frac=0.22, hot=1.5, debris=0.0),
        # The mid-size impact late in its run: hot, with debris far out.
        dict(name="force_65k", kind="force", n=65536, frac=0.2, hot=1.5, debris=0.05),
        # The roofline impact, as bench.py times it.
        dict(name="force_262k", kind="force", n=262144, frac=0.25, hot=0.0, debris=0.0),
        # The stepper on the small configuration: bound by launches.
        dict(name="steps_2k", kind="steps", n=2048, frac=0.25, hot=0.0, debris=0.0, steps=16),
        # The stepper at an odd size in the middle of the sweep's range.
        dict(name="steps_21k", kind="steps", n=21001, frac=0.15, hot=0.0, debris=0.0, steps=8),
        # Settling two bodies of a mid-size system.
        dict(name="separate_30k", kind="separate", n=30000, frac=0.3, hot=0.0, debris=0.0, steps=8),
        # The 64-simulation sweep: N uniform in [4,096, 32,768].
        dict(name="ensemble_64", kind="ensemble", sims=64, n_min=4096, n_max=32768, log=False, steps=1),
        # What the request loop keeps resident: N log-uniform in [2,048, 65,536].
        dict(name="ensemble_mix", kind="ensemble", sims=8, n_min=2048, n_max=65536, log=True, steps=2),
        # The recentring that the loop makes every RecenterRate steps.
        dict(name="recenter_65k", kind="recenter", n=65536, frac=0.2, hot=1.5, debris=0.0),
        # The final analysis of a mid-size run.
        dict(name="earth_moon_65k", kind="earth_moon", n=65536, frac=0.2, hot=1.5, debris=0.15),
    ]


def _log_int(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["force", "force", "force", "steps", "steps", "separate", "ensemble", "ensemble", "recenter",
                       "earth_moon"])
    frac = round(rng.uniform(0.1, 0.3), 3)
    hot = rng.choice([0.0, 0.5, 1.5])
    debris = rng.choice([0.0, 0.0, 0.02, 0.1])
    if kind == "force":
        return dict(kind=kind, n=_log_int(rng, 1024, 262144), frac=frac, hot=hot, debris=debris)
    if kind == "steps":
        return dict(kind=kind, n=_log_int(rng, 1024, 65536), frac=frac, hot=0.0, debris=0.0,
                    steps=rng.choice([1, 4, 8, 12]))
    if kind == "separate":
        return dict(kind=kind, n=_log_int(rng, 1024, 65536), frac=frac, hot=0.0, debris=0.0,
                    steps=rng.choice([1, 8, 12]))
    if kind == "ensemble":
        log = rng.random() < 0.5
        return dict(kind=kind, sims=_log_int(rng, 2, 48), n_min=2048 if log else 4096, n_max=rng.choice([16384, 32768]),
                    log=log, steps=rng.choice([1, 2]))
    return dict(kind=kind, n=_log_int(rng, 2048, 131072), frac=frac, hot=hot,
                debris=0.15 if kind == "earth_moon" else debris)


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------


def _impact(case, seed):
    """A seeded impact as host arrays: (pos, vel, fc, mc, info)."""
    ni = max(1, int(round(case["frac"] * case["n"])))
    rng = np.random.default_rng([seed, case["n"]])
    pos, vel, fc, mc, info = gi.make_impact(
        case["n"] - ni, ni, seed=1 + seed % (1 << 31), angle_deg=float(rng.uniform(30.0, 60.0)),
        speed_vesc=float(rng.uniform(1.0, 1.4)), target_spin=float(rng.uniform(0.0, 0.6)))
    n = len(pos)
    if case["hot"] > 0.0:
        vel[:, :3] += rng.normal(0.0, case["hot"], (n, 3)).astype(np.float32)
    if case["debris"] > 0.0:
        out = fc.NFe + np.flatnonzero(rng.random(n - fc.NFe) < case["debris"])
        r = np.linalg.norm(pos[out, :3], axis=1, keepdims=True)
        u = rng.normal(size=(len(out), 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        far = np.exp(rng.uniform(math.log(2.5), math.log(15.0), (len(out), 1))) * max(float(r.max()), 1.0)
        pos[out, :3] = (u * far).astype(np.float32)
        vel[out, :3] += (u * rng.uniform(0.0, 10.0, (len(out), 1))).astype(np.float32)
    return pos, vel, fc, mc, info


def _bodies(case, seed):
    """The same bodies as the generator settles them: order [Fe1, Si1, Fe2,
    Si2], bodies apart, and the generator's constants with their borders."""
    pos, vel, _, _, info = _impact(case, seed)
    f1, f2, s1 = info.nfe1, info.nfe2, info.nsi1
    order = np.r_[0:f1, f1 + f2:f1 + f2 + s1, f1:f1 + f2, f1 + f2 + s1:len(pos)]
    fc, mc = gi.separate_constants(gi.units(gi.generator_setup_defaults(len(pos))))
    for c in (fc, mc):
        c.boarder1, c.boarder2, c.boarder3 = f1, f1 + s1, f1 + s1 + f2
    return pos[order], vel[order], fc, mc


def _ensemble(case, seed):
    """The sweep's sizes belong to the case, its impacts to the seed."""
    cfg = _sizes(case)
    for k, c in enumerate(cfg):
        rng = np.random.default_rng([seed, k])
        c.update(seed=1 + (seed * 1000 + k) % (1 << 40), angle_deg=float(rng.uniform(30.0, 60.0)),
                 speed_vesc=float(rng.uniform(1.0, 1.4)), target_spin=float(rng.uniform(0.0, 0.6)))
    return gi.make_ensemble(cfg)


def _sizes(case):
    return gi.ensemble_configs(case["sims"], n_range=(case["n_min"], case["n_max"]), log_uniform_n=case["log"])


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


class _Buffer(gi.DeviceArray):
    """A torch tensor of float4 records where the bindings take a DeviceArray."""

    def __init__(self, t):
        self.tensor, self.n, self.nbytes, self.ptr = t, len(t), 16 * len(t), C.c_void_p(t.data_ptr())

    def close(self):
        self.ptr = C.c_void_p()


def prepare(case, seed):
    s = {"kind": case["kind"], "steps": case.get("steps", 0)}
    if case["kind"] == "ensemble":
        pos, vel, n, fc, mc, _ = _ensemble(case, seed)
        s["pos0"], s["vel0"] = _gpu(pos), _gpu(vel)
        s["pos"], s["vel"] = s["pos0"].clone(), s["vel0"].clone()
        s["buffers"] = _Buffer(s["pos"]), _Buffer(s["vel"])
        torch.cuda.synchronize()
        s["ensemble"] = gi.Ensemble(*s["buffers"], n, fc, mc)
        return s
    if case["kind"] == "separate":
        pos, vel, s["fc"], s["mc"] = _bodies(case, seed)
    else:
        pos, vel, s["fc"], s["mc"], s["info"] = _impact(case, seed)
    s["n"] = len(pos)
    s["pos0"], s["vel0"] = _gpu(pos), _gpu(vel)
    s["pos"], s["vel"] = s["pos0"].clone(), s["vel0"].clone()
    s["force"] = torch.zeros_like(s["pos"])
    if case["kind"] == "recenter":
        rng = np.random.default_rng([seed, 7])
        s["com"], s["mean"] = rng.uniform(-1.0, 1.0, 3).tolist(), rng.uniform(-0.1, 0.1, 3).tolist()
    return s


def run(s):
    kind = s["kind"]
    if kind == "force":
        gi.force_collision(s["pos"].data_ptr(), s["vel"].data_ptr(), s["force"].data_ptr(), s["n"], s["fc"])
        return {"force": s["force"]}
    if kind == "earth_moon":
        i = s["info"]
        r = gi.find_earth_moon(s["pos"].data_ptr(), s["vel"].data_ptr(), s["n"], i.nfe1, i.nfe2, i.nsi1, MASS_FE,
                               with_groups=True)
        return r
    # a job starts from its initial state
    s["pos"].copy_(s["pos0"])
    s["vel"].copy_(s["vel0"])
    out = {"pos": s["pos"], "vel": s["vel"]}
    if kind == "ensemble":
        s["ensemble"].steps(s["steps"])
        return out
    P, V, F = s["pos"].data_ptr(), s["vel"].data_ptr(), s["force"].data_ptr()
    if kind == "steps":
        gi.impact_steps(P, V, F, s["n"], s["fc"], s["mc"], s["steps"])
    elif kind == "separate":
        gi.call("gi_separate_steps", P, V, F, s["n"], C.byref(s["fc"]), C.byref(s["mc"]), 8.0, 8.0, s["steps"], None)
    else:
        gi.recenter_float(P, V, s["n"], s["fc"].NFe, MASS_FE, 1.0, s["com"], s["mean"])
    return out


# ---------------------------------------------------------------------------
# Work: each unordered pair's gravity once (20 operations), each particle's
# records read and written once
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        n = np.array([c["n_target"] + c["n_impactor"] for c in _sizes(case)], dtype=np.float64)
        return {"bytes": case["steps"] * 64.0 * n.sum(), "flops": case["steps"] * 10.0 * float((n * n).sum())}
    n = float(case["n"])
    if kind == "force":
        return {"bytes": 48.0 * n, "flops": 10.0 * n * n}
    if kind == "steps":
        return {"bytes": case["steps"] * 64.0 * n, "flops": case["steps"] * 10.0 * n * n}
    if kind == "separate":
        a, b = (1.0 - case["frac"]) * n, case["frac"] * n
        return {"bytes": case["steps"] * 64.0 * n, "flops": case["steps"] * 10.0 * (a * a + b * b)}
    if kind == "recenter":
        return {"bytes": 96.0 * n, "flops": 30.0 * n}
    return {"bytes": 36.0 * n, "flops": 200.0 * n}


# ---------------------------------------------------------------------------
# 64 bits
# ---------------------------------------------------------------------------


def _force64(x, v, nfe, L):
    """The force of one simulation in FP64 from positions and velocities in
    FP64.  Whether a pair is in contact, which shell it is in and whether it
    recedes are decisions of the law on float values: they are taken on the
    values rounded to float, in the law's own operation order."""
    n = len(x)
    xf, vf = x.float(), v.float()
    fe = torch.arange(n, device=x.device) < nfe
    f = torch.zeros_like(x)
    step = max(1, min(n, (1 << 26) // n))
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [x[None, :, k] - x[a:b, None, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        df = [xf[None, :, k] - xf[a:b, None, k] for k in range(3)]
        near = (df[0] * df[0] + df[1] * df[1] + df[2] * df[2]).sqrt() < 1.0
        both = fe[a:b, None].to(torch.uint8) + fe[None, :].to(torch.uint8)
        g = torch.tensor([1.0, L.GMassFeSi, L.GMassFeFe], dtype=torch.float64, device=x.device)
        w = g[both.long()] * r2.clamp_min(1e-300).pow(-1.5)
        w[near] = 0.0
        for k in range(3):
            f[a:b, k] += (w * d[k]).sum(1)
        i, j = near.nonzero(as_tuple=True)
        i, j = i[i + a != j], j[i + a != j]
        i = i + a
        p, pf, u = x[j] - x[i], xf[j] - xf[i], vf[j] - vf[i]
        q = pf[:, 0] * pf[:, 0] + pf[:, 1] * pf[:, 1] + pf[:, 2] * pf[:, 2]
        rf = q.sqrt()
        away = (pf[:, 0] * u[:, 0] + pf[:, 1] * u[:, 1] + pf[:, 2] * u[:, 2]) >= 1.0
        t = fe[i].long() + fe[j].long()
        outer = torch.tensor([L.ShellBreakSi, L.ShellBreakFeSi1, L.ShellBreakFe], device=x.device)[t] <= rf
        mixed = (t == 1) & (L.ShellBreakFeSi2 <= rf)
        K = torch.tensor([L.KSiSi, L.KFeSi, L.KFeFe], dtype=torch.float64, device=x.device)[t]
        KR = torch.tensor([L.KRSiSi, L.KRFeSi, L.KRFeFe], dtype=torch.float64, device=x.device)[t]
        KR = torch.where(mixed, torch.full_like(KR, L.KRMix), KR)
        K = torch.where(outer | ~away, K, KR)
        r = p.norm(dim=1)
        f.index_add_(0, i, ((g[t] - K * (1.0 - r * r)) / r)[:, None] * p)
    return f


def _steps64(pos, vel, nfe, law, dt, dtm, damp, steps, parts):
    """Positions and velocities after `steps` steps; parts: the ranges that
    interact, each with its iron first."""
    x, v = pos[:, :3].double(), vel[:, :3].double()
    f = torch.zeros_like(x)
    for _ in range(steps):
        for (a, b), k in zip(parts, nfe):
            f[a:b] = _force64(x[a:b], v[a:b], k, law)
        v = v + (f - damp * v) * dtm[:, None]
        x = x + v * dt
    return x, v


def _full(xyz, like):
    return torch.cat([xyz, like[:, 3:].double()], 1)


def _step_masses(n, nfe, m, parts):
    t = torch.full((n,), m.DtOverMassSi, dtype=torch.float64, device=DEV)
    for (a, _), k in zip(parts, nfe):
        t[a:a + k] = m.DtOverMassFe
    return t


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        pos, vel, n, fc, mc, _ = _ensemble(case, seed)
        P, V = _gpu(pos), _gpu(vel)
        xs, vs, a = [], [], 0
        for s in range(len(n)):
            b = a + int(n[s])
            parts = [(0, b - a)]
            x, v = _steps64(P[a:b], V[a:b], [fc[s].NFe], fc[s], mc[s].Dt,
                               _step_masses(b - a, [fc[s].NFe], mc[s], parts), 0.0, case["steps"], parts)
            xs.append(x)
            vs.append(v)
            a = b
        return {"pos": _full(torch.cat(xs), P), "vel": _full(torch.cat(vs), V)}
    if kind == "separate":
        pos, vel, fc, mc = _bodies(case, seed)
        parts = [(0, fc.boarder2), (fc.boarder2, len(pos))]
        nfe, damp = [fc.boarder1, fc.boarder3 - fc.boarder2], 8.0
    else:
        pos, vel, fc, mc, info = _impact(case, seed)
        parts, nfe, damp = [(0, len(pos))], [fc.NFe], 0.0
    P, V = _gpu(pos), _gpu(vel)
    n = len(pos)
    if kind == "force":
        return {"force": _full(_force64(P[:, :3].double(), V[:, :3].double(), fc.NFe, fc), torch.zeros_like(P))}
    if kind in ("steps", "separate"):
        x, v = _steps64(P, V, nfe, fc, mc.Dt, _step_masses(n, nfe, mc, parts), damp, case["steps"], parts)
        return {"pos": _full(x, P), "vel": _full(v, V)}
    m = torch.where(torch.arange(n, device=DEV) < fc.NFe, MASS_FE, 1.0).double()[:, None]
    x, v = P[:, :3].double(), V[:, :3].double()
    if kind == "recenter":
        rng = np.random.default_rng([seed, 7])
        com, mean = (torch.tensor(rng.uniform(-w, w, 3), device=DEV) for w in (1.0, 0.1))
        return {"pos": _full(x + (com - (m * x).sum(0) / m.sum()), P),
                "vel": _full(v + (mean - (m * v).sum(0) / m.sum()), V)}
    return None  # earth_moon: groups are whole numbers, and its sums are in 64 bits already
