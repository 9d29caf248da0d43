"""The performance cases of this framework: what its users have it compute, at the sizes they use.

A case is a plain dict; `prepare` makes what a program has in hand before the call, `run` is one pass
through the public entry points, `work` what the pass cannot do without, and `exact` its result in
64 bits where plain torch gives it.

Paths:
- "pk":         `spectrum_matter` of one cosmology (background, modes, P(k)): the interactive call.
- "sets":       `solve_sets`, one k grid over many parameter sets: scans and likelihood batches.
- "spectra":    `surrogate.solve_spectra`, log P(k) of many parameter rows: training data.
- "sources":    a kept plan that saves the CMB sources (S_T, S_E, S_ψ) of every mode.
- "problems":   `spectrum_matter_problems`, problems of several model families in one launch.
- "tangent":    `spectrum_matter_tangent`, forward-mode ∂ log P / ∂ log θ.
- "cmb":        `spectrum_cmb_sets`, TT/EE/ψψ to l = 2500.
- "background": `solvebg_sets` of a batch large enough for the GPU.
- "train":      Adam steps of the surrogate's network.  "infer": its forward pass.

The adaptive solves stop at their tolerances (rtol = 1e-5, backgrounds 1e-7): they have no 64-bit
value short of integrating the whole Einstein-Boltzmann system and its recombination history again
at tight tolerance, so `exact` is None for them.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "symboltz.jl_amd"))

from symboltz import models, workloads  # noqa: E402
from symboltz import surrogate as sg  # noqa: E402
from symboltz.bessel import SphericalBesselCache  # noqa: E402
from symboltz.cmb import spectrum_cmb_sets  # noqa: E402
from symboltz.constants import k_dimensionless  # noqa: E402
from symboltz.mlp import Mlp  # noqa: E402
from symboltz.problem import (CosmologyProblem, _gpu_model, solve_sets, solvebg, solvebg_sets,  # noqa: E402
                              spectrum_matter, spectrum_matter_problems, spectrum_matter_tangent)
from symboltz.solver import SAVE_SOURCES  # noqa: E402

FAMILIES = {
    "massless10": models.LCDM(lmax=10, h=False),                        # n = 38
    "lcdm5": models.LCDM(lmax=5),                                       # n = 47, the CLASS-comparison model
    "lcdm6": models.LCDM(lmax=6),                                       # n = 54, the surrogate's model
    "w0wa6": models.w0waCDM(lmax=6),                                    # n = 56
    "nu100": models.LCDM(lmax_g=16, lmax_nu=16, lmax_h=10, nx=4),       # n = 100
    "lcdm32": models.LCDM(lmax=32),                                     # n = 236
}
WIDTHS = [len(sg.PARAMS), 512, 512, 512, 512, 256]                      # the surrogate's network
LR = 1e-3


def listed():
    return [
        # a quick look at a handful of wavenumbers: nothing but latency
        {"name": "pk few k", "path": "pk", "model": "lcdm5", "n_k": 5, "k_min": 1e-3, "k_max": 0.1},
        # the massless-ν spectrum on its usual 100 k
        {"name": "pk massless 100 k", "path": "pk", "model": "massless10", "n_k": 100, "k_min": 1e-4, "k_max": 1.0},
        # the batched solve of the benchmark: 128 cosmologies x 512 k to 10/Mpc
        {"name": "sets massless 128x512", "path": "sets", "model": "massless10", "n_sets": 128, "n_k": 512,
         "k_min": 1e-5, "k_max": 10.0},
        # a likelihood batch of the massive-ν model with long hierarchies, ragged
        {"name": "sets nu100 13x201", "path": "sets", "model": "nu100", "n_sets": 13, "n_k": 201, "k_min": 1e-4,
         "k_max": 5.0},
        # a chunk of the surrogate's training spectra on its own grid
        {"name": "spectra lcdm6 31x256", "path": "spectra", "n_sets": 31, "n_k": 256},
        # CMB sources of the massive-ν model on a fine time grid
        {"name": "sources nu100 200x1000", "path": "sources", "model": "nu100", "n_k": 200, "n_tau": 1000,
         "k_min": 1e-5, "k_max": 0.5},
        # a stream of requests over five model families (38 to 236 unknowns)
        {"name": "problems 20x64", "path": "problems", "n_sets": 20, "n_k": 64, "k_min": 1e-4, "k_max": 1.0},
        # derivatives of P(k) with respect to Ω_c0 and Ω_b0, as a Fisher forecast asks for
        {"name": "tangent lcdm5 20 k", "path": "tangent", "model": "lcdm5", "n_k": 20, "k_min": 3e-4, "k_max": 0.25},
        # CMB power spectra of four cosmologies
        {"name": "cmb lcdm5 4 sets", "path": "cmb", "model": "lcdm5", "n_sets": 4},
        # the backgrounds of a batch of cosmologies
        {"name": "background lcdm6 1000", "path": "background", "model": "lcdm6", "n_sets": 1000},
        # surrogate training: 16 Adam steps of batch 1024
        {"name": "train 16x1024", "path": "train", "n_steps": 16, "batch": 1024},
        # surrogate serving: a large batch of requests
        {"name": "infer 65536", "path": "infer", "rows": 65536},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(_log(rng, lo, hi)))))


def draw(rng):
    path = rng.choice(["pk", "pk", "sets", "sets", "spectra", "sources", "problems", "tangent", "cmb", "background",
                       "train", "infer"])
    if path == "pk":
        m = rng.choice(["massless10", "lcdm5", "lcdm6", "w0wa6", "nu100"])
        return {"path": path, "model": m, "n_k": _logint(rng, 3, 600), "k_min": _log(rng, 1e-5, 1e-3),
                "k_max": _log(rng, 0.02, 1.0 if m == "w0wa6" else 5.0)}
    if path == "sets":
        m = rng.choice(["massless10", "lcdm6", "nu100"])
        cap = 40000 if m == "massless10" else 5000
        n_sets = _logint(rng, 2, 128)
        return {"path": path, "model": m, "n_sets": n_sets, "n_k": _logint(rng, 8, max(9, min(700, cap // n_sets))),
                "k_min": _log(rng, 1e-5, 1e-3), "k_max": _log(rng, 0.1, 10.0 if m == "massless10" else 5.0)}
    if path == "spectra":
        return {"path": path, "n_sets": _logint(rng, 3, 40), "n_k": 256}
    if path == "sources":
        return {"path": path, "model": rng.choice(["massless10", "lcdm5", "nu100"]), "n_k": _logint(rng, 12, 400),
                "n_tau": _logint(rng, 50, 1500), "k_min": _log(rng, 1e-5, 1e-3), "k_max": _log(rng, 0.05, 0.5)}
    if path == "problems":
        return {"path": path, "n_sets": _logint(rng, 5, 60), "n_k": _logint(rng, 8, 64), "k_min": _log(rng, 1e-4, 1e-3),
                "k_max": _log(rng, 0.1, 1.0)}
    if path == "tangent":
        return {"path": path, "model": rng.choice(["massless10", "lcdm5"]), "n_k": _logint(rng, 4, 100),
                "k_min": _log(rng, 1e-4, 1e-3), "k_max": _log(rng, 0.05, 0.25)}
    if path == "cmb":
        return {"path": path, "model": "lcdm5", "n_sets": rng.randint(1, 10)}
    if path == "background":
        return {"path": path, "model": rng.choice(["massless10", "lcdm6", "nu100"]), "n_sets": _logint(rng, 256, 2000)}
    if path == "train":
        return {"path": path, "n_steps": _logint(rng, 2, 32), "batch": rng.choice([64, 250, 512, 1024, 2048])}
    return {"path": path, "rows": _logint(rng, 1, 65536)}


def _cosmology(M, rng):
    """A parameter set of model M drawn from the ranges of the batched workloads."""
    h = rng.uniform(0.60, 0.75)
    p = dict(models.parameters_Planck18(M), h=h, Omega_b0=rng.uniform(0.020, 0.024) / h**2,
             Omega_c0=rng.uniform(0.10, 0.14) / h**2, ln_As1e10=rng.uniform(2.9, 3.2), ns=rng.uniform(0.92, 1.0),
             z_re=rng.uniform(6.2, 10.3))
    if M == FAMILIES["massless10"]:
        p.update(Neff=3.046)
    elif M == FAMILIES["nu100"]:
        p.update(N=1, m_eV=rng.uniform(0.06, 0.30), Neff=2.046)
    elif M.has_h:
        p.update(N=3, m_eV=rng.uniform(0.06, 0.30) / 3)
    if M.de == "w0wa":
        p.update(w0=rng.uniform(-0.95, -0.8), wa=rng.uniform(-0.04, 0.3))
    return p


def _weights(rng):
    """Random network parameters in the framework's order (weights [in][out] of every layer, then biases)."""
    W = [rng.normal(0, math.sqrt(2.0 / a), (a, b)) for a, b in zip(WIDTHS, WIDTHS[1:])]
    b = [rng.normal(0, 0.02, n) for n in WIDTHS[1:]]
    return np.concatenate([w.ravel() for w in W] + b).astype(np.float32)


def _rows(case, rng):
    """(inputs, targets) of the surrogate's network; targets only for training."""
    n = case["batch"] * case["n_steps"] if case["path"] == "train" else case["rows"]
    X = rng.uniform(-1, 1, (n, WIDTHS[0])).astype(np.float32)
    return X, rng.normal(0, 1, (n, WIDTHS[-1])).astype(np.float32) if case["path"] == "train" else None


_bessel = {}


def _bessel_cache():
    """The Bessel table to l = 2500 that a program keeps for all its spectra."""
    if not _bessel:
        ls = np.unique(np.round(np.exp(np.linspace(math.log(2), math.log(2500), 200))).astype(int))
        _bessel["jl"] = SphericalBesselCache(ls)
        _bessel["jl"].context()
    return _bessel["jl"]


def prepare(case, seed):
    rng = np.random.default_rng([seed, 17])
    path = case["path"]
    s = {"path": path, "case": case}
    if path in ("pk", "sets", "sources", "tangent"):
        M = FAMILIES[case["model"]]
        ks = np.geomspace(case["k_min"], case["k_max"], case["n_k"])
        sets = [_cosmology(M, rng) for _ in range(case.get("n_sets", 1))]
        s.update(M=M, sets=sets, ks=k_dimensionless(ks, sets[0]["h"]))
        _gpu_model(M)                                    # the compiled model, kept by the process
        if path in ("pk", "tangent"):
            s["prob"] = CosmologyProblem(M, sets[0])
        if path == "sources":
            bg = solvebg(CosmologyProblem(M, sets[0]))
            gm = _gpu_model(M)
            gm.upload_background(0, bg.t, bg.u, bg.du, bg.P)
            t0 = np.clip(np.minimum(1e-2 / s["ks"], 1e-4), bg.t[0], bg.t[-1])
            s["plan"] = gm.plan(np.zeros(case["n_k"], np.int32), s["ks"], t0, save=SAVE_SOURCES,
                                saveat=workloads.source_taus(bg.t[0], bg.t[-1], case["n_tau"]))
    elif path == "spectra":
        s.update(X=rng.uniform(sg.LO, sg.HI, (case["n_sets"], len(sg.LO))), ks=sg.k_grid(case["n_k"]))
    elif path == "problems":
        fams = workloads.mixed_families()
        s["probs"] = [CosmologyProblem(fams[i % len(fams)], _cosmology(fams[i % len(fams)], rng))
                      for i in range(case["n_sets"])]
        s["ks"] = k_dimensionless(np.geomspace(case["k_min"], case["k_max"], case["n_k"]), 0.67)
        for M in fams:
            _gpu_model(M)
    elif path == "cmb":
        M = FAMILIES[case["model"]]
        s["probs"] = [CosmologyProblem(M, _cosmology(M, rng)) for _ in range(case["n_sets"])]
        s["bgs"] = [solvebg(p) for p in s["probs"]]
        s["jl"] = _bessel_cache()
        _gpu_model(M)
    elif path == "background":
        M = FAMILIES[case["model"]]
        s["probs"] = [CosmologyProblem(M, _cosmology(M, rng)) for _ in range(case["n_sets"])]
    else:
        X, T = _rows(case, rng)
        net = Mlp(WIDTHS, max_batch=case["batch"] if path == "train" else 65536, seed=seed % 1000)
        net.set_params(_weights(rng))
        s.update(net=net, X=X)
        if path == "train":
            net.set_data(X, T)
            s["order"] = rng.permutation(len(X))
    return s


def _table(rows):
    """Arrays of different lengths as the rows of one, NaN past their ends."""
    out = np.full((len(rows), 1280) + rows[0].shape[1:], np.nan)
    for o, r in zip(out, rows):
        o[:len(r)] = r
    return out


def run(s):
    path, case = s["path"], s["case"]
    if path == "pk":
        P, sol = spectrum_matter(s["prob"], s["ks"])
        return {"P": P, "retcode": sol.pts["retcode"]}
    if path == "sets":
        P, res, _ = solve_sets(s["M"], s["sets"], s["ks"])
        return {"P": P, "retcode": res["retcode"]}
    if path == "spectra":
        return {"logP": sg.solve_spectra(s["X"], s["ks"])[0]}
    if path == "sources":
        s["plan"].run()
        S = s["plan"].sources()
        return {"S_T": S[:, :, 0], "S_E": S[:, :, 1], "S_psi": S[:, :, 2], "retcode": s["plan"].fetch()["retcode"]}
    if path == "problems":
        return {"P": spectrum_matter_problems(s["probs"], s["ks"])}
    if path == "tangent":
        J, P = spectrum_matter_tangent(s["prob"], s["ks"], ["Omega_c0", "Omega_b0"])
        return {"J": J, "P": P}
    if path == "cmb":
        D = spectrum_cmb_sets(["TT", "EE", "ψψ"], s["probs"], s["jl"], normalization="Dl", bgs=s["bgs"])
        return {"TT": D[:, :, 0], "EE": D[:, :, 1], "psipsi": D[:, :, 2]}
    if path == "background":
        bgs = solvebg_sets(s["probs"])
        return {"P": np.stack([b.P for b in bgs]), "t": _table([b.t for b in bgs]), "u": _table([b.u for b in bgs])}
    if path == "train":
        loss, _ = s["net"].train(s["order"], case["batch"], LR)
        return {"loss": loss, "params": s["net"].get_params()}
    return {"y": s["net"].forward(s["X"])[0]}


# Steps of one mode at rtol = 1e-5 against k (H0/c), and the flops of one Rodas5P step of n unknowns.
_STEPS = ([0.045, 4.5, 14.0, 45.0, 141.0, 447.0, 1415.0, 4475.0, 14150.0, 44750.0],
          [96, 110, 135, 240, 505, 1160, 2200, 3010, 3250, 3400])


def _mode_flops(ks_mpc, n):
    steps = np.interp(np.log(np.asarray(ks_mpc) * 4470.0), np.log(_STEPS[0]), _STEPS[1])
    return float(steps.sum()) * (340.0 * n - 2500.0)


def work(case):
    path = case["path"]
    table = 11 * 900 * 8.0                               # one background table: 900 knots of t, u, du
    if path in ("pk", "sets", "sources", "tangent", "spectra"):
        n = FAMILIES["lcdm6" if path == "spectra" else case["model"]].n_unknowns
        ks = sg.k_grid(case["n_k"]) if path == "spectra" else np.geomspace(case["k_min"], case["k_max"], case["n_k"])
        sets = case.get("n_sets", 1)
        out = sets * len(ks) * 8.0
        flops = sets * _mode_flops(ks, n)
        if path == "tangent":
            flops *= 4                                   # two parameters, primal and tangent
        if path == "sources":
            out = len(ks) * case["n_tau"] * 24.0
            flops += len(ks) * case["n_tau"] * 20.0 * n
        return {"bytes": sets * table + out, "flops": flops}
    if path == "problems":
        fams = workloads.mixed_families()
        ks = np.geomspace(case["k_min"], case["k_max"], case["n_k"])
        return {"bytes": case["n_sets"] * (table + len(ks) * 8.0),
                "flops": sum(_mode_flops(ks, fams[i % len(fams)].n_unknowns) for i in range(case["n_sets"]))}
    if path == "cmb":
        nk, nt, nl = 10300.0, 300.0, 152.0               # fine k, times, multipoles
        ks = np.geomspace(3e-6, 2.2, 131)
        return {"bytes": case["n_sets"] * (table + nk * nl * 24.0),
                "flops": case["n_sets"] * (_mode_flops(ks, 47) + nk * nt * nl * 18.0)}
    if path == "background":                             # 900 steps of 9 right-hand sides, ~1,000 flops each
        return {"bytes": case["n_sets"] * table, "flops": case["n_sets"] * 900 * 9 * 1000.0}
    macs = float(sum(a * b for a, b in zip(WIDTHS, WIDTHS[1:])))
    if path == "train":
        rows = float(case["n_steps"] * case["batch"])
        return {"bytes": rows * 4 * (WIDTHS[0] + WIDTHS[-1]) + case["n_steps"] * macs * 28, "flops": 6 * rows * macs}
    return {"bytes": case["rows"] * 4.0 * (WIDTHS[0] + WIDTHS[-1]) + macs * 2, "flops": 2 * case["rows"] * macs}


def _unpack(p):
    W, b, o = [], [], 0
    for a, c in zip(WIDTHS, WIDTHS[1:]):
        W.append(p[o:o + a * c].reshape(a, c).clone())
        o += a * c
    for c in WIDTHS[1:]:
        b.append(p[o:o + c].clone())
        o += c
    return W, b


def _forward(W, b, x):
    for i, (w, c) in enumerate(zip(W, b)):
        x = x @ w + c
        if i < len(W) - 1:
            x = torch.nn.functional.gelu(x)
    return x


def exact(case, seed):
    path = case["path"]
    if path not in ("train", "infer"):
        return None
    rng = np.random.default_rng([seed, 17])
    X, T = _rows(case, rng)
    W, b = _unpack(torch.from_numpy(_weights(rng)).double())
    if path == "infer":
        y = torch.cat([_forward(W, b, torch.from_numpy(X[i:i + 8192]).double()) for i in range(0, len(X), 8192)])
        return {"y": y.numpy()}
    if case["n_steps"] * case["batch"] > 20000:
        return None
    order = rng.permutation(len(X))
    ps = [p.requires_grad_() for p in W + b]
    opt = torch.optim.Adam(ps, lr=LR, betas=(0.9, 0.999), eps=1e-8)
    loss = []
    for i in range(case["n_steps"]):
        at = order[i * case["batch"]:(i + 1) * case["batch"]]
        opt.zero_grad()
        e = torch.mean((_forward(W, b, torch.from_numpy(X[at]).double()) - torch.from_numpy(T[at]).double()) ** 2)
        e.backward()
        opt.step()
        loss.append(e.item())
    return {"loss": np.array(loss), "params": torch.cat([p.detach().reshape(-1) for p in ps]).numpy()}
