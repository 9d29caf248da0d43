"""The kernels of the models without one hierarchy per lane (a hierarchy beyond l = 17, five momentum
bins beside massless neutrinos), whose names the other models share: the 16-lane and the 32-lane row bodies
behind sbz_wave4_kernel and sbz_wave2h_kernel, the one-mode tangent (lanes of more than 12 slots), and the
row tickets of the mixed-model launch; against the one-mode kernel and the oracle.  Bounds as where these
bodies were tested before (test_wave_emu.py, test_configs.py, test_stream.py): states 1e-8 of the one-mode
kernel's in the emulator and 1e-6 on the device, 1e-4 of the oracle's."""
import numpy as np
import pytest

from conftest import Setup
from emu.emu import WaveEmu
from symboltz import models
from symboltz.solver import has_group, model_source

ROWS16 = models.LCDM(lmax=18, h=False)
ROWS32 = models.LCDM(lmax=4, nx=5)
TANGENT = models.LCDM(lmax=12, h=False)


def rel(a, b):
    return np.max(np.abs(a - b) / np.maximum(np.abs(b).max(axis=-1, keepdims=True), 1e-300))


def starts(S, ks):
    return np.clip(np.minimum(1e-2 / np.where(ks > 0, ks, 1.0), 1e-4), S.t[0], S.t[-1])


@pytest.mark.parametrize("M, variant", [(ROWS16, "wave4"), (ROWS32, "wave2h")], ids=["16 lanes", "32 lanes"])
def test_emulated_row_bodies_match_oracle_and_one_mode_kernel(M, variant):
    """More instances than rows, so that rows refill, and two that fail at their start."""
    S = Setup(M, models.parameters_Planck18(M))
    src = model_source(M).full_src
    assert not has_group(src)
    E = WaveEmu(src)
    assert (E.L.emu_has_wave4(), E.L.emu_has_wave2h()) == ((1, 0) if variant == "wave4" else (0, 1))
    ks = np.array([5.0, 0.3, 0.0, 3.0, 1.0, np.nan, 2.0] if variant == "wave4" else [3.0, 0.0, 0.3, np.nan, 1.0])
    t0 = starts(S, ks)
    good = np.isfinite(ks) & (ks > 0)
    r = E.solve(S.P, S.t, S.u, S.du, ks, t0, **{variant: True})
    w = E.solve(S.P, S.t, S.u, S.du, ks, t0)
    assert list(r["retcode"]) == [0 if g else 4 for g in good]
    o = S.O.solve(ks[good], t0[good])
    assert rel(r["u"][good], o["u"]) < 1e-4
    assert rel(r["u"][good], w["u"][good]) < 1e-8
    assert np.all(np.abs(r["stats"][good, 0] - w["stats"][good, 0]) <= 2)


def test_emulated_one_mode_tangent_matches_oracle_differences():
    """u equals the plain kernel's, and s + f(τ0) dτ0/dlog θ the central difference of oracle solves at
    log θ ± h (1e-3, as test_wave_emu.py holds the tangent to)."""
    from oracle import oracle
    from symboltz import _lib
    S = Setup(TANGENT, models.parameters_Planck18(TANGENT))
    src = model_source(TANGENT).full_src
    assert "\n#define SBZ_GM 13\n" in src     # one slot more than the tangent in groups takes
    E = WaveEmu(src)
    assert E.L.emu_has_tan() == 1
    ks = np.array([1.0, 5.0])
    t0 = starts(S, ks)
    h, x, tight = 1e-3, np.log(S.pars["Omega_c0"]), []
    for sgn in (1, -1):
        P = models.make_params(S.M, dict(S.pars, Omega_c0=np.exp(x + sgn * h)))
        tight.append(_lib.background_solve(P, 1e-10, 1e-10, 100000)[:4])
    g = E.solve_tangent([(S.P, S.t, S.u, S.du)] + tight, ks, t0, 0.5 / h)
    w = E.solve(S.P, S.t, S.u, S.du, ks, t0)
    assert list(g["retcode"]) == [0, 0]
    assert rel(g["u"], w["u"]) < 1e-8 and np.all(g["stats"][:, 0] == w["stats"][:, 0])
    fd = []
    for P, t, u, du in tight:
        o = oracle.Oracle(S.M, P, t, u, du).solve(ks, t0, rtol=1e-9, atol=1e-9, maxiters=10**6)
        assert np.all(o["retcode"] == 0)
        fd.append(o["u"])
    fd = (fd[0] - fd[1]) / (2 * h)
    s = g["s"] + g["fend"] * (tight[0][1][-1] - tight[1][1][-1]) / (2 * h)
    assert rel(s, fd) < 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("M, algo", [(ROWS16, 4), (ROWS32, 6)], ids=["16 lanes", "32 lanes"])
def test_gpu_row_bodies_match_one_mode_kernel_and_oracle(M, algo):
    from symboltz.solver import ALGO_WAVE, GpuModel
    S = Setup(M, models.parameters_Planck18(M))
    gm = GpuModel(M)
    try:
        assert gm.group == 0
        gm.upload_background(0, S.t, S.u, S.du, S.P)
        ks = np.geomspace(0.05, 300.0, 37)
        t0 = starts(S, ks)
        out = {}
        for a, lanes in ((algo, 3), (ALGO_WAVE, 0)):   # three wavefronts: rows refill
            print(f"case: n = {M.n_unknowns}, 37 k, algo {a}", flush=True)
            plan = gm.plan(np.zeros(len(ks), np.int32), ks, t0, algo=a, lanes=lanes)
            plan.run()
            out[a] = plan.fetch()
            plan.close()
        r, w = out[algo], out[ALGO_WAVE]
        assert np.all(r["retcode"] == 0) and np.all(w["retcode"] == 0)
        assert rel(r["u"], w["u"]) < 1e-6
        assert np.all(np.abs(r["stats"][:, 0] - w["stats"][:, 0]) <= 2 + 0.01 * w["stats"][:, 0])
        o = S.O.solve(ks[::6], t0[::6])
        assert rel(r["u"][::6], o["u"]) < 1e-4
    finally:
        gm.close()


@pytest.mark.gpu
def test_gpu_one_mode_tangent_matches_tight_oracle_differences():
    """d log P / d log θ against central differences of oracle solves at rtol 1e-9 (1e-3, the bar of
    test/runtests.jl:363-377).  Differences of rtol 1e-5 solves are no reference here: at k = 300 they are
    off by 8e-3, the GPU's and the oracle's alike."""
    from oracle import oracle
    from symboltz import _lib
    from symboltz.problem import CosmologyProblem, spectrum_matter, spectrum_matter_tangent
    prob = CosmologyProblem(TANGENT, models.parameters_Planck18(TANGENT))
    ks = np.geomspace(1.0, 300.0, 8)
    names = ["Omega_c0", "Omega_b0"]
    print("case: n = 44, 8 k, tangent of two parameters", flush=True)
    J, P = spectrum_matter_tangent(prob, ks, names)
    P0, _ = spectrum_matter(prob, ks)
    assert np.max(np.abs(P / P0 - 1)) < 1e-6
    h = 1e-3
    for j, nm in enumerate(names):
        logP = []
        for sgn in (1, -1):
            pars = dict(models.parameters_Planck18(TANGENT))
            pars[nm] *= np.exp(sgn * h)
            Q, t, u, du = _lib.background_solve(models.make_params(TANGENT, pars), 1e-10, 1e-10, 100000)[:4]
            O = oracle.Oracle(TANGENT, Q, t, u, du)
            o = O.solve(ks, np.clip(np.minimum(1e-2 / ks, 1e-4), t[0], t[-1]), rtol=1e-9, atol=1e-9, maxiters=10**6)
            logP.append(np.log([O.p0(k) * O.delta_m(k, t[-1], o["u"][i])**2 for i, k in enumerate(ks)]))
        assert np.max(np.abs(J[:, j] - (logP[0] - logP[1]) / (2 * h))) < 1e-3, nm


@pytest.mark.gpu
def test_gpu_mixed_launch_with_row_tickets_matches_per_family():
    """A row family with twice the resident wavefronts' worth of modes takes row tickets, beside a family
    with one hierarchy per lane; with fewer it runs in its one-mode body."""
    from symboltz.multi import MultiModel
    from symboltz.solver import ALGO_WAVE, GpuModel
    fams = [ROWS16, models.LCDM(lmax=10, h=False)]
    gms = [GpuModel(M) for M in fams]
    mm = MultiModel(gms)
    try:
        assert mm.rows() == [4, 4]
        setups = [Setup(M, models.parameters_Planck18(M)) for M in fams]
        for g, S in zip(gms, setups):
            g.upload_background(0, S.t, S.u, S.du, S.P)
        for n in (3 * mm.capacity(), 40):
            ks = np.geomspace(0.05, 60.0, n)
            print(f"case: {n} modes of n = {ROWS16.n_unknowns} beside 33 of n = 38", flush=True)
            plans, ref = [], []
            for g, S, k in zip(gms, setups, (ks, np.geomspace(0.05, 60.0, 33))):
                plans.append(g.plan(np.zeros(len(k), np.int32), k, starts(S, k)))
                p = g.plan(np.zeros(len(k), np.int32), k, starts(S, k), algo=ALGO_WAVE)
                p.run()
                ref.append(p.fetch())
                p.close()
            mm.run(plans)
            for p, r in zip(plans, ref):
                got = p.fetch()
                p.close()
                assert np.all(got["retcode"] == 0)
                assert rel(got["u"], r["u"]) < 1e-6
    finally:
        mm.close()
        for g in gms:
            g.close()
