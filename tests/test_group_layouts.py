"""The kernels with one hierarchy per lane at the layouts where their compile-time rules switch: 12 slots per
lane (the last with both sweeps' factors kept and the background's look-ahead interval), 13 (the first
without), and five momentum bins without massless neutrinos (seven hierarchies, all eight lanes in use);
against the one-mode kernel and the oracle, with the bounds of test_group.py."""
import numpy as np
import pytest

from conftest import Setup
from emu.emu import WaveEmu
from symboltz import models
from symboltz.solver import has_group, model_source
from test_group import TOL, compare

LAYOUTS = {"12 slots": (dict(lmax_g=11, lmax_nu=4, lmax_h=3, nx=1), 12, 8),
           "13 slots": (dict(lmax=12, h=False), 13, 4),
           "five bins, no massless neutrinos": (dict(lmax=6, nu=False, nx=5), 7, 8)}


@pytest.mark.parametrize("name", list(LAYOUTS))
def test_emulated_layouts_match_one_mode_kernel_and_oracle(name):
    kw, slots, lanes = LAYOUTS[name]
    M = models.LCDM(**kw)
    S = Setup(M, models.parameters_Planck18(M))
    src = model_source(M).full_src
    assert has_group(src) and f"\n#define SBZ_GM {slots}\n" in src and f"\n#define SBZ_GL {lanes}\n" in src
    # the emulator's slot of the alternative layout runs the saving group kernel
    E = WaveEmu(src.replace("sbz_wave_kernel_altlu", "sbz_wave_kernel_other")
                .replace("sbz_group_save_kernel", "sbz_wave_kernel_altlu"))
    ks = np.concatenate([np.geomspace(0.05, 2.0, 3), [0.0]])
    t0 = np.clip(np.minimum(1e-2 / np.where(ks > 0, ks, 1.0), 1e-4), S.t[0], S.t[-1])
    saveat = np.linspace(0.05, 0.95 * S.t[-1], 5)
    w = E.solve(S.P, S.t, S.u, S.du, ks, t0, saveat=saveat, sources=True, srcbg=True)
    g = E.solve(S.P, S.t, S.u, S.du, ks, t0, saveat=saveat, sources=True, srcbg=True, altlu=True)
    assert list(w["retcode"]) == [0] * 3 + [4]
    compare(g, w, 3)
    o = S.O.solve(ks[:3], t0[:3])
    assert np.max(np.abs(g["u"][:3] - o["u"]) / np.abs(o["u"]).max(axis=1, keepdims=True)) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(lmax=11), dict(lmax=12, h=False), dict(lmax=6, nu=False, nx=5)],
                         ids=["12 slots", "13 slots", "five bins"])
def test_gpu_layouts_match_one_mode_kernel(kw):
    """Two sets, two wavefronts (groups refill), states and sources saved; and without saves."""
    from symboltz.solver import ALGO_WAVE, SAVE_SOURCES, SAVE_STATES, GpuModel
    M = models.LCDM(**kw)
    p = models.parameters_Planck18(M)
    gm = GpuModel(M)
    try:
        sets = [Setup(M, dict(p, h=h)) for h in (0.67, 0.7)]
        for i, S in enumerate(sets):
            gm.upload_background(i, S.t, S.u, S.du, S.P)
        n_k = 19
        ks = np.tile(np.geomspace(0.01, 100.0, n_k), 2)
        iset = np.repeat(np.arange(2, dtype=np.int32), n_k)
        t0 = np.array([np.clip(min(1e-2 / k, 1e-4), sets[i].t[0], 1.0) for k, i in zip(ks, iset)])
        taus = np.linspace(0.05, 0.9 * min(S.t[-1] for S in sets), 11)
        out = {}
        for algo in (0, ALGO_WAVE):
            print(f"case: n = {M.n_unknowns}, 2 x {n_k} k, algo {algo}", flush=True)
            plan = gm.plan(iset, ks, t0, saveat=taus, lanes=2, save=SAVE_STATES | SAVE_SOURCES, algo=algo)
            plan.run()
            out[algo] = dict(plan.fetch(), src=plan.sources())
            plan.close()
        assert np.all(out[ALGO_WAVE]["retcode"] == 0)
        compare(out[0], out[ALGO_WAVE], len(ks))
        plan = gm.plan(iset, ks, t0, lanes=2)
        plan.run()
        u = plan.fetch()["u"]
        plan.close()
        assert np.max(np.abs(u - out[0]["u"]) / np.abs(u).max(axis=1, keepdims=True)) < TOL
    finally:
        gm.close()
