"""The kernels with one hierarchy per lane (algo 0 of the models that have them) against the
one-mode kernel and the oracle, at the edges of their lane layout: the shortest hierarchies, the
longest that fit, 4 and 8 lanes per mode, every group of a wavefront filled and refilled, saves,
sources and the failure codes; and their compiled code, against a fault of the compiler's register
allocation (KERNEL_FLAGS of symboltz.build)."""
import re
import subprocess

import numpy as np
import pytest

from conftest import Setup
from emu.emu import WaveEmu
from symboltz import models
from symboltz.build import KERNEL_FLAGS
from symboltz.solver import has_group, model_source

# Both kernels take the same steps from the same start, in another order of summation: what differs
# is rounding, amplified by the stiff start to at most 1e-6 of the largest state (the bound that
# the row kernels' tests hold to), a tenth of the local error that the steps are accepted with.
TOL = 1e-6


def compare(g, w, n_ok):
    assert list(g["retcode"]) == list(w["retcode"])
    assert np.all(np.abs(g["stats"][:n_ok, 0] - w["stats"][:n_ok, 0]) <= 2 + 0.01 * w["stats"][:n_ok, 0])
    for q in ("u", "usave"):
        if w.get(q) is not None:
            sc = np.abs(w[q][:n_ok]).max(axis=-1, keepdims=True)
            assert np.max(np.abs(g[q][:n_ok] - w[q][:n_ok]) / sc) < TOL, q
    if w.get("src") is not None:
        sc = np.abs(w["src"][:n_ok]).max(axis=1, keepdims=True)
        assert np.max(np.abs(g["src"][:n_ok] - w["src"][:n_ok]) / sc) < TOL


CASES = {
    "4 lanes, shortest": (dict(lmax=3, h=False), 4),
    "8 lanes, longest": (dict(lmax_g=17, lmax_nu=4, lmax_h=3, nx=2), 8),
    "dark-energy fluid, shortest": (dict(lmax=3), 8),
}


@pytest.mark.parametrize("name", list(CASES))
def test_emulated_group_kernel_matches_one_mode_kernel_and_oracle(name):
    kw, lanes = CASES[name]
    M = (models.w0waCDM if "fluid" in name else models.LCDM)(**kw)
    S = Setup(M, dict(models.parameters_Planck18(M), **(dict(w0=-0.9, wa=0.1) if "fluid" in name else {})))
    src = model_source(M).full_src
    assert has_group(src) and f"\n#define SBZ_GL {lanes}\n" in src
    # the emulator's slot of the alternative layout runs the saving group kernel
    E = WaveEmu(src.replace("sbz_wave_kernel_altlu", "sbz_wave_kernel_other")
                .replace("sbz_group_save_kernel", "sbz_wave_kernel_altlu"))
    ks = np.concatenate([np.geomspace(0.05, 3.0, 64 // lanes + 1 if lanes > 4 else 4), [0.0, np.nan]])
    ok = len(ks) - 2
    t0 = np.clip(np.minimum(1e-2 / np.where(ks > 0, ks, 1.0), 1e-4), S.t[0], S.t[-1])
    saveat = np.concatenate([[t0[:ok].min()], np.linspace(0.05, S.t[-1], 6), [S.t[-1]]])
    w = E.solve(S.P, S.t, S.u, S.du, ks, t0, saveat=saveat, sources=True, srcbg=True)
    g = E.solve(S.P, S.t, S.u, S.du, ks, t0, saveat=saveat, sources=True, srcbg=True, altlu=True)
    assert list(w["retcode"]) == [0] * ok + [4, 4]
    w["src"][:, -2:] = g["src"][:, -2:] = 1.0   # at τ0 the visibility's χ = 0 terms are not finite
    compare(g, w, ok)
    o = S.O.solve(ks[:ok], t0[:ok])
    assert np.max(np.abs(g["u"][:ok] - o["u"]) / np.abs(o["u"]).max(axis=1, keepdims=True)) < 1e-4
    f = E.solve(S.P, S.t, S.u, S.du, ks, t0, maxiters=20, altlu=True)
    f1 = E.solve(S.P, S.t, S.u, S.du, ks, t0, maxiters=20)
    assert list(f["retcode"]) == list(f1["retcode"]) and f["retcode"][0] == 1


def test_models_that_need_16_lanes_have_no_group_kernel():
    for nx in (4, 5):
        assert has_group(model_source(models.LCDM(lmax=4, nx=nx)).full_src) == (nx == 4)


@pytest.mark.parametrize("kw", [dict(lmax=10, h=False), dict(lmax=6)], ids=["n38", "n54"])
def test_no_vector_copy_before_a_join_restores_the_exec_mask(kw, tmp_path):
    """A vector register copied at the head of a join block before `s_or_b64 exec` keeps its value
    only in the lanes of the branch just left; the other lanes' copies are lost."""
    src, asm = tmp_path / "m.hip", tmp_path / "m.s"
    src.write_text(model_source(models.LCDM(**kw)).full_src)
    subprocess.run(["hipcc"] + KERNEL_FLAGS + ["--cuda-device-only", "-S", str(src), "-o", str(asm)], check=True,
                   stderr=subprocess.DEVNULL)
    bad, kernels = [], 0
    for m in re.finditer(r"\n(sbz_\w+):[^\n]*\n(.*?)\n\.Lfunc_end", asm.read_text(), re.S):
        kernels += 1
        joins = set(re.findall(r"s_cbranch_execn?z (\.LBB\S+)", m.group(2)))
        for block in re.split(r"\n(?=\.LBB)", m.group(2)):
            label, _, body = block.partition(":")
            if label not in joins:
                continue
            head = []
            for line in body.split("\n")[1:]:
                t = line.split(";")[0].strip()
                if t.startswith("s_or_b64 exec, exec"):
                    if head and all(re.match(r"v_accvgpr|v_mov_b(32|64)\S* v\S+ v|scratch_", h) for h in head):
                        bad.append((m.group(1), label, head[0]))
                    break
                if re.match(r"s_cbranch|s_branch|s_endpgm|s_\w+ exec|s_\w+_saveexec", t):
                    break
                if t.startswith(("v_", "ds_", "global_", "scratch_")) and not t.startswith(("v_readlane", "v_writelane")):
                    head.append(t)
    assert kernels >= 8 and not bad, bad


@pytest.mark.gpu
@pytest.mark.parametrize("kw, n_k, lanes", [
    (dict(lmax=10, h=False), 1, 0), (dict(lmax=10, h=False), 33, 2), (dict(lmax=5), 7, 1), (dict(lmax=5), 17, 2),
    pytest.param(dict(lmax=4, nx=5), 9, 1, marks=pytest.mark.skip(
        reason="with 16 lanes per mode this comparison did not return on the device and the cause is not known; "
               "models with five momentum bins and more have no such kernel")),
    (dict(lmax_g=17, lmax_nu=4, lmax_h=3, nx=2), 9, 1)])
def test_gpu_group_kernel_matches_one_mode_kernel(kw, n_k, lanes):
    """Two sets on time grids of their own; `lanes` wavefronts, so that groups fill up and refill."""
    from symboltz.solver import ALGO_WAVE, SAVE_SOURCES, SAVE_STATES, SAVEAT_PER_SET, GpuModel
    M = models.LCDM(**kw)
    p = models.parameters_Planck18(M)
    gm = GpuModel(M)
    try:
        sets = [Setup(M, dict(p, h=h)) for h in (0.67, 0.7)]
        for i, S in enumerate(sets):
            gm.upload_background(i, S.t, S.u, S.du, S.P)
        ks = np.tile(np.geomspace(0.01, 300.0, n_k), 2)
        iset = np.repeat(np.arange(2, dtype=np.int32), n_k)
        t0 = np.array([np.clip(min(1e-2 / k, 1e-4), sets[i].t[0], 1.0) for k, i in zip(ks, iset)])
        rows = np.stack([np.linspace(0.05, 0.9 * S.t[-1], 11) for S in sets])
        out = {}
        for algo in (0, ALGO_WAVE):
            plan = gm.plan(iset, ks, t0, saveat=rows, lanes=lanes, save=SAVE_STATES | SAVE_SOURCES | SAVEAT_PER_SET,
                           algo=algo)
            plan.run()
            out[algo] = dict(plan.fetch(), src=plan.sources())
            plan.close()
        print(f"case: n = {M.n_unknowns}, 2 x {n_k} k, {lanes} wavefronts", flush=True)
        assert np.all(out[ALGO_WAVE]["retcode"] == 0)
        compare(out[0], out[ALGO_WAVE], len(ks))
        # without saves, repeated, and replayed from a graph: the same states
        plan = gm.plan(iset, ks, t0, lanes=lanes)
        plan.run()
        u = plan.fetch()["u"]
        assert np.max(np.abs(u - out[0]["u"]) / np.abs(u).max(axis=1, keepdims=True)) < TOL
        for _ in range(3):
            plan.run_graph()
            np.testing.assert_array_equal(plan.fetch()["u"], u)
        plan.close()
    finally:
        gm.close()


def test_emulated_group_tangent_with_two_instances_per_wavefront(massless10):
    """Four lanes per group, so two instances share a wavefront and one slot refills: u equals the plain
    kernel's, and s + f(τ0) dτ0/dlog θ the central difference of oracle solves at log θ ± h on the same tight
    backgrounds (1e-3, the bar that the 8-lane model's test holds to)."""
    from oracle import oracle
    from symboltz import _lib
    S = massless10
    E = WaveEmu(model_source(S.M).full_src)
    ks = np.array([0.5, 30.0, 4.0])
    t0 = np.clip(np.minimum(1e-2 / ks, 1e-4), S.t[0], S.t[-1])
    h, x, tight = 1e-3, np.log(S.pars["Omega_c0"]), []
    for sgn in (1, -1):
        P = models.make_params(S.M, dict(S.pars, Omega_c0=np.exp(x + sgn * h)))
        tight.append(_lib.background_solve(P, 1e-10, 1e-10, 100000)[:4])
    g = E.solve_tangent([(S.P, S.t, S.u, S.du)] + tight, ks, t0, 0.5 / h)
    g1 = E.solve(S.P, S.t, S.u, S.du, ks, t0)
    compare(dict(u=g["u"], retcode=g["retcode"], stats=g["stats"]), g1 | dict(usave=None, src=None), 3)
    fd = []
    for P, t, u, du in tight:
        o = oracle.Oracle(S.M, P, t, u, du).solve(ks, t0, rtol=1e-9, atol=1e-9, maxiters=10**6)
        assert np.all(o["retcode"] == 0)
        fd.append(o["u"])
    fd = (fd[0] - fd[1]) / (2 * h)
    s = g["s"] + g["fend"] * (tight[0][1][-1] - tight[1][1][-1]) / (2 * h)
    assert np.all(np.max(np.abs(s - fd), axis=1) < 1e-3 * np.abs(fd).max(axis=1))
