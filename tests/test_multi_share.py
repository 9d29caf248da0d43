"""Modes per entry of a mixed-model launch (csrc/sbz_multi_share.h): it ends for every mix of
families, empty ones among them, takes the fewest modes per wavefront that keep the entries resident,
and the launch gives the per-family results."""
import ctypes
import itertools
import subprocess

import numpy as np
import pytest

from symboltz import build

INTS = ctypes.POINTER(ctypes.c_int)


@pytest.fixture(scope="module")
def share(tmp_path_factory):
    d = tmp_path_factory.mktemp("share")
    (d / "s.cpp").write_text(f'#include "{build.CSRC / "sbz_multi_share.h"}"\nextern "C" void share(int n, const int* a, '
                             "const int* b, const int* c, int r, int* p) { sbz_multi_share(n, a, b, c, r, p); }\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(d / "s.cpp"), "-o", str(d / "s.so")], check=True)
    L = ctypes.CDLL(str(d / "s.so"))

    def call(fams, resident):
        cols = [np.array(c, dtype=np.int32) for c in zip(*fams)] + [np.zeros(len(fams), np.int32)]
        n_inst, rows, group, per = cols
        p = [c.ctypes.data_as(INTS) for c in cols]
        L.share(len(fams), p[0], p[1], p[2], resident, p[3])
        return [int(x) for x in per]
    return call


def by_definition(fams, resident):
    for s in range(1, 17):
        per = [1 if n == 0 or r == 1 else min(s, g) if g else r for n, r, g in fams]
        if sum(-(-n // q) for (n, _, _), q in zip(fams, per)) <= resident:
            break
    return per


@pytest.mark.parametrize("resident", [1, 64, 1024])
def test_share_is_the_smallest_that_keeps_the_entries_resident(share, resident):
    kinds = [(4, 16), (2, 8), (4, 0), (1, 0)]     # (rows, group): 4 and 8 lanes per mode, a row body, one mode
    for ns in itertools.product([0, 1, 17, 1024, 20000], repeat=3):
        for ks in itertools.product(kinds, repeat=3):
            fams = [(n, r, g) for n, (r, g) in zip(ns, ks)]
            assert share(fams, resident) == by_definition(fams, resident), (fams, resident)


@pytest.mark.gpu
def test_launch_with_more_entries_than_wavefronts_and_empty_families():
    """One family holds more modes than the wavefronts' groups, the other two hold none; a few attempts per
    mode (MaxIters) are enough: the states equal those of the family's own launch."""
    from conftest import Setup
    from symboltz import models
    from symboltz.multi import MultiModel
    from symboltz.solver import GpuModel
    fams = [models.LCDM(lmax=10, h=False), models.w0waCDM(lmax=6), models.LCDM(lmax=6)]
    gms = [GpuModel(M) for M in fams]
    mm = MultiModel(gms)
    plans = []
    try:
        S = Setup(fams[0])
        gms[0].upload_background(0, S.t, S.u, S.du, S.P)
        n = 17 * mm.capacity()
        ks = np.geomspace(0.1, 1000.0, n)
        t0 = np.clip(np.minimum(1e-2 / ks, 1e-4), S.t[0], S.t[-1])
        print(f"case: {n} modes of n = 38, two empty families, 4 attempts each", flush=True)
        plans = [gms[0].plan(np.zeros(n, np.int32), ks, t0, maxiters=4)]
        plans += [g.plan(np.zeros(0, np.int32), np.zeros(0), np.zeros(0)) for g in gms[1:]]
        mm.run(plans)
        got = plans[0].fetch()
        plans[0].run()
        ref = plans[0].fetch()
        assert np.all(got["retcode"] == 1)
        np.testing.assert_array_equal(got["retcode"], ref["retcode"])
        np.testing.assert_array_equal(got["u"], ref["u"])
    finally:
        for p in plans:
            p.close()
        mm.close()
        for g in gms:
            g.close()
