"""The host background solve takes all columns of its Jacobian from one evaluation, f at the stored
state and both again after a rejected attempt: every knot equals, bit for bit, that of the solve that evaluates
them anew column by column (the device's way, compiled for the host as the library was before, with errno set by
the math functions)."""
import ctypes
import subprocess

import numpy as np
import pytest

from symboltz import _lib, build, models

DP, IP = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)


@pytest.fixture(scope="module")
def anew(tmp_path_factory):
    d = tmp_path_factory.mktemp("bg")
    (d / "bg.cpp").write_text(f"""#include <hip/hip_runtime.h>
#include <cmath>
#define SBZ_BG_REUSE 0
#include "{build.CSRC / "sbz_bgsolve.h"}"
static_assert(SBZ_BG_REUSE == 0, "");
extern "C" int bg(double* P, double rt, double at, int n, double* t, double* u, double* du, int* nk, int* nr) {{
    double tf;
    return sbz_bg_solve(P, rt, at, n, t, u, du, nk, nr, &tf);
}}
""")
    subprocess.run(["hipcc", "-fPIC", "-shared", "-I", str(build.INCLUDE)] + build.HIP_FLAGS +
                   [str(d / "bg.cpp"), "-o", str(d / "bg.so")], check=True, stderr=subprocess.DEVNULL)
    L = ctypes.CDLL(str(d / "bg.so"))
    L.bg.argtypes = [DP, ctypes.c_double, ctypes.c_double, ctypes.c_int, DP, DP, DP, IP, IP]

    def solve(P, rtol, atol, n=20000):
        P, nk, nr = P.copy(), ctypes.c_int(), ctypes.c_int()
        t, u, du = np.zeros(n), np.zeros((n, 5)), np.zeros((n, 5))
        assert L.bg(_lib.ptr(P), rtol, atol, n, _lib.ptr(t), _lib.ptr(u), _lib.ptr(du), ctypes.byref(nk),
                    ctypes.byref(nr)) == 0
        return P, t[:nk.value], u[:nk.value], du[:nk.value], nr.value
    return solve


MODELS = [models.LCDM(lmax=5), models.LCDM(lmax=10, h=False), models.w0waCDM(lmax=6), models.LCDM(lmax=5, nu=False),
          models.LCDM(lmax=5, reionization=False), models.LCDM(lmax=5, Hswitch=0, Heswitch=0)]


@pytest.mark.parametrize("i", range(len(MODELS)))
def test_host_background_is_bit_for_bit_that_of_separate_evaluations(anew, i):
    M, rng = MODELS[i], np.random.default_rng(i)
    pars = models.parameters_Planck18(M)
    for tol in (1e-7, 1e-5, 1e-10):
        h = rng.uniform(0.6, 0.75)
        P = models.make_params(M, dict(pars, h=h, Omega_b0=rng.uniform(0.02, 0.024) / h**2,
                                       Omega_c0=rng.uniform(0.1, 0.14) / h**2))
        got, ref = _lib.background_solve(P, tol, tol, 20000), anew(P, tol, tol)
        assert got[4] == ref[4]
        for a, b in zip(got[:4], ref[:4]):
            np.testing.assert_array_equal(a, b)
