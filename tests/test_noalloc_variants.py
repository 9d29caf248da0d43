"""The no-allocation batch takes algo 0, the kernel variant of a plan by default, and says so where it refuses
another."""
import ctypes

import numpy as np
import pytest

from symboltz import _lib

pytestmark = pytest.mark.gpu


def test_noalloc_takes_algo_0_and_its_refusal_says_so(massless10):
    from symboltz.solver import ALGO_WAVE4, GpuModel, _Opts
    S = massless10
    gm = GpuModel(S.M)
    try:
        gm.upload_background(0, S.t, S.u, S.du, S.P)
        ks, t0, iset = np.array([1.0]), np.array([1e-4]), np.zeros(1, np.int32)
        u = np.zeros((1, gm.n))
        ret = np.zeros(1, np.int32)
        ip = ctypes.POINTER(ctypes.c_int)

        def call(algo):
            o = _Opts(1e-5, 1e-5, 100000, 0, 0, algo)
            return gm.L.sbz_solve_batch_noalloc(gm.h, _lib.ptr(iset, ctypes.c_int), _lib.ptr(ks), _lib.ptr(t0), 1,
                                                ctypes.byref(o), None, 0, _lib.ptr(u), None,
                                                ret.ctypes.data_as(ip), None)
        assert call(0) == 0 and ret[0] == 0 and np.all(np.isfinite(u))
        assert call(ALGO_WAVE4) != 0
        assert "algo 0" in gm.L.sbz_last_error().decode()
    finally:
        gm.close()
