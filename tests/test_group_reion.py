"""The reionization term of the kernels with one hierarchy per lane (sbz_greion of csrc/sbz_group.h)
and its τ-derivative far above the transition, where the exponent of its logistic form is large: finite,
and nothing beside x_e >= 1e-4."""
import ctypes

import numpy as np

from emu.emu import build
from symboltz import models
from symboltz.solver import model_source


def test_term_and_derivative_are_finite_for_every_exponent():
    src = model_source(models.LCDM(lmax=3, h=False)).full_src + """
extern "C" void emu_greion(double opz, double dopz, double kk, double fre, double n, double* out) {
    const Dual z(opz, dopz);
    const Dual r = sbz_greion<Dual>(z, sbz_sqrt(z), 1.08, fre, kk, n);
    out[0] = r.v;
    out[1] = r.d;
    out[2] = sbz_greion<double>(opz, sqrt(opz), 1.08, fre, kk, n);
}
"""
    L = ctypes.CDLL(str(build(src)))
    dp = ctypes.POINTER(ctypes.c_double)
    L.emu_greion.argtypes = [ctypes.c_double] * 5 + [dp]
    zre = 8.67
    for n in (1.0, 1.5):
        for width in (0.5, 1e-6, 1e-9):                          # in 1 + z
            kk = -2.0 / (n * zre**(n - 1) * width)               # -2K of tanh(K (f(z_re) - f(z)))
            for ex in (-40.0, 0.0, 40.0, 200.0, 299.0, 301.0, 400.0, 650.0, 689.0, 689.99, 691.0, 1e6):
                opz = (max(zre**n - ex / kk, 1.0)) ** (1 / n)    # the exponent is kk (f_re - f(z))
                o = np.zeros(3)
                L.emu_greion(opz, -opz * 14.0 * np.sqrt(opz), kk, zre**n, n, o.ctypes.data_as(dp))
                assert np.all(np.isfinite(o)) and o[0] == o[2], (n, width, ex, o)
                if ex >= 400.0:
                    assert 0.0 <= o[0] < 1e-100 and abs(o[1]) < 1e-100, (n, width, ex, o)
