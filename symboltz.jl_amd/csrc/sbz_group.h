// One hierarchy per lane: a mode is a group of SBZ_GL neighbouring lanes (4 or 8), so a
// wavefront integrates 64 / SBZ_GL modes with the same Rodas5P step as the other kernels.
//
// Lane s of a group holds one species' multipoles l = 0, 1, ... in registers (slot l): photon
// temperature (lane 0), photon polarization (lane 1), massless ν, each massive-ν momentum bin; the
// group's last lane holds the fluids and the potential in the slots
//   0: δ_c  1: θ_c  2: Φ  3: δ_b  4: θ_b  [5: δ_X  6: θ_X].
// In these slots every lane's own equations are tridiagonal, and the lanes couple only through
//   Φ' = p·u and Ψ = q·u (every row), Π_γ = F_2 + G_0 + G_2 (rows F_2, G_0, G_2): group sums, and
//   F_1 ↔ θ_b: one exchange between the group's first and last lane.
// W = I/(γh) - J is solved in that form: θ_b (with δ_b) is eliminated into F_1, every lane sweeps its
// tridiagonal system from the top multipole down and back up (every pivot stays ≥ 1/(γh)), and Π_γ,
// Φ', Ψ enter as a rank-3 Woodbury correction whose functionals read slots 0..2 (0..6 in the last
// lane), so the sweep back up over l ≥ 3 starts from the corrected values.
//
// The state, the stage inputs and the factors stay in registers; f_n and as many of ∂f/∂τ, K_1..K_4 as four
// workgroups per CU leave room for lie in LDS, one column per lane (SbzGVecs).  Lanes exchange nothing through
// LDS but the background, and there is no workgroup barrier inside the stages.  Lanes of 17 slots (n = 100) do
// not fit the registers: 752 B of scratch per lane, beside the moves to and from the accumulation registers.
//
// Bound by instruction issue: an attempt takes 5.1 k instructions at n = 54, 6.3 k at n = 38 and 9.1 k at
// n = 100 (2.2 k of them moves to and from the accumulation registers), a third of them FP64 multiply-adds, at
// five to six cycles each (eight at n = 100), however many of the groups work; the kernels of one and of several
// modes before took 33 to 58 us an attempt, at 39 % VALU, this one 13 to 33.  65,536 modes: n = 38 (128 sets x 512 k) 446 -> 66 ms,
// n = 100 (64 sets x 1024 k) 2,212 -> 332 ms.  100 modes of n = 38: 77 -> 39 ms.  Between those sizes, 2 and
// 12,000 modes from 1 to 2,000 H0/c against the faster of the kernels before: n = 59 (18 slots, 4 lanes) 57 / 73 and
// 65 / 77 ms, n = 89 (12 slots) 36 / 100 and 38 / 155 ms, n = 131 (18 slots, 8 lanes) 59 / 110 and 79 / 231 ms.
#pragma once

#ifndef SBZ_ALWAYS
#define SBZ_ALWAYS __attribute__((always_inline))
#endif
template <int V>
struct SbzInt { static constexpr int value = V; };

// 1/x to about one unit in the last place: the hardware estimate and two Newton steps (the IEEE
// division is a chain twice as long, and the pivots and weights it serves need no exact rounding).
SBZ_DEV double sbz_rcp(double x) {
#if defined(__AMDGCN__)
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
#else
    return 1.0 / x;
#endif
}

SBZ_DEV Dual sbz_rcp(Dual x) {
    const double r = sbz_rcp(x.v);
    return Dual(r, -x.d * (r * r));
}
// 1/sqrt(x), x > 0, to about one unit in the last place (estimate and two Newton steps)
SBZ_DEV double sbz_rsq(double x) {
#if defined(__AMDGCN__)
    double r = __builtin_amdgcn_rsq(x);
    const double hx = 0.5 * x;
    r = __builtin_fma(__builtin_fma(-hx * r, r, 0.5), r, r);
    return __builtin_fma(__builtin_fma(-hx * r, r, 0.5), r, r);
#else
    return 1.0 / sqrt(x);
#endif
}
SBZ_DEV Dual sbz_rsq(Dual x) {
    const double r = sbz_rsq(x.v);
    return Dual(r, -0.5 * x.d * (r * r * r));
}

// p ? x : y on values (a conditional of two lvalues would select addresses and keep them in memory)
SBZ_DEV double sbz_sel(bool p, double x, double y) { return p ? x : y; }
SBZ_DEV Dual sbz_sel(bool p, Dual x, Dual y) { return Dual(p ? x.v : y.v, p ? x.d : y.d); }

// Exchange between mirrored lanes of a group (lane i and GL - 1 - i) and the sum over a group,
// identical in each of its lanes (all 64 lanes active).
template <int GL>
SBZ_DEV double sbz_gmirror(double v) {
    return sbz_dpp<GL == 4 ? 0x1B : 0x141>(v);   // quad_perm [3,2,1,0], row_half_mirror
}
template <int GL>
SBZ_DEV double sbz_gsum(double v) {
    v += sbz_dpp<0xB1>(v);    // quad_perm [1,0,3,2]
    v += sbz_dpp<0x4E>(v);    // quad_perm [2,3,0,1]
    if constexpr (GL >= 8) v += sbz_dpp<0x141>(v);    // row_half_mirror
    return v;
}

// v of lane 0 plus v of lane 1, in these two lanes (Π_γ, which only their rows read)
SBZ_DEV double sbz_gpair(double v) { return v + sbz_dpp<0xB1>(v); }

// The background quantities the equations read at one time.
enum {
    SBZ_GB_KD, SBZ_GB_IT, SBZ_GB_HC, SBZ_GB_IH, SBZ_GB_A2, SBZ_GB_CS, SBZ_GB_RG, SBZ_GB_RN, SBZ_GB_RC, SBZ_GB_RB,
    SBZ_GB_IRB,
    SBZ_GB_FH,                                    // ρ_h / Iρ = (ρ_h + P_h) / (Iρ + I_P/3)
    SBZ_GB_E0 = SBZ_GB_FH + (SBZ_NX > 0),         // E_i, then 1/E_i
    SBZ_GB_X0 = SBZ_GB_E0 + 2 * SBZ_NX,           // ρ_X, w_X, 1/(1 + w_X), dw_X/dτ
    SBZ_NGB = SBZ_GB_X0 + 4 * SBZ_HAS_W0WA
};
// The set's constants of the background formulas (sbz_gconst), kept in LDS per group.
enum {
    SBZ_GC_RG, SBZ_GC_RN, SBZ_GC_RC, SBZ_GC_RB, SBZ_GC_IRB, SBZ_GC_RX, SBZ_GC_DE, SBZ_GC_W0, SBZ_GC_WA, SBZ_GC_T0,
    SBZ_GC_NH, SBZ_GC_KR, SBZ_GC_FHE, SBZ_GC_KD, SBZ_GC_KT, SBZ_GC_MU0, SBZ_GC_MU1, SBZ_GC_X1, SBZ_GC_F1, SBZ_GC_K1,
    SBZ_GC_N1, SBZ_GC_X2, SBZ_GC_F2, SBZ_GC_K2, SBZ_GC_N2, SBZ_GC_EHE,
    SBZ_GC_FH, SBZ_GC_Y0 = SBZ_GC_FH + (SBZ_NX > 0), SBZ_GC_BIN = SBZ_GC_Y0 + (SBZ_NX > 0),   // x_i², w_i
    SBZ_NGC = SBZ_GC_BIN + 2 * SBZ_NX
};
SBZ_DEV void sbz_gconst(const double* P, double* o) {
    using namespace sbzc;
    const double k38 = 3.0 / (8.0 * PI), h = P[SBZ_P_H], YHe = P[SBZ_P_YHE], fHe = P[SBZ_P_FHE], H0SI = H100 * h;
    const double cb = k38 * P[SBZ_P_OMB], cnh = (1.0 - YHe) * (H0SI * H0SI / GN / mH);
    const double ke = 2.0 * PI * me * kB / (hP * hP);          // λ_e^-2 = ke T_b
    o[SBZ_GC_RG] = k38 * P[SBZ_P_OMG];
    o[SBZ_GC_RN] = k38 * P[SBZ_P_OMNU];
    o[SBZ_GC_RC] = k38 * P[SBZ_P_OMC];
    o[SBZ_GC_RB] = cb;
    o[SBZ_GC_IRB] = 1.0 / cb;
    o[SBZ_GC_RX] = k38 * P[SBZ_P_OMDE];
    o[SBZ_GC_DE] = P[SBZ_P_DE];
    o[SBZ_GC_W0] = P[SBZ_P_W0];
    o[SBZ_GC_WA] = P[SBZ_P_WA];
    o[SBZ_GC_T0] = P[SBZ_P_T0];
    o[SBZ_GC_NH] = cnh;
    o[SBZ_GC_KR] = ke * sqrt(ke) / cnh;
    o[SBZ_GC_FHE] = fHe;
    o[SBZ_GC_KD] = -(sigmaT * c_) / H0SI * cnh;
    o[SBZ_GC_KT] = (8.0 / 3.0 * sigmaT * aR / H100) / (me * c_) / h;
    o[SBZ_GC_MU0] = kB / (mH * c_ * c_) * (1.0 + (mH / mHe - 1.0) * YHe);
    o[SBZ_GC_MU1] = kB / (mH * c_ * c_) * (1.0 - YHe);
    const double re = P[SBZ_P_REION] != 0.0 ? 1.0 : 0.0;
    o[SBZ_GC_X1] = re * (1.0 + fHe);
    o[SBZ_GC_F1] = P[SBZ_P_RE1F];
    o[SBZ_GC_K1] = -2.0 * P[SBZ_P_RE1K];
    o[SBZ_GC_N1] = P[SBZ_P_NRE1];
    o[SBZ_GC_X2] = re * fHe;
    o[SBZ_GC_F2] = P[SBZ_P_RE2F];
    o[SBZ_GC_K2] = -2.0 * P[SBZ_P_RE2K];
    o[SBZ_GC_N2] = P[SBZ_P_NRE2];
    o[SBZ_GC_EHE] = -EHep_inf_1s / kB;
    if constexpr (SBZ_NX > 0) {
        o[SBZ_GC_FH] = k38 * P[SBZ_P_OMH] / P[SBZ_P_IRHO0];
        o[SBZ_GC_Y0] = P[SBZ_P_Y0H];
#pragma unroll
        for (int i = 0; i < SBZ_NX; ++i) {
            o[SBZ_GC_BIN + 2 * i] = P[SBZ_P_X + i] * P[SBZ_P_X + i];
            o[SBZ_GC_BIN + 2 * i + 1] = P[SBZ_P_W + i];
        }
    }
}

// x_e of one reionization: ½ X (1 + tanh(K (f(z_re) - f(z)))) = X / (1 + exp(-2K (f(z_re) - f(z)))),
// f(z) = (1 + z)^n (kk = -2K; the exponent is capped where the term is below 1e-130, nothing beside x_e, and
// far from where the exponential times the exponent's τ-derivative, large for a narrow transition, overflows)
template <class T>
SBZ_DEV T sbz_greion(T opz, T sq, double xmax, double fre, double kk, double n) {
    T fz = (n == 1.5) ? sq * opz : opz;
    if (n != 1.5 && n != 1.0) fz = sbz_pow(opz, n);
    T ar = kk * (fre - fz);
    if (dval(ar) > 300.0) ar = T(300.0);
    return xmax * sbz_rcp(1.0 + sbz_exp(ar));
}

// The background row at time tau (T = double, or Dual for its τ-derivative): the values of
// sbz_pt_background in a form with few divisions (powers of 1/a, reciprocal square roots, the
// reionization terms as logistic functions) and without the quantities the groups do not read.
template <class T>
SBZ_DEV void sbz_gbg(const double* __restrict__ gc, const double* __restrict__ kt, int nk, int& idx, T tau, T* o) {
    const double* ku = kt + nk;
    const double* kdu = kt + 6 * (size_t)nk;
    const double tv = dval(tau);
    // the spline data of the cursor's interval and of the next in one round trip to memory: a step usually
    // crosses a knot in some lane, and to find the interval first would take three more, one after another.
    // Lanes of up to 12 slots only (128 x 512 massless 107 -> 101 ms): with 17 the registers are taken and
    // the saving kernel loses more than it gains (54.0 -> 55.1 ms).
    constexpr bool AHEAD = SBZ_GM <= 12;
    const int i2 = !AHEAD ? idx + 1 : idx + 2 < nk ? idx + 2 : nk - 1;
    double ta = kt[idx], tb = kt[idx + 1], ua[4], ub[4], da[4], db[4];
    const double tc = kt[i2];
    const bool next = AHEAD && idx < nk - 2 && tv >= tb && (idx + 1 >= nk - 2 || tv < tc);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double u0 = ku[idx * 5 + j], u1 = ku[(idx + 1) * 5 + j], u2 = ku[i2 * 5 + j];
        const double d0 = kdu[idx * 5 + j], d1 = kdu[(idx + 1) * 5 + j], d2 = kdu[i2 * 5 + j];
        ua[j] = sbz_sel(next, u1, u0);
        ub[j] = sbz_sel(next, u2, u1);
        da[j] = sbz_sel(next, d1, d0);
        db[j] = sbz_sel(next, d2, d1);
    }
    ta = sbz_sel(next, tb, ta);
    tb = sbz_sel(next, tc, tb);
    idx += next;
    if ((idx > 0 && tv < ta) || (idx < nk - 2 && tv >= tb)) {
        while (idx > 0 && tv < kt[idx]) --idx;
        while (idx < nk - 2 && tv >= kt[idx + 1]) ++idx;
        ta = kt[idx];
        tb = kt[idx + 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            ua[j] = ku[idx * 5 + j];
            ub[j] = ku[(idx + 1) * 5 + j];
            da[j] = kdu[idx * 5 + j];
            db[j] = kdu[(idx + 1) * 5 + j];
        }
    }
    const double hk = tb - ta, ihk = sbz_rcp(hk);
    const T x = (tau - ta) * ihk;
    T s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double dl = ub[j] - ua[j], ha = hk * da[j], hb = hk * db[j];
        s[j] = ua[j] + x * (ha + x * ((3.0 * dl - 2.0 * ha - hb) + x * (ha + hb - 2.0 * dl)));
    }
    const T a = s[0], ia = sbz_rcp(a), ia2 = ia * ia, ia3 = ia2 * ia, ia4 = ia2 * ia2, a2 = a * a;
    const T rg = gc[SBZ_GC_RG] * ia4, rn = gc[SBZ_GC_RN] * ia4, rc = gc[SBZ_GC_RC] * ia3, rb = gc[SBZ_GC_RB] * ia3;
    const T irb = gc[SBZ_GC_IRB] * (a2 * a);
    T tot = rg + rn + rc + rb;
    if constexpr (SBZ_NX > 0) {
        const T y = gc[SBZ_GC_Y0] * a, y2 = y * y, fh = gc[SBZ_GC_FH] * ia4;
        T Ir(0.0);
#pragma unroll
        for (int i = 0; i < SBZ_NX; ++i) {
            const T e2 = gc[SBZ_GC_BIN + 2 * i] + y2, IE = sbz_rsq(e2), E = e2 * IE;
            Ir = Ir + gc[SBZ_GC_BIN + 2 * i + 1] * E;
            o[SBZ_GB_E0 + i] = E;
            o[SBZ_GB_E0 + SBZ_NX + i] = IE;
        }
        tot = tot + fh * Ir;
        o[SBZ_GB_FH] = fh;
    }
    T rx(gc[SBZ_GC_RX]), wx(-1.0);
    if (gc[SBZ_GC_DE] == 1.0) {
        const double w0 = gc[SBZ_GC_W0], wa = gc[SBZ_GC_WA];
        rx = gc[SBZ_GC_RX] * sbz_pow(a, -3.0 * (1.0 + w0 + wa)) * sbz_exp(-3.0 * wa * (1.0 - a));
        wx = w0 + wa * (1.0 - a);
    }
    tot = (8.0 * sbzc::PI / 3.0) * (tot + rx);
    const T rs = sbz_rsq(tot), Hc = tot * rs * a, IH = rs * ia;
    const T dT = s[3], Tg = gc[SBZ_GC_T0] * ia, Tb = dT + Tg;
    const T rt = sbz_rsq(Tb);                         // T_b^-1/2
    const T R = sbz_exp(gc[SBZ_GC_EHE] * (rt * rt)) * (gc[SBZ_GC_KR] * (Tb * (Tb * rt))) * irb;   // Saha, He++
    const double fHe = gc[SBZ_GC_FHE];
    const T id = sbz_rcp((1.0 + fHe) + R), q = fHe * (R * id), z = 1.0 + 4.0 * (q * id);
    T Xe = s[1] + fHe * s[2] + 2.0 * (q * sbz_rcp(1.0 + z * sbz_rsq(z)));
    const T sq = ia * sbz_rsq(ia);
    Xe = Xe + sbz_greion(ia, sq, gc[SBZ_GC_X1], gc[SBZ_GC_F1], gc[SBZ_GC_K1], gc[SBZ_GC_N1]);
    Xe = Xe + sbz_greion(ia, sq, gc[SBZ_GC_X2], gc[SBZ_GC_F2], gc[SBZ_GC_K2], gc[SBZ_GC_N2]);
    const T Tg2 = Tg * Tg;
    const T DTb = -2.0 * (Tb * Hc) - (gc[SBZ_GC_KT] * a) * ((Tg2 * Tg2) * (Xe * (sbz_rcp((1.0 + fHe) + Xe) * dT)));
    o[SBZ_GB_KD] = (gc[SBZ_GC_KD] * a) * (Xe * rb);
    o[SBZ_GB_IT] = sbz_rcp(tau);
    o[SBZ_GB_HC] = Hc;
    o[SBZ_GB_IH] = IH;
    o[SBZ_GB_A2] = a2;
    o[SBZ_GB_CS] = (gc[SBZ_GC_MU0] + gc[SBZ_GC_MU1] * Xe) * (Tb - (1.0 / 3.0) * (DTb * IH));
    o[SBZ_GB_RG] = rg;
    o[SBZ_GB_RN] = rn;
    o[SBZ_GB_RC] = rc;
    o[SBZ_GB_RB] = rb;
    o[SBZ_GB_IRB] = irb;
    if constexpr (SBZ_HAS_W0WA) {
        const bool de = gc[SBZ_GC_DE] == 1.0;
        const T iw = sbz_rcp(1.0 + wx), wd = (-gc[SBZ_GC_WA]) * (a * Hc);
        o[SBZ_GB_X0] = rx;
        o[SBZ_GB_X0 + 1] = wx;
        o[SBZ_GB_X0 + 2] = sbz_sel(de, iw, T(0.0));
        o[SBZ_GB_X0 + 3] = sbz_sel(de, wd, T(0.0));
    }
}

// The same row from a background vector with τ-derivatives (B[i], dB[i]: a source background row).
SBZ_DEV void sbz_gb_row(const double* __restrict__ B, Dual* o) {
    auto get = [&](int i) SBZ_ALWAYS { return Dual(B[i], B[SBZ_NB + i]); };
    auto rec = [&](Dual x, int i) SBZ_ALWAYS { return Dual(B[i], -x.d * B[i] * B[i]); };   // 1/x, stored at i
    const Dual a = get(1), Hc = get(2), rb = get(8);
    o[SBZ_GB_KD] = get(3);
    o[SBZ_GB_IT] = rec(get(0), SBZ_B_ITAU);
    o[SBZ_GB_HC] = Hc;
    o[SBZ_GB_IH] = rec(Hc, SBZ_B_IHC);
    o[SBZ_GB_A2] = a * a;
    o[SBZ_GB_CS] = get(4);
    o[SBZ_GB_RG] = get(5);
    o[SBZ_GB_RN] = get(6);
    o[SBZ_GB_RC] = get(7);
    o[SBZ_GB_RB] = rb;
    o[SBZ_GB_IRB] = rec(rb, SBZ_B_IRB);
    if constexpr (SBZ_NX > 0) {
        o[SBZ_GB_FH] = get(9) * rec(get(11), SBZ_B_IIRHO);
#pragma unroll
        for (int i = 0; i < SBZ_NX; ++i) {
            const Dual E = get(16 + i);
            o[SBZ_GB_E0 + i] = E;
            o[SBZ_GB_E0 + SBZ_NX + i] = rec(E, SBZ_B_IE0 + i);
        }
    }
    if constexpr (SBZ_HAS_W0WA) {
        const Dual w = get(14);
        o[SBZ_GB_X0] = get(13);
        o[SBZ_GB_X0 + 1] = w;
        o[SBZ_GB_X0 + 2] = rec(w, SBZ_B_IWX1);
        o[SBZ_GB_X0 + 3] = get(15);
    }
}

// The step's vectors f_n, ∂f/∂τ, K1..K4: as many of the first as four workgroups per CU leave room for
// lie in LDS (one column per lane).  Those past the 256 directly addressable registers cost two moves
// per access otherwise.
#ifndef SBZ_GLDS
#define SBZ_GLDS 40960   // LDS of a workgroup: four fit a CU's 160 KB
#endif
struct SbzGroupFixed {
    double gb[64 / SBZ_GL][6][SBZ_NGB];    // background at t_n, at the stage times c_2..c_5 and at t + h
    double dgb[64 / SBZ_GL][2][SBZ_NGB];   // its τ-derivative at t_n and at t + h
    double gc[64 / SBZ_GL][SBZ_NGC];
    int mode[64 / SBZ_GL];
};
constexpr int sbz_gkl(int room) {
    const int n = room / (64 * SBZ_GM * 8);
    return n > 6 ? 6 : n;
}
constexpr int SBZ_GKL = sbz_gkl(SBZ_GLDS - (int)sizeof(SbzGroupFixed));   // vectors in LDS
static_assert(SBZ_GKL >= 1, "f_n lies in LDS");
// a starting mode's scratch, in the vectors after f_n: its constants, a state and its derivative
constexpr int SBZ_GSTART = SBZ_NC + 2 * SBZ_N;
constexpr int SBZ_GST = 64 * SBZ_GM + (64 / SBZ_GL) * SBZ_GSTART;
static_assert(5 * SBZ_NGB >= SBZ_NB && SBZ_NCHAIN <= SBZ_GL, "a starting mode's background and chains fit its group");
struct SbzGroupLDS {
    SbzGroupFixed f;
    double kv[SBZ_GKL * SBZ_GM * 64 > SBZ_GST ? SBZ_GKL * SBZ_GM * 64 : SBZ_GST];
};
// Vector j of a lane (0: f_n, 1: ∂f/∂τ, 1 + s: K_s): in LDS when there is room, else in registers.
struct SbzGVecs {
    double* kv;
    double r[SBZ_GKL < 6 ? 6 - SBZ_GKL : 1][SBZ_GM];
    template <int J>
    SBZ_DEV double get(int l) const {
        if constexpr (J < SBZ_GKL) return kv[(J * SBZ_GM + l) * 64];
        else return r[J - SBZ_GKL][l];
    }
    template <int J>
    SBZ_DEV void set(int l, double x) {
        if constexpr (J < SBZ_GKL) kv[(J * SBZ_GM + l) * 64] = x;
        else r[J - SBZ_GKL][l] = x;
    }
};

// A lane's role in its group and its mode's constants.
struct SbzGCtx {
    int lane, g, kind, L, bin;             // kind 0: F, 1: G, 2: massless ν, 3: massive-ν bin, 4: fluids and Φ, 5: empty
    bool isF, isG, isN, isH, isO;
    double k, ik, ik2, k2;
    double mF, mG, mN, one;                // 1 in the lane of F, G, ν and in the last lane, else 0
    double w0, w2;                         // a massive-ν bin's weight, and weight x² (0 elsewhere)
    double sk0, skE, be0, beE, m1;         // s k = sk0 + skE / E; row 1's Ψ entry be0 + beE E; slip in F_1 over κ̇
    double al0, al2, al3;                  // constant entries of α
    double pi0, pi2;                       // Π_γ = Σ pi0 u_0 + pi2 u_2
    double cs2x;
};

// The coefficients of a lane's rows at one time (T = double, or Dual with the τ-derivatives).
template <class T>
struct SbzGCoef {
    T sk, dd, dd0, d1, top, a01;           // tridiagonal part
    T p0, p2, p3, q2;                      // Φ' and Ψ functionals
    T be1, ga0, ga2, m1, m4;               // rows' Ψ and Π_γ entries; slip θ_b - θ_γ in F_1 and θ_b
    T o33, o43;                            // δ_b, θ_b block
    T x55, x56, x65, x66, al5, p5;         // w0wa block
};

template <class T, class LD>
SBZ_DEV void sbz_gcoef(const SbzGCtx& c, LD ld, SbzGCoef<T>& C) {
    const T kd = ld(SBZ_GB_KD), Hc = ld(SBZ_GB_HC), A2 = ld(SBZ_GB_A2), IH = ld(SBZ_GB_IH);
    const T rg = ld(SBZ_GB_RG), cs = ld(SBZ_GB_CS);
    const T c1 = (-4.0 / 3.0 * sbzc::PI) * (A2 * IH);
    const T cq = (-8.0 * sbzc::PI * c.ik2) * A2;
    // what another lane holds enters with a factor 0: one instruction where a select takes two
    T r2 = c.mF * rg + c.mN * ld(SBZ_GB_RN);
    T r0 = r2 + c.one * ld(SBZ_GB_RC);
    C.sk = T(c.sk0);
    C.be1 = T(c.be0);
    if constexpr (SBZ_NX > 0) {
        const T E = ld(SBZ_GB_E0 + c.bin), IE = ld(SBZ_GB_E0 + SBZ_NX + c.bin), fh = ld(SBZ_GB_FH);
        r0 = r0 + fh * (c.w0 * E);
        r2 = r2 + fh * (c.w2 * IE);
        C.sk = C.sk + c.skE * IE;
        C.be1 = C.be1 + c.beE * E;
    }
    C.q2 = c.one + cq * r2;
    C.p0 = c1 * r0;
    C.p2 = -(Hc * C.q2) - (c.one * c.k2 * (1.0 / 3.0)) * IH;
    C.p3 = c.one * (c1 * ld(SBZ_GB_RB));
    C.a01 = C.sk + c.one;
    C.dd0 = c.mG * kd;
    C.dd = C.dd0 + c.mF * kd;
    C.d1 = C.dd0 - c.one * Hc;
    C.top = C.dd - (c.L + 1.0) * ld(SBZ_GB_IT);
    C.ga0 = -0.5 * C.dd0;
    C.ga2 = -0.1 * C.dd;
    C.m1 = c.m1 * kd;
    const T kr = c.one * (kd * (rg * ld(SBZ_GB_IRB)));
    C.m4 = (4.0 / 3.0) * kr;
    C.o33 = (-3.0 * c.one) * (Hc * cs);
    C.o43 = (c.one * c.k2) * cs;
    if constexpr (SBZ_HAS_W0WA) {
        const T w = ld(SBZ_GB_X0 + 1), iw = ld(SBZ_GB_X0 + 2), w1 = 1.0 + w;
        const T ca2 = w - (1.0 / 3.0) * (ld(SBZ_GB_X0 + 3) * (IH * iw));
        C.x55 = (-3.0 * c.one) * (Hc * (c.cs2x - w));
        C.x56 = -(c.one * w1) - (9.0 * c.one * c.ik2) * ((Hc * Hc) * (w1 * (c.cs2x - ca2)));
        C.x65 = (c.one * c.cs2x * c.k2) * iw;
        C.x66 = -(c.one * (1.0 - 3.0 * c.cs2x)) * Hc;
        C.al5 = (3.0 * c.one) * w1;
        C.p5 = c.one * (c1 * ld(SBZ_GB_X0));
    }
}

// The coefficients without their derivatives.
SBZ_DEV void sbz_gvalues(const SbzGCoef<Dual>& D, SbzGCoef<double>& C) {
    C.sk = D.sk.v; C.dd = D.dd.v; C.dd0 = D.dd0.v; C.d1 = D.d1.v; C.top = D.top.v; C.a01 = D.a01.v;
    C.p0 = D.p0.v; C.p2 = D.p2.v; C.p3 = D.p3.v; C.q2 = D.q2.v;
    C.be1 = D.be1.v; C.ga0 = D.ga0.v; C.ga2 = D.ga2.v; C.m1 = D.m1.v; C.m4 = D.m4.v;
    C.o33 = D.o33.v; C.o43 = D.o43.v;
    if constexpr (SBZ_HAS_W0WA) {
        C.x55 = D.x55.v; C.x56 = D.x56.v; C.x65 = D.x65.v; C.x66 = D.x66.v; C.al5 = D.al5.v; C.p5 = D.p5.v;
    }
}

// s k of the rows l (0 past the end of a shorter hierarchy): sk[seg(l)]
SBZ_DEV constexpr int sbz_gseg(int l) {
    int s = 0;
    for (int i = 0; i < SBZ_GNTOP; ++i) s += l > sbz_gtops[i];
    return s < SBZ_GNTOP ? s : SBZ_GNTOP - 1;
}
SBZ_DEV constexpr bool sbz_gtop(int l) {
    for (int i = 0; i < SBZ_GNTOP; ++i)
        if (l == sbz_gtops[i]) return true;
    return false;
}
SBZ_DEV constexpr double sbz_grl(int l) { return l / (2.0 * l + 1.0); }
SBZ_DEV constexpr double sbz_grl1(int l) { return (l + 1.0) / (2.0 * l + 1.0); }
SBZ_DEV void sbz_gsk(const SbzGCtx& c, double sk, double* skm) {
    skm[0] = sk;
#pragma unroll
    for (int i = 1; i < SBZ_GNTOP; ++i) skm[i] = sbz_sel(c.L > sbz_gtops[i - 1], sk, 0.0);
}

// f = J u (ADD: f += J u): the rows of a lane.  Psi and Pig return Ψ and (in the group's lanes 0 and 1) Π_γ.
template <bool ADD>
SBZ_DEV void sbz_grhs(const SbzGCtx& c, const SbzGCoef<double>& C, const double* u, double* f, double& Psi, double& Pig) {
    constexpr int M = SBZ_GM, GL = SBZ_GL;
    // θ_b - θ_γ (θ_γ = ¾ k F_1): the same number in both lanes, so what F_1 loses to the drag θ_b gains
    // to rounding of the difference, not of its large terms
    const double own = sbz_sel(c.isO, u[4], u[1]), mir = sbz_gmirror<GL>(own);
    const double slip = __builtin_fma(-0.75 * c.k, sbz_sel(c.isO, mir, own), sbz_sel(c.isO, own, mir));
    double fp = C.p0 * u[0] + C.p2 * u[2] + C.p3 * u[3];
    if constexpr (SBZ_HAS_W0WA) fp += C.p5 * u[5];
    const double dPhi = sbz_gsum<GL>(fp);
    Psi = sbz_gsum<GL>(C.q2 * u[2]);
    Pig = sbz_gpair(c.pi0 * u[0] + c.pi2 * u[2]);
    double skm[SBZ_GNTOP];
    sbz_gsk(c, C.sk, skm);
    auto row = [&](int l, double x) SBZ_ALWAYS {
        if constexpr (ADD) f[l] += x;
        else f[l] = x;
    };
    row(0, C.dd0 * u[0] - C.a01 * u[1] + c.al0 * dPhi + C.ga0 * Pig);
    row(1, C.d1 * u[1] + C.sk * (1.0 / 3.0 * u[0] - 2.0 / 3.0 * u[2]) + C.be1 * Psi + C.m1 * slip);
    row(2, C.dd * u[2] + C.sk * (2.0 / 5.0 * u[1] - 3.0 / 5.0 * u[3]) + c.al2 * dPhi + C.ga2 * Pig);
#pragma unroll
    for (int l = 3; l < M; ++l) {
        const double sk = skm[sbz_gseg(l)];
        double x = sbz_grl(l) * u[l - 1];
        if (l + 1 < M) x -= sbz_grl1(l) * u[l + 1];
        if (sbz_gtop(l)) {
            const bool t = c.L == l;
            row(l, sbz_sel(t, C.top, C.dd) * u[l] + sk * sbz_sel(t, u[l - 1], x));
        } else {
            row(l, C.dd * u[l] + sk * x);
        }
    }
    f[3] += C.o33 * u[3] - c.one * u[4] + c.al3 * dPhi;
    f[4] += C.o43 * u[3] + C.d1 * (c.one * u[4]) + (c.one * c.k2) * Psi + C.m4 * slip;
    if constexpr (SBZ_HAS_W0WA) {
        f[5] += C.x55 * u[5] + C.x56 * u[6] + C.al5 * dPhi;
        f[6] += C.x65 * u[5] + C.x66 * u[6] + (c.one * c.k2) * Psi;
    }
}

// out = ∂f/∂τ at fixed u; dPsi returns (∂q/∂τ)·u.
SBZ_DEV void sbz_gdfdt(const SbzGCtx& c, const SbzGCoef<Dual>& C, const double* u, double* out, double& dPsi) {
    constexpr int M = SBZ_GM, GL = SBZ_GL;
    const double own = sbz_sel(c.isO, u[4], u[1]), mir = sbz_gmirror<GL>(own);
    const double slip = __builtin_fma(-0.75 * c.k, sbz_sel(c.isO, mir, own), sbz_sel(c.isO, own, mir));
    double fp = C.p0.d * u[0] + C.p2.d * u[2] + C.p3.d * u[3], fv = C.p0.v * u[0] + C.p2.v * u[2] + C.p3.v * u[3];
    if constexpr (SBZ_HAS_W0WA) {
        fp += C.p5.d * u[5];
        fv += C.p5.v * u[5];
    }
    const double ddPhi = sbz_gsum<GL>(fp), Psi = sbz_gsum<GL>(C.q2.v * u[2]);
    dPsi = sbz_gsum<GL>(C.q2.d * u[2]);
    const double Pig = sbz_gpair(c.pi0 * u[0] + c.pi2 * u[2]);
    double skm[SBZ_GNTOP];
    sbz_gsk(c, C.sk.d, skm);
    out[0] = C.dd0.d * u[0] - C.a01.d * u[1] + c.al0 * ddPhi + C.ga0.d * Pig;
    out[1] = C.d1.d * u[1] + C.sk.d * (1.0 / 3.0 * u[0] - 2.0 / 3.0 * u[2]) + C.be1.v * dPsi + C.be1.d * Psi + C.m1.d * slip;
    out[2] = C.dd.d * u[2] + C.sk.d * (2.0 / 5.0 * u[1] - 3.0 / 5.0 * u[3]) + c.al2 * ddPhi + C.ga2.d * Pig;
#pragma unroll
    for (int l = 3; l < M; ++l) {
        const double sk = skm[sbz_gseg(l)];
        const double up = (l + 1 < M) ? u[l + 1] : 0.0;
        if (sbz_gtop(l)) {
            const bool t = c.L == l;
            out[l] = sbz_sel(t, C.top.d, C.dd.d) * u[l] + sk * sbz_sel(t, u[l - 1], sbz_grl(l) * u[l - 1] - sbz_grl1(l) * up);
        } else {
            out[l] = C.dd.d * u[l] + sk * (sbz_grl(l) * u[l - 1] - sbz_grl1(l) * up);
        }
    }
    out[3] += C.o33.d * u[3] + c.al3 * ddPhi;
    out[4] += C.o43.d * u[3] + C.d1.d * (c.one * u[4]) + (c.one * c.k2) * dPsi + C.m4.d * slip;
    if constexpr (SBZ_HAS_W0WA) {
        const double dPhi = sbz_gsum<GL>(fv);
        out[5] += C.x55.d * u[5] + C.x56.d * u[6] + C.al5.v * ddPhi + C.al5.d * dPhi;
        out[6] += C.x65.d * u[5] + C.x66.d * u[6] + (c.one * c.k2) * dPsi;
    }
}

// Factor of u_{l-1} in row l over s k: l/(2l+1), and 1 in a hierarchy's last row.
SBZ_DEV double sbz_gca(const SbzGCtx& c, int l) { return sbz_gtop(l) ? sbz_sel(c.L == l, 1.0, sbz_grl(l)) : sbz_grl(l); }

// Lanes of up to 12 slots keep both sweeps' factors of a row, longer ones, short of registers, s k / d_l.
constexpr bool SBZ_GKEEP = SBZ_GM <= 12;

// The factored W of a lane.
constexpr int SBZ_GNB = SBZ_HAS_W0WA ? 7 : 5;   // slots the Woodbury correction reaches
struct SbzGFac {
    double cinv[SBZ_GM];                   // reciprocal pivots of the downward elimination
    double cs[SBZ_GM];                     // s k / d_l (rows l >= 3), times (l - 1's) l/(2l-1) of the downward sweep
    double cb[SBZ_GKEEP ? SBZ_GM : 1];     // the same times l/(2l+1) (1 in the last row), of the sweep back up
    double g0, g1, h1, h2;                 // the couplings of the rows 0..2, over their pivots
    double m1, m4D, o43, i3, iD;           // F_1 ↔ θ_b, and the (δ_b, θ_b) block
    double i5, x65, x56i5, iD6;            // the (δ_X, θ_X) block
    double p0, p2, p3, p5, q2;
    double zg[SBZ_GNB], za[SBZ_GNB], zb[SBZ_GNB];   // A^-1 γ, A^-1 α, A^-1 β (A: with Π_γ for the last two)
    double icg, pg, qg, c11, c12, c21, c22;
};

// T^-1 on the slots 0..2 and the last lane's block, given slots l ≥ 3 already swept down into b[2];
// y[0..NB) receives the solution (slots 3.. in the last lane only).
SBZ_DEV void sbz_gborder(const SbzGCtx& c, const SbzGFac& F, const double* b, double* y) {
    constexpr int GL = SBZ_GL;
    const double r3 = b[3] * F.i3, y4 = (b[4] + F.o43 * r3) * F.iD;
    const double t4 = sbz_gmirror<GL>(y4);
    const double b1 = b[1] - F.g1 * b[2] + F.m1 * t4;
    const double b0 = b[0] - F.g0 * b1;
    y[0] = b0 * F.cinv[0];
    y[1] = b1 * F.cinv[1] + F.h1 * y[0];
    y[2] = b[2] * F.cinv[2] + F.h2 * y[1];
    y[4] = y4 + F.m4D * sbz_gmirror<GL>(y[1]);
    y[3] = r3 - F.i3 * (c.one * y[4]);
    if constexpr (SBZ_HAS_W0WA) {
        const double r5 = b[5] * F.i5;
        y[6] = (b[6] + F.x65 * r5) * F.iD6;
        y[5] = r5 + F.x56i5 * y[6];
    }
}
SBZ_DEV double sbz_gp(const SbzGFac& F, const double* y) {
    double s = F.p0 * y[0] + F.p2 * y[2] + F.p3 * y[3];
    if constexpr (SBZ_HAS_W0WA) s += F.p5 * y[5];
    return s;
}

// W = ig I - J at t_n, factored (C: the coefficients there).
SBZ_DEV void sbz_gfactor(const SbzGCtx& c, const SbzGCoef<double>& C, double ig, SbzGFac& F) {
    constexpr int M = SBZ_GM, GL = SBZ_GL;
    double skm[SBZ_GNTOP];
    sbz_gsk(c, C.sk, skm);
    // θ_b eliminated into F_1: the pivots of δ_b and of θ_b, D = ig + ℋ - κ̇R + c_s²k² / (ig + 3ℋc_s²) with
    // κ̇R = m4; the damping of F_1 by κ̇ less its part carried along by θ_b, -κ̇ - κ̇²R / D =
    // -κ̇ (D + κ̇R) / D, in this form without cancellation
    F.i3 = sbz_rcp(ig - C.o33);
    const double e = ig - c.one * C.d1 + C.o43 * F.i3;     // D + κ̇R
    F.iD = sbz_rcp(e - C.m4);
    F.o43 = C.o43;
    F.m1 = C.m1;
    F.m4D = (-0.75 * c.k) * (C.m4 * F.iD);
    const double fr = sbz_gmirror<GL>(e * F.iD);
    double cb = 0.0;
    // d_l = ig - J[l][l] + (s k)² (l+1)/(2l+1) (l+1)/(2l+3) / d_{l+1}, from the top multipole down
#pragma unroll
    for (int l = M - 1; l >= 3; --l) {
        const double sk = skm[sbz_gseg(l)];
        double cd = C.dd;
        if (sbz_gtop(l)) cd = sbz_sel(c.L == l, C.top, cd);
        double d = ig - cd;
        if (l + 1 < M) d += (sk * sbz_grl1(l)) * cb;
        F.cinv[l] = sbz_rcp(d);
        const double cs = sk * F.cinv[l];
        cb = sbz_gca(c, l) * cs;
        if constexpr (SBZ_GKEEP) {
            F.cs[l] = sbz_grl1(l - 1) * cs;
            F.cb[l] = cb;
        } else {
            F.cs[l] = cs;
        }
    }
    F.cinv[2] = sbz_rcp(ig - C.dd + (C.sk * (3.0 / 5.0)) * cb);
    F.g1 = (2.0 / 3.0 * C.sk) * F.cinv[2];
    F.h2 = (2.0 / 5.0 * C.sk) * F.cinv[2];
    F.cinv[1] = sbz_rcp(ig - sbz_sel(c.isF, C.dd * fr, C.d1) + (2.0 / 3.0 * C.sk) * F.h2);
    F.g0 = C.a01 * F.cinv[1];
    F.h1 = (1.0 / 3.0 * C.sk) * F.cinv[1];
    F.cinv[0] = sbz_rcp(ig - C.dd0 + C.a01 * F.h1);
    if constexpr (SBZ_HAS_W0WA) {
        F.i5 = sbz_rcp(ig - C.x55);
        F.x65 = C.x65;
        F.x56i5 = C.x56 * F.i5;
        F.iD6 = sbz_rcp(ig - C.x66 - C.x65 * F.x56i5);
        F.p5 = C.p5;
    }
    F.p0 = C.p0;
    F.p2 = C.p2;
    F.p3 = C.p3;
    F.q2 = C.q2;
    double b[SBZ_GNB] = {};
    b[0] = C.ga0;
    b[2] = C.ga2;
    sbz_gborder(c, F, b, F.zg);
    b[0] = c.al0;
    b[2] = c.al2;
    b[3] = c.al3;
    if constexpr (SBZ_HAS_W0WA) b[5] = C.al5;
    sbz_gborder(c, F, b, F.za);
#pragma unroll
    for (int j = 0; j < SBZ_GNB; ++j) b[j] = 0.0;
    b[1] = C.be1;
    b[4] = c.one * c.k2;
    if constexpr (SBZ_HAS_W0WA) b[6] = c.one * c.k2;
    sbz_gborder(c, F, b, F.zb);
    const double gg = sbz_gsum<GL>(c.pi0 * F.zg[0] + c.pi2 * F.zg[2]);
    const double ga = sbz_gsum<GL>(c.pi0 * F.za[0] + c.pi2 * F.za[2]);
    const double gb = sbz_gsum<GL>(c.pi0 * F.zb[0] + c.pi2 * F.zb[2]);
    F.pg = sbz_gsum<GL>(sbz_gp(F, F.zg));
    F.qg = sbz_gsum<GL>(F.q2 * F.zg[2]);
    double pa = sbz_gsum<GL>(sbz_gp(F, F.za)), qa = sbz_gsum<GL>(F.q2 * F.za[2]);
    double pb = sbz_gsum<GL>(sbz_gp(F, F.zb)), qb = sbz_gsum<GL>(F.q2 * F.zb[2]);
    F.icg = 1.0 / (1.0 - gg);
    const double ta = ga * F.icg, tb = gb * F.icg;
#pragma unroll
    for (int j = 0; j < SBZ_GNB; ++j) {
        F.za[j] += ta * F.zg[j];
        F.zb[j] += tb * F.zg[j];
    }
    const double c11 = 1.0 - (pa + ta * F.pg), c12 = -(pb + tb * F.pg);
    const double c21 = -(qa + ta * F.qg), c22 = 1.0 - (qb + tb * F.qg);
    const double idet = 1.0 / (c11 * c22 - c12 * c21);
    F.c11 = c22 * idet;
    F.c12 = -c12 * idet;
    F.c21 = -c21 * idet;
    F.c22 = c11 * idet;
}

// b <- W^-1 b
SBZ_DEV void sbz_gsolve(const SbzGCtx& c, const SbzGFac& F, double* b) {
    constexpr int M = SBZ_GM, GL = SBZ_GL, NB = SBZ_GNB;
    double o[NB];   // the last lane's own right-hand side (its slots ≥ 3 are not a hierarchy)
#pragma unroll
    for (int j = 0; j < NB; ++j) o[j] = b[j];
#pragma unroll
    for (int l = M - 1; l >= 3; --l) b[l - 1] -= SBZ_GKEEP ? F.cs[l] * b[l] : sbz_grl1(l - 1) * (F.cs[l] * b[l]);
    o[2] = b[2];
    double y[NB];
    sbz_gborder(c, F, o, y);
    const double sg = sbz_gsum<GL>(c.pi0 * y[0] + c.pi2 * y[2]);
    const double sp = sbz_gsum<GL>(sbz_gp(F, y)), sq = sbz_gsum<GL>(F.q2 * y[2]);
    const double t = sg * F.icg, s1 = sp + F.pg * t, s2 = sq + F.qg * t;
    const double xa = F.c11 * s1 + F.c12 * s2, xb = F.c21 * s1 + F.c22 * s2;
#pragma unroll
    for (int j = 0; j < NB; ++j) y[j] += F.zg[j] * t + F.za[j] * xa + F.zb[j] * xb;
#pragma unroll
    for (int l = 0; l < 3; ++l) b[l] = y[l];
#pragma unroll
    for (int l = 3; l < M; ++l) {
        if constexpr (SBZ_GKEEP) b[l] = b[l] * F.cinv[l] + F.cb[l] * b[l - 1];
        else b[l] = b[l] * F.cinv[l] + F.cs[l] * (sbz_gca(c, l) * b[l - 1]);
        if (l < NB) b[l] = sbz_sel(c.isO, y[l], b[l]);
    }
}

// State component of a lane's slot (-1: none).
SBZ_DEV int sbz_gcomp(const SbzGCtx& c, int l) { return sbz_g_comp[c.lane * SBZ_GM + l]; }

SBZ_DEV SbzGCtx sbz_gctx() {
    SbzGCtx c;
    c.lane = threadIdx.x & (SBZ_GL - 1);
    c.g = threadIdx.x / SBZ_GL;
    c.kind = sbz_g_kind[c.lane];
    c.L = sbz_g_L[c.lane];
    c.bin = sbz_g_bin[c.lane];
    c.isF = c.kind == 0;
    c.isG = c.kind == 1;
    c.isN = c.kind == 2;
    c.isH = c.kind == 3;
    c.isO = c.kind == 4;
    c.one = c.isO ? 1.0 : 0.0;
    c.mF = c.isF ? 1.0 : 0.0;
    c.mG = c.isG ? 1.0 : 0.0;
    c.mN = c.isN ? 1.0 : 0.0;
    c.pi0 = c.isG ? 1.0 : 0.0;
    c.pi2 = (c.isF || c.isG) ? 1.0 : 0.0;
    return c;
}
// the constants of wavenumber k in the set P
SBZ_DEV void sbz_gmode(SbzGCtx& c, const double* P, double k) {
    c.k = k;
    c.ik = 1.0 / k;
    c.k2 = k * k;
    c.ik2 = 1.0 / c.k2;
    const double x = c.isH ? P[SBZ_P_X + c.bin] : 0.0;      // momentum of a massive-ν bin
    const double dl = c.isH ? -x / (1.0 + exp(-x)) : 0.0;   // d ln f0 / d ln x
    c.w0 = c.isH ? P[SBZ_P_W + c.bin] : 0.0;
    c.w2 = c.w0 * x * x;
    c.sk0 = (c.isF || c.isG || c.isN) ? k : 0.0;
    c.skE = k * x;
    c.be0 = (c.isF || c.isN) ? 4.0 / 3.0 * k : c.isO ? c.k2 : 0.0;
    c.beE = c.isH ? -1.0 / 3.0 * k * dl / x : 0.0;
    c.m1 = c.isF ? -4.0 / 3.0 * c.ik : 0.0;
    c.al0 = (c.isF || c.isN) ? 4.0 : c.isH ? -dl : 3.0 * c.one;
    c.al2 = c.one;
    c.al3 = 3.0 * c.one;
    c.cs2x = P[SBZ_P_CS2X];
}

// The groups of one wavefront integrate instances pulled from a's queue until it is empty.  With
// SAVE, saved states and CMB sources too (the sources' background from a.srcbg).
template <bool SAVE>
SBZ_DEV void sbz_group_run(const SbzSolveArgs& a, SbzGroupLDS& S) {
    constexpr int GL = SBZ_GL, NG = 64 / GL, M = SBZ_GM;
    SbzGCtx c = sbz_gctx();
    double (*const gb)[SBZ_NGB] = S.f.gb[c.g];
    double (*const dgb)[SBZ_NGB] = S.f.dgb[c.g];
    double* const gc = S.f.gc[c.g];
    SbzGVecs V;
    V.kv = S.kv + threadIdx.x;   // this lane's columns in LDS
    // a launch with fewer instances than groups spreads them over its wavefronts: each takes no more
    // than its share, the step time of a wavefront does not depend on how many of its groups work
    const int share = (a.n_inst + a.S - 1) / a.S;
    // per-group state; a group without a mode keeps a valid set's tables so its steps stay finite
    bool have = false, exhausted = c.g >= share;
    int inst = 0;
    int set = a.inst_set[a.order ? a.order[0] : 0];
    const double* P = a.params + (size_t)set * SBZ_NPAR;
    const double* kt = a.knots + a.knot_off[set];
    int nk = a.knot_n[set];
    double t = kt[0], t1 = kt[nk - 1], dt = 1e-3 * (kt[nk - 1] - kt[0]);
    int bidx = 0, bidx2 = 0;
    long long iters = 0;
    int st_acc = 0, st_rej = 0, st_f = 0, st_j = 0;
    int ret = SBZ_RET_SUCCESS;
    const double lq0 = log(SBZ_CTL_QOLDINIT);
    double lqold = lq0;   // log of the last accepted error estimate (PI controller)
    int isave = 0;
    const double* saveat = nullptr;
    double u[M];
#pragma unroll
    for (int l = 0; l < M; ++l) {
        u[l] = 0.0;
        V.set<0>(l, 0.0);
    }
    sbz_gmode(c, P, 1.0);
    if (c.lane == 0) sbz_gconst(P, gc);
    auto finish = [&]() SBZ_ALWAYS {
        double* o = a.out_u + (size_t)inst * SBZ_N;
#pragma unroll
        for (int l = 0; l < M; ++l) {
            const int q = sbz_gcomp(c, l);
            if (q >= 0) o[q] = u[l];
        }
        if (c.lane == 0) {
            a.retcode[inst] = ret;
            long long* st = a.stats + (size_t)inst * 6;
            st[0] = st_acc;
            st[1] = st_rej;
            st[2] = st_f;
            st[3] = st_j;
            st[4] = st_j;
            st[5] = 8ll * st_j;
        }
        have = false;
    };
    auto group_all = [&](bool p) SBZ_ALWAYS {   // p in every lane of the group (a ballot: evaluated by every lane)
        const unsigned long long m = __ballot(p), mask = (1ull << (GL & 63)) - 1;
        return ((m >> (GL * c.g)) & mask) == mask;
    };
    auto coef_at = [&](int slot, SbzGCoef<double>& C) SBZ_ALWAYS {
        const double* row = gb[slot];
        sbz_gcoef<double>(c, [&](int i) { return row[i]; }, C);
    };
    // the background at time tau into the group's row `slot` (and its derivative into dslot), by this lane
    auto bg_dual = [&](int slot, int dslot, int& idx, double tau) SBZ_ALWAYS {
        Dual o[SBZ_NGB];
        sbz_gbg<Dual>(gc, kt, nk, idx, Dual(tau, 1.0), o);
#pragma unroll
        for (int i = 0; i < SBZ_NGB; ++i) gb[slot][i] = o[i].v;
        if (dslot >= 0) {
#pragma unroll
            for (int i = 0; i < SBZ_NGB; ++i) dgb[dslot][i] = o[i].d;
        }
    };
    auto bg_plain = [&](int slot, int& idx, double tau) SBZ_ALWAYS {
        double o[SBZ_NGB];
        sbz_gbg<double>(gc, kt, nk, idx, tau, o);
#pragma unroll
        for (int i = 0; i < SBZ_NGB; ++i) gb[slot][i] = o[i];
    };
    // saves in (t - hprev, tn] (step), or at and before the start: Hermite dense output, sources
    auto saves = [&](bool act, bool step, double tprev, double hprev, double tn, const double* un,
                     const double* fn) SBZ_ALWAYS {
        bool pend = act && isave < a.n_save && saveat[isave] <= tn;
        while (__any(pend)) {
            const int is = pend ? isave : 0;
            const double ts = pend ? saveat[is] : tn;
            const double th = step ? (ts - tprev) / hprev : 1.0;
            const double h00 = (1 + 2 * th) * (1 - th) * (1 - th), h10 = th * (1 - th) * (1 - th);
            const double h01 = th * th * (3 - 2 * th), h11 = th * th * (th - 1);
            double y[M];
#pragma unroll
            for (int l = 0; l < M; ++l)
                y[l] = step ? h00 * u[l] + h10 * hprev * V.get<0>(l) + h01 * un[l] + h11 * hprev * fn[l] : un[l];
            if (pend && a.out_save) {
                double* o = a.out_save + ((size_t)inst * a.n_save + is) * SBZ_N;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const int q = sbz_gcomp(c, l);
                    if (q >= 0) o[q] = y[l];
                }
            }
            if (a.out_src) {
                const double* sb = a.srcbg + ((size_t)set * a.n_save + is) * SBZ_SRCBG_STRIDE;
                // its row passes through slots that are rewritten before they are read again
                double* stage = gb[1];
                double* dstage = dgb[1];
                __syncthreads();
                if (c.lane == 0) {
                    Dual row[SBZ_NGB];
                    sbz_gb_row(sb, row);
#pragma unroll
                    for (int i = 0; i < SBZ_NGB; ++i) {
                        stage[i] = row[i].v;
                        dstage[i] = row[i].d;
                    }
                }
                __syncthreads();
                SbzGCoef<Dual> D;
                sbz_gcoef<Dual>(c, [&](int i) { return Dual(stage[i], dstage[i]); }, D);
                SbzGCoef<double> C;
                coef_at(1, C);
                double fy[M], gy[M], dt_[M], Psi, Pig, dPsi, e0, e1;
                sbz_grhs<false>(c, C, y, fy, Psi, Pig);    // u'
                sbz_grhs<false>(c, C, fy, gy, e0, e1);            // J u'; Ψ and Π_γ of u'
                sbz_gdfdt(c, D, y, dt_, dPsi);
                const double DPsi = e0 + dPsi, Pigd = e1;
                // u'' = ∂f/∂τ + J u'
                const double Pigdd = sbz_gsum<GL>(c.pi0 * (gy[0] + dt_[0]) + c.pi2 * (gy[2] + dt_[2]));
                const double F0 = sbz_gsum<GL>(c.isF ? y[0] : 0.0), Phi = sbz_gsum<GL>(c.one * y[2]);
                const double dPhi = sbz_gsum<GL>(c.one * fy[2]);
                const double thb = sbz_gsum<GL>(c.one * y[4]), thbd = sbz_gsum<GL>(c.one * fy[4]);
                const double kd = sb[3], kdd = sb[SBZ_NB + 3], ddkd = sb[2 * SBZ_NB], eK = exp(-sb[24]), tau = sb[0];
                const double v = -kd * eK, vd = (-kdd + kd * kd) * eK, vdd = (-ddkd + 3 * kd * kdd - kd * kd * kd) * eK;
                const double tau0 = P[SBZ_P_TAU0], trec = P[SBZ_P_TAUREC], chi = tau0 - tau;
                if (pend && ret == SBZ_RET_SUCCESS && c.lane == 0) {
                    double* o = a.out_src + ((size_t)inst * a.n_save + is) * 3;
                    o[0] = v * (F0 / 4 + Psi + Pig / 16) + eK * (DPsi + dPhi) + (vd * thb + v * thbd) * c.ik2 +
                           (3.0 / 16.0) * c.ik2 * (vdd * Pig + 2 * vd * Pigd + v * Pigdd);
                    o[1] = (tau < tau0) ? (3.0 / 16.0) * v * Pig / ((c.k * chi) * (c.k * chi)) : 0.0;
                    o[2] = (tau >= trec && tau < tau0) ? -(Psi + Phi) * (tau - trec) / (tau0 - trec) / chi : 0.0;
                }
            }
            isave += pend;
            pend = act && isave < a.n_save && saveat[isave] <= tn;
        }
    };
    for (;;) {
        // ---- modes that ended write their results; groups without a mode pull the next and start it
        if (have && (ret != SBZ_RET_SUCCESS || !(t < t1))) finish();
        const bool need = !have && !exhausted;
        if (__any(need)) {
            if (need && c.lane == 0) S.f.mode[c.g] = sbz_pull(a, (int)(blockIdx.x % (unsigned)a.n_xcd));
            __syncthreads();
            const int qi = S.f.mode[c.g];
            __syncthreads();
            const bool fresh = need && qi >= 0;
            if (need && !fresh) exhausted = true;
            if (__any(fresh)) {
                // The start runs on the border and chain functions of the one-mode kernels, from LDS: at the
                // initial time f(t + dt0, u0 + dt0 f0) - f(t, u0) is down to the rounding of its terms, and the
                // first step, which sets the whole step sequence, follows it.
                const WaveCtx wc = sbz_wave_ctx(c.lane);
                double* const Bs = gb[1];                       // the background vector B[]
                double* const Cs = S.kv + 64 * M + c.g * SBZ_GSTART;
                double* const v0 = Cs + SBZ_NC;
                double* const v1 = v0 + SBZ_N;
                if (fresh) {
                    inst = a.order ? a.order[qi] : qi;
                    set = a.inst_set[inst];
                    P = a.params + (size_t)set * SBZ_NPAR;
                    kt = a.knots + a.knot_off[set];
                    nk = a.knot_n[set];
                    sbz_gmode(c, P, a.inst_k[inst]);
                    t1 = kt[nk - 1];
                    t = a.inst_t0[inst];
                    bidx = bidx2 = sbz_find_knot(kt, nk, t);
                    st_acc = st_rej = st_f = st_j = 0;
                    iters = 0;
                    ret = SBZ_RET_SUCCESS;
                    lqold = lq0;
                    isave = 0;
                    if (SAVE) saveat = a.saveat ? a.saveat + (size_t)set * a.saveat_stride : nullptr;
                    if (c.lane == 0) {
                        double C[SBZ_NC], B[SBZ_NB];
                        sbz_consts(P, C);
                        sbz_consts_k(C, c.k);
                        int kk = bidx;
                        sbz_bg_plain(P, kt, nk, kk, t, B);
                        sbz_ic(B, C, c.k, v0);
#pragma unroll
                        for (int q = 0; q < SBZ_NC; ++q) Cs[q] = C[q];
#pragma unroll
                        for (int q = 0; q < SBZ_NB; ++q) Bs[q] = B[q];
                        sbz_gconst(P, gc);
                    }
                }
                __syncthreads();
                if (fresh) {
                    sbz_wave_apply(wc, Bs, nullptr, Cs, c.k, v0, v1);
                    if (c.lane == 0) {
                        int kk = bidx;
                        bg_dual(0, 0, kk, t);
                    }
                }
                __syncthreads();
                double f[M];
                if (fresh) {
#pragma unroll
                    for (int l = 0; l < M; ++l) {
                        const int q = sbz_gcomp(c, l);
                        u[l] = (q >= 0) ? v0[q] : 0.0;
                        f[l] = (q >= 0) ? v1[q] : 0.0;
                    }
                } else {
#pragma unroll
                    for (int l = 0; l < M; ++l) f[l] = 0.0;
                }
                bool fin = (c.k > 0.0) && (c.k == c.k);
#pragma unroll
                for (int l = 0; l < M; ++l) fin = fin && (u[l] == u[l]) && fabs(u[l]) <= 1e300;
                const bool fin_g = group_all(fin);
                if (fresh && !fin_g) ret = SBZ_RET_INITIALFAILURE;
                // Hairer–Wanner initial step of the starting groups
                const bool init = fresh && ret == SBZ_RET_SUCCESS && t1 > t;
                double d0 = 0.0, d1 = 0.0;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const double sk = a.atol + fabs(u[l]) * a.rtol;
                    d0 += (u[l] / sk) * (u[l] / sk);
                    d1 += (f[l] / sk) * (f[l] / sk);
                }
                d0 = sqrt(sbz_gsum<GL>(d0) / SBZ_N);
                d1 = sqrt(sbz_gsum<GL>(d1) / SBZ_N);
                double dt0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
                dt0 = fmin(dt0, t1 - t);
                __syncthreads();
                if (init) {
#pragma unroll
                    for (int l = 0; l < M; ++l) {
                        const int q = sbz_gcomp(c, l);
                        if (q >= 0) v0[q] = u[l] + dt0 * f[l];
                    }
                    if (c.lane == 0) {
                        double B[SBZ_NB];
                        int kk = bidx;
                        sbz_bg_plain(P, kt, nk, kk, t + dt0, B);
#pragma unroll
                        for (int q = 0; q < SBZ_NB; ++q) Bs[q] = B[q];
                    }
                }
                __syncthreads();
                if (init) sbz_wave_apply(wc, Bs, nullptr, Cs, c.k, v0, v1);
                __syncthreads();
                double d2 = 0.0;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const int q = sbz_gcomp(c, l);
                    const double sk = a.atol + fabs(u[l]) * a.rtol;
                    const double r = (q >= 0) ? (v1[q] - f[l]) / sk : 0.0;
                    d2 += r * r;
                }
                d2 = sqrt(sbz_gsum<GL>(d2) / SBZ_N) / dt0;
                if (init) {
                    const double mx = fmax(d1, d2);
                    const double dt1 = (mx <= 1e-15) ? fmax(1e-6, dt0 * 1e-3) : pow(0.01 / mx, 1.0 / 6.0);
                    dt = fmin(fmin(100.0 * dt0, dt1), t1 - t);
                    st_f += 2;
#pragma unroll
                    for (int l = 0; l < M; ++l) V.set<0>(l, f[l]);
                }
                if (fresh && !init) {
#pragma unroll
                    for (int l = 0; l < M; ++l) V.set<0>(l, 0.0);
                }
                __syncthreads();
                if constexpr (SAVE) {
                    if (a.n_save > 0) saves(fresh, false, t, 1.0, t, u, u);
                }
                if (fresh) have = true;
            }
        }
        if (!__any(have)) break;
        // ---- per-group checks before the attempt (a group that stops here writes its mode above, next)
        bool live = have && ret == SBZ_RET_SUCCESS && t < t1;
        if (live) {
            if (++iters > a.maxiters) ret = SBZ_RET_MAXITERS;
            else if (t + dt >= t1 - 1e-12 * fabs(t1)) dt = t1 - t;
            else if (dt < 1e-14 * fabs(t)) ret = SBZ_RET_DTLESSTHANMIN;
            live = ret == SBZ_RET_SUCCESS;
        }
        const double h = live ? dt : 1e-3 * (t1 - kt[0]);   // groups without a mode: a harmless step
        const double idt = sbz_rcp(h), ig = idt * (1.0 / SBZ_R5_GAMMA);
        // background at the stage times c_2..c_5 and at t + h (with d/dτ: the next step's t_n), one lane
        // each; four-lane groups take t + h in a second pass
        if constexpr (GL >= 8) {
            if (c.lane < 5) {
                const double cl = (c.lane == 0) ? SBZ_R5_C2 : (c.lane == 1) ? SBZ_R5_C3 : (c.lane == 2) ? SBZ_R5_C4
                                : (c.lane == 3) ? SBZ_R5_C5 : 1.0;
                bg_dual(c.lane + 1, c.lane == 4 ? 1 : -1, bidx, t + cl * h);
            }
        } else {
            const double cl = (c.lane == 0) ? SBZ_R5_C2 : (c.lane == 1) ? SBZ_R5_C3 : (c.lane == 2) ? SBZ_R5_C4 : SBZ_R5_C5;
            bg_plain(c.lane + 1, bidx, t + cl * h);
            if (c.lane == 0) bg_dual(5, 1, bidx2, t + h);
        }
        __syncthreads();
        SbzGFac F;
        {
            SbzGCoef<Dual> D;
            const double* r0 = gb[0];
            const double* rd = dgb[0];
            sbz_gcoef<Dual>(c, [&](int i) SBZ_ALWAYS { return Dual(r0[i], rd[i]); }, D);
            double e0, DT[M];
            sbz_gdfdt(c, D, u, DT, e0);
#pragma unroll
            for (int l = 0; l < M; ++l) V.set<1>(l, DT[l]);
            SbzGCoef<double> C;
            sbz_gvalues(D, C);
            sbz_gfactor(c, C, ig, F);
        }
        if (live) st_j++;
        double us[M], b[M], P7[M], P8[M];   // stage input, right-hand side, and Σ c_7j K_j, Σ c_8j K_j
        SbzGCoef<double> C;
        // stage s <= 5: one read of K_1..K_{s-1} serves the stage input and the right-hand side's Σ c_sj K_j / h
        auto stage = [&](auto SC) SBZ_ALWAYS {
            constexpr int s = decltype(SC)::value;
            const double hd = h * SbzR5::d[s];
#pragma unroll
            for (int l = 0; l < M; ++l) {
                double kj[4] = {};
                if constexpr (s > 1) kj[0] = V.get<2>(l);
                if constexpr (s > 2) kj[1] = V.get<3>(l);
                if constexpr (s > 3) kj[2] = V.get<4>(l);
                if constexpr (s > 4) kj[3] = V.get<5>(l);
                b[l] = hd * V.get<1>(l);
                if constexpr (s == 1) {
                    b[l] += V.get<0>(l);
                } else {
                    double acc = u[l], cs = 0.0;
#pragma unroll
                    for (int j = 1; j < s; ++j) {
                        acc += SbzR5::A[s][j - 1] * kj[j - 1];
                        cs += SbzR5::C[s][j - 1] * kj[j - 1];
                    }
                    us[l] = acc;
                    b[l] += idt * cs;
                }
            }
            if constexpr (s > 1) {
                double e0, e1;
                coef_at(s - 1, C);
                sbz_grhs<true>(c, C, us, b, e0, e1);
            }
            sbz_gsolve(c, F, b);
            if constexpr (s <= 4) {
#pragma unroll
                for (int l = 0; l < M; ++l) V.set<s + 1>(l, b[l]);
            }
        };
        stage(SbzInt<1>{});
        stage(SbzInt<2>{});
        stage(SbzInt<3>{});
        stage(SbzInt<4>{});
        stage(SbzInt<5>{});
        // with K_5 (in b) known, the sums over K_1..K_5 of the last three stages in one pass: K_1..K_5 end
        // here, and stages 7, 8 only add the previous stage to their input
#pragma unroll
        for (int l = 0; l < M; ++l) {
            const double k1 = V.get<2>(l), k2 = V.get<3>(l), k3 = V.get<4>(l), k4 = V.get<5>(l), k5 = b[l];
            us[l] = u[l] + SBZ_R5_A61 * k1 + SBZ_R5_A62 * k2 + SBZ_R5_A63 * k3 + SBZ_R5_A64 * k4 + SBZ_R5_A65 * k5;
            P7[l] = SBZ_R5_C71 * k1 + SBZ_R5_C72 * k2 + SBZ_R5_C73 * k3 + SBZ_R5_C74 * k4 + SBZ_R5_C75 * k5;
            P8[l] = SBZ_R5_C81 * k1 + SBZ_R5_C82 * k2 + SBZ_R5_C83 * k3 + SBZ_R5_C84 * k4 + SBZ_R5_C85 * k5;
            b[l] = idt * (SBZ_R5_C61 * k1 + SBZ_R5_C62 * k2 + SBZ_R5_C63 * k3 + SBZ_R5_C64 * k4 + SBZ_R5_C65 * k5);
        }
        coef_at(5, C);   // stages 6 to 8 and f at t + h share the time t + h
        double e0, e1;
        sbz_grhs<true>(c, C, us, b, e0, e1);
        sbz_gsolve(c, F, b);
#pragma unroll
        for (int l = 0; l < M; ++l) {
            us[l] += b[l];
            P8[l] += SBZ_R5_C86 * b[l];
            b[l] = idt * (P7[l] + SBZ_R5_C76 * b[l]);
        }
        sbz_grhs<true>(c, C, us, b, e0, e1);
        sbz_gsolve(c, F, b);
#pragma unroll
        for (int l = 0; l < M; ++l) {
            us[l] += b[l];
            b[l] = idt * (P8[l] + SBZ_R5_C87 * b[l]);
        }
        sbz_grhs<true>(c, C, us, b, e0, e1);
        sbz_gsolve(c, F, b);
        // u_{n+1} = stage-8 input + k8; error estimate k8
        double ss = 0.0, mx = 0.0;
#pragma unroll
        for (int l = 0; l < M; ++l) {
            us[l] += b[l];
            const double au = fabs(us[l]), q = b[l] * sbz_rcp(a.atol + fmax(fabs(u[l]), au) * a.rtol);
            mx = fmax(mx, au);
            ss += q * q;
        }
        const bool fin_g = group_all((ss == ss) && mx <= 1e300);   // a non-finite state has a non-finite k8
        ss = sbz_gsum<GL>(ss);
        const double EEst = fin_g ? sqrt(ss / SBZ_N) : __builtin_inf();
        const bool acc = live && EEst <= 1.0;
        if (live) st_f += acc ? 8 : 7;
        // PI controller: EEst^β1 qold^-β2 through one logarithm and one exponential
        const double lE = log(EEst);
        const double ex = exp(SBZ_CTL_BETA1 * ((EEst < __builtin_inf()) ? lE : 0.0) - (acc ? SBZ_CTL_BETA2 * lqold : 0.0));
        if (__any(acc)) {
            double f1[M];
            sbz_grhs<false>(c, C, us, f1, e0, e1);   // f(t + h, u_{n+1}): the next step's first stage, the dense output
            double tn = t + h;
            if (tn >= t1 - 1e-14 * fabs(t1)) tn = t1;
            __syncthreads();
            if (acc) {   // the background at t + h is the next step's at t_n
                for (int i = c.lane; i < SBZ_NGB; i += GL) {
                    gb[0][i] = gb[5][i];
                    dgb[0][i] = dgb[1][i];
                }
            }
            __syncthreads();
            if constexpr (SAVE) {
                if (a.n_save > 0) saves(acc, true, t, h, tn, us, f1);
            }
            if (acc) {
                const double q = (EEst == 0.0) ? 1.0 / SBZ_CTL_QMAX
                                               : fmax(1.0 / SBZ_CTL_QMAX, fmin(1.0 / SBZ_CTL_QMIN, ex / SBZ_CTL_GAMMA));
                lqold = fmax(lE, lq0);
                t = tn;
                st_acc++;
                dt = h / q;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    u[l] = us[l];
                    V.set<0>(l, f1[l]);
                }
            }
        }
        if (live && !acc) {
            const double q11r = (EEst < __builtin_inf()) ? ex : 1.0 / SBZ_CTL_QMIN;
            dt = h / fmin(1.0 / SBZ_CTL_QMIN, q11r / SBZ_CTL_GAMMA);
            st_rej++;
        }
        __syncthreads();
    }
}

// The several-modes body under the name that the mixed-model kernels call.
template <bool FUSED, int LN>
SBZ_DEV void sbz_waverow_run(const SbzSolveArgs& a, SbzGroupLDS* S) {
    sbz_group_run<false>(a, *S);
}
