// Tangent solve with one hierarchy per lane: u and s = ∂u/∂log θ of one instance in the eight groups
// (the last two idle) of SBZ_GL lanes that share its step sequence.  The equations are sbz_wave_tan_body's: with
//   J_θ v = (f(v; B₊) - f(v; B₋)) / (2h)
// a stage solves  W x_u = b_u  and  W x_s = b_s + J_θ x_u, where b_s holds f(s_in; B) + J_θ u_in.
//
// The groups' roles:
//   0: u, with the background of θ      1: s, with that of θ, one stage behind
//   2, 3: J_θ u_in,  4, 5: J_θ x_u, with the backgrounds of log θ ± h, for the stage that group 1 is at.
// A step is nine passes in which every group evaluates one right-hand side and solves one system (what
// it does not need it discards), so it takes little longer than a plain step: in one group after
// another it would take four right-hand sides and two solves per stage.  The vectors that change
// groups (u_in and x_u of group 0, one pass later; the groups' right-hand sides) go through LDS.
//
// Bound by instruction issue, as the plain step: 6.8 k instructions an attempt at n = 47 (19 us).  20 k for two
// parameters (n = 47): 277 ms a call before, 97 now: 38 ms of kernel, the rest mostly the host's five background
// solves (θ, and θ ± h of each parameter at a tight tolerance), one after another.
#pragma once

constexpr int SBZ_GTR = 8;                              // groups per instance
constexpr int SBZ_GTI = 64 / SBZ_GL / SBZ_GTR;          // instances per wavefront
struct SbzGTanLDS {
    double gb[64 / SBZ_GL][6][SBZ_NGB];    // as SbzGroupFixed
    double dgb[64 / SBZ_GL][2][SBZ_NGB];
    double gc[64 / SBZ_GL][SBZ_NGC];
    double ta[10][8], tc[10][8], td[10];   // a_sj, c_sj, d_s by stage (rows 0 and 9: zero)
    double kv[9][SBZ_GM][64];              // columns of the lanes: f_n, ∂f/∂τ, K_1..K_7
    double xv[3][SBZ_GM][64];              // u_in, x_u; a group's right-hand side
    double sc[SBZ_GTI][2];
    int mode[SBZ_GTI];
};
static_assert(64 / SBZ_GL * SBZ_GSTART <= 8 * SBZ_GM * 64, "a starting instance's scratch lies in the K_s");

SBZ_DEV void sbz_gtan_run(const SbzSolveArgs& a, SbzGTanLDS& S) {
    constexpr int M = SBZ_GM, GL = SBZ_GL;
    SbzGCtx c = sbz_gctx();
    const int role = c.g % SBZ_GTR, slot = c.g / SBZ_GTR;
    const bool lag = role != 0, isS = role == 1, isD = role >= 2 && role <= 5;
    const int c0 = slot * SBZ_GTR * GL + c.lane;        // this lane's column in the instance's group 0
    double (*const gb)[SBZ_NGB] = S.gb[c.g];
    double (*const dgb)[SBZ_NGB] = S.dgb[c.g];
    double* const gc = S.gc[c.g];
    double* const kv = &S.kv[0][0][threadIdx.x];
    // row j - 1 from here on is the group's stage of pass j
    const double *const ta = S.ta[lag ? 0 : 1], *const tc = S.tc[lag ? 0 : 1], *const td = S.td + (lag ? 0 : 1);
    auto K = [&](int j, int l) SBZ_ALWAYS -> double& { return kv[(j * M + l) * 64]; };
    for (int e = threadIdx.x; e < 80; e += 64) {
        const int s = e / 8, i = e % 8;
        const bool in = s >= 2 && s <= 8 && i < s - 1;
        S.ta[s][i] = in ? SbzR5::A[in ? s : 0][i] : 0.0;
        S.tc[s][i] = in ? SbzR5::C[in ? s : 0][i] : 0.0;
        if (i == 0) S.td[s] = (s <= 8) ? SbzR5::d[s <= 8 ? s : 0] : 0.0;
    }
    const int share = (a.n_inst + a.S - 1) / a.S;
    bool have = false, exhausted = slot >= share;
    int inst = 0;
    int set = a.inst_set[a.order ? a.order[0] : 0];
    const double* P = a.params + (size_t)set * SBZ_NPAR;   // θ
    const double* kt = a.knots + a.knot_off[set];          // this group's background
    int nk = a.knot_n[set];
    double t = kt[0], tb = kt[0], t1 = kt[nk - 1], dt = 1e-3 * (t1 - tb), tsc = 0.0;
    int bidx = 0, bidx2 = 0;
    long long iters = 0;
    int st_acc = 0, st_rej = 0, st_f = 0, st_j = 0;
    int ret = SBZ_RET_SUCCESS;
    const double lq0 = log(SBZ_CTL_QOLDINIT);
    double lqold = lq0;
    double u[M];   // u_n (group 0), s_n (group 1)
#pragma unroll
    for (int l = 0; l < M; ++l) {
        u[l] = 0.0;
#pragma unroll
        for (int j = 0; j < 9; ++j) K(j, l) = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) S.xv[j][l][threadIdx.x] = 0.0;
    }
    sbz_gmode(c, P, 1.0);
    if (c.lane == 0) sbz_gconst(P, gc);
    __syncthreads();
    auto group_all = [&](bool p) SBZ_ALWAYS {
        const unsigned long long m = __ballot(p), mask = (1ull << GL) - 1;
        return ((m >> (GL * c.g)) & mask) == mask;
    };
    auto bg = [&](auto TC, int sl, int dsl, int& idx, double tau) SBZ_ALWAYS {
        using T = decltype(TC);
        T o[SBZ_NGB];
        sbz_gbg<T>(gc, kt, nk, idx, T(tau) + TC, o);
#pragma unroll
        for (int i = 0; i < SBZ_NGB; ++i) gb[sl][i] = dval(o[i]);
        if (dsl >= 0) {
#pragma unroll
            for (int i = 0; i < SBZ_NGB; ++i) dgb[dsl][i] = dder(o[i]);
        }
    };
    const Dual seed(0.0, 1.0);
    // the groups' values f to group 1: Δ_u of the groups 2, 3 and Δ_x of the groups 4, 5
    auto gather = [&](const double* f, bool du, bool dx, double* d) SBZ_ALWAYS {
        if (isD) {
#pragma unroll
            for (int l = 0; l < M; ++l) S.xv[2][l][threadIdx.x] = f[l];
        }
        __syncthreads();
#pragma unroll
        for (int l = 0; l < M; ++l) {
            d[l] = 0.0;
            if (du) d[l] = S.xv[2][l][c0 + 2 * GL] - S.xv[2][l][c0 + 3 * GL];
            if (dx) d[l] += S.xv[2][l][c0 + 4 * GL] - S.xv[2][l][c0 + 5 * GL];
            d[l] = isS ? tsc * d[l] : 0.0;
        }
        __syncthreads();
    };
    for (;;) {
        // ---- instances that ended write their results; idle slots pull the next and start it
        if (have && (ret != SBZ_RET_SUCCESS || !(t < t1))) {
            double* o = (isS ? a.out_s : a.out_u) + (size_t)inst * SBZ_N;
            double* of = a.out_fend + (size_t)inst * SBZ_N;
#pragma unroll
            for (int l = 0; l < M; ++l) {
                const int q = sbz_gcomp(c, l);
                if (q >= 0 && role <= 1) o[q] = u[l];
                if (q >= 0 && role == 0) of[q] = K(0, l);
            }
            if (c.lane == 0 && role == 0) {
                a.retcode[inst] = ret;
                long long* st = a.stats + (size_t)inst * 6;
                st[0] = st_acc;
                st[1] = st_rej;
                st[2] = st_f;
                st[3] = st_j;
                st[4] = st_j;
                st[5] = 16ll * st_j;
            }
            have = false;
        }
        const bool need = !have && !exhausted;
        if (__any(need)) {
            if (need && role == 0 && c.lane == 0) S.mode[slot] = sbz_pull(a, (int)(blockIdx.x % (unsigned)a.n_xcd));
            __syncthreads();
            const int qi = S.mode[slot];
            __syncthreads();
            const bool fresh = need && qi >= 0;
            if (need && !fresh) exhausted = true;
            if (__any(fresh)) {
                // on the one-mode kernels' functions, from LDS, as the plain start (sbz_group_run)
                const WaveCtx wc = sbz_wave_ctx(c.lane);
                double* const Bs = gb[1];
                double* const scr = &S.kv[1][0][0];
                double* const Cs = scr + c.g * SBZ_GSTART;
                double* const v0 = Cs + SBZ_NC;
                double* const v1 = v0 + SBZ_N;
                // the vector q of another group of the instance
                auto of = [&](int r, const double* q) SBZ_ALWAYS { return q + (r - role) * SBZ_GSTART; };
                if (fresh) {
                    inst = a.order ? a.order[qi] : qi;
                    const int s0 = a.inst_set[inst];
                    set = (role == 2 || role == 4) ? a.inst_setp[inst] : (role == 3 || role == 5) ? a.inst_setm[inst] : s0;
                    P = a.params + (size_t)s0 * SBZ_NPAR;
                    tb = a.knots[a.knot_off[s0]];
                    t1 = a.knots[a.knot_off[s0] + a.knot_n[s0] - 1];
                    kt = a.knots + a.knot_off[set];
                    nk = a.knot_n[set];
                    tsc = a.inst_tscale[inst];
                    sbz_gmode(c, P, a.inst_k[inst]);
                    t = a.inst_t0[inst];
                    bidx = bidx2 = sbz_find_knot(kt, nk, t);
                    st_acc = st_rej = st_f = st_j = 0;
                    iters = 0;
                    ret = SBZ_RET_SUCCESS;
                    lqold = lq0;
                    if (c.lane == 0) {
                        double C[SBZ_NC], B[SBZ_NB];
                        const double* Pq = a.params + (size_t)set * SBZ_NPAR;
                        sbz_consts(P, C);
                        sbz_consts_k(C, c.k);
                        int kk = bidx;
                        sbz_bg_plain(Pq, kt, nk, kk, t, B);
                        sbz_ic(B, C, c.k, v0);
#pragma unroll
                        for (int q = 0; q < SBZ_NC; ++q) Cs[q] = C[q];
#pragma unroll
                        for (int q = 0; q < SBZ_NB; ++q) Bs[q] = B[q];
                        sbz_gconst(Pq, gc);
                    }
                }
                __syncthreads();
                // u_0 of θ in every group but 1, which holds s_0 = (u_0(θ + h) - u_0(θ - h)) / (2h)
                double f[M], d[M];
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const int q = sbz_gcomp(c, l);
                    double v = 0.0;
                    if (fresh && q >= 0) v = isS ? (of(2, v0)[q] - of(3, v0)[q]) * tsc : of(0, v0)[q];
                    if (fresh) u[l] = v;
                }
                __syncthreads();
                if (fresh) {
#pragma unroll
                    for (int l = 0; l < M; ++l) {
                        const int q = sbz_gcomp(c, l);
                        if (q >= 0) v0[q] = u[l];
                    }
                }
                __syncthreads();
                if (fresh) {
                    sbz_wave_apply(wc, Bs, nullptr, Cs, c.k, v0, v1);
                    if (c.lane == 0) {
                        int kk = bidx;
                        bg(seed, 0, 0, kk, t);
                    }
                }
                __syncthreads();
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const int q = sbz_gcomp(c, l);
                    f[l] = (fresh && q >= 0) ? v1[q] : 0.0;
                }
                gather(f, true, false, d);
                bool fin = (c.k > 0.0) && (c.k == c.k);
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    f[l] += d[l];
                    fin = fin && (u[l] == u[l]) && fabs(u[l]) <= 1e300;
                }
                const bool fin_g = group_all(fin);
                if (fresh && c.lane == 0 && role <= 1) S.sc[slot][role] = fin_g ? 0.0 : 1.0;
                __syncthreads();
                if (fresh && (S.sc[slot][0] != 0.0 || S.sc[slot][1] != 0.0)) ret = SBZ_RET_INITIALFAILURE;
                __syncthreads();
                // Hairer–Wanner initial step of the primal
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
                if (init && role == 0) {
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
                if (init && role == 0) sbz_wave_apply(wc, Bs, nullptr, Cs, c.k, v0, v1);
                __syncthreads();
                double d2 = 0.0;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    const int q = sbz_gcomp(c, l);
                    const double sk = a.atol + fabs(u[l]) * a.rtol;
                    const double r = (q >= 0 && init) ? (v1[q] - f[l]) / sk : 0.0;
                    d2 += r * r;
                }
                d2 = sqrt(sbz_gsum<GL>(d2) / SBZ_N) / dt0;
                if (init) {
                    const double mx = fmax(d1, d2);
                    const double dt1 = (mx <= 1e-15) ? fmax(1e-6, dt0 * 1e-3) : pow(0.01 / mx, 1.0 / 6.0);
                    if (role == 0 && c.lane == 0) S.sc[slot][0] = fmin(fmin(100.0 * dt0, dt1), t1 - t);
                    st_f += 2;
                }
                __syncthreads();
                if (init) dt = S.sc[slot][0];
                if (fresh) {
#pragma unroll
                    for (int l = 0; l < M; ++l) K(0, l) = init || role == 0 ? f[l] : 0.0;
                    have = true;
                }
                __syncthreads();
            }
        }
        if (!__any(have)) break;
        // ---- per-instance checks before the attempt, alike in all its groups
        bool live = have && ret == SBZ_RET_SUCCESS && t < t1;
        if (live) {
            if (++iters > a.maxiters) ret = SBZ_RET_MAXITERS;
            else if (t + dt >= t1 - 1e-12 * fabs(t1)) dt = t1 - t;
            else if (dt < 1e-14 * fabs(t)) ret = SBZ_RET_DTLESSTHANMIN;
            live = ret == SBZ_RET_SUCCESS;
        }
        const double h = live ? dt : 1e-3 * (t1 - tb);
        const double idt = sbz_rcp(h), ig = idt * (1.0 / SBZ_R5_GAMMA);
        if constexpr (GL >= 8) {
            if (c.lane < 5) {
                const double cl = (c.lane == 0) ? SBZ_R5_C2 : (c.lane == 1) ? SBZ_R5_C3 : (c.lane == 2) ? SBZ_R5_C4
                                : (c.lane == 3) ? SBZ_R5_C5 : 1.0;
                bg(seed, c.lane + 1, c.lane == 4 ? 1 : -1, bidx, t + cl * h);
            }
        } else {
            const double cl = (c.lane == 0) ? SBZ_R5_C2 : (c.lane == 1) ? SBZ_R5_C3 : (c.lane == 2) ? SBZ_R5_C4 : SBZ_R5_C5;
            bg(0.0, c.lane + 1, -1, bidx, t + cl * h);
            if (c.lane == 0) bg(seed, 5, 1, bidx2, t + h);
        }
        if (role == 0) {
#pragma unroll
            for (int l = 0; l < M; ++l) S.xv[0][l][threadIdx.x] = u[l];
        }
        __syncthreads();
        SbzGFac F;
        double x[M], d[M];
        {
            SbzGCoef<Dual> D;
            const double* r0 = gb[0];
            const double* rd = dgb[0];
            sbz_gcoef<Dual>(c, [&](int i) SBZ_ALWAYS { return Dual(r0[i], rd[i]); }, D);
            double e0, DT[M];
#pragma unroll
            for (int l = 0; l < M; ++l) x[l] = sbz_sel(role <= 1, u[l], S.xv[0][l][c0]);
            sbz_gdfdt(c, D, x, DT, e0);
            gather(DT, true, false, d);
#pragma unroll
            for (int l = 0; l < M; ++l) K(1, l) = DT[l] + d[l];
            SbzGCoef<double> C;
            sbz_gvalues(D, C);
            sbz_gfactor(c, C, ig, F);
        }
        if (live) st_j++;
        double us[M], un[M], f1[M], ss = 0.0, mx = 0.0, e0, e1;
        SbzGCoef<double> C;
#pragma unroll
        for (int l = 0; l < M; ++l) un[l] = f1[l] = 0.0;
        // the background rows of the stages 1..9
        auto row_at = [&](int j) SBZ_ALWAYS {
            constexpr int bs[11] = {0, 0, 1, 2, 3, 4, 5, 5, 5, 5, 5};
            const double* r = gb[lag ? bs[j - 1] : bs[j]];
            return (role == 4 || role == 5) ? (const double*)gb[0] : r;
        };
        // pass j: stage j of group 0, j - 1 of the others
        auto pass = [&](auto JC) SBZ_ALWAYS {
            constexpr int j = decltype(JC)::value;
            double cs[M], f[M];
#pragma unroll
            for (int l = 0; l < M; ++l) {
                us[l] = u[l];
                cs[l] = 0.0;
            }
#pragma unroll
            for (int i = 1; i <= 7; ++i) {
                if (i > j - 1) continue;
                const double ai = ta[8 * (j - 1) + i - 1], ci = tc[8 * (j - 1) + i - 1];
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    double ki = K(i + 1, l);
                    if (i == j - 1) ki = sbz_sel(lag, 0.0, ki);   // not there yet
                    us[l] += ai * ki;
                    cs[l] += ci * ki;
                }
            }
            if constexpr (j == 9) {
#pragma unroll
                for (int l = 0; l < M; ++l) us[l] = sbz_sel(role == 0, un[l], us[l]);
            }
            if constexpr (j == 1) {
#pragma unroll
                for (int l = 0; l < M; ++l) f[l] = K(0, l);
            } else {
                const double* row = row_at(j);
                sbz_gcoef<double>(c, [&](int i) SBZ_ALWAYS { return row[i]; }, C);
                const double (*const xin)[64] = S.xv[role >= 4];
#pragma unroll
                for (int l = 0; l < M; ++l) x[l] = sbz_sel(role <= 1, us[l], xin[l][c0]);
                __syncthreads();
                sbz_grhs<false>(c, C, x, f, e0, e1);
                gather(f, j >= 3, true, d);
                if constexpr (j == 2) {   // stage 1 of group 1 starts from its f_n
#pragma unroll
                    for (int l = 0; l < M; ++l) f[l] = sbz_sel(lag, K(0, l), f[l]);
                }
                if constexpr (j == 9) {
#pragma unroll
                    for (int l = 0; l < M; ++l) f1[l] = f[l];
                }
#pragma unroll
                for (int l = 0; l < M; ++l) f[l] += d[l];
            }
            const double hd = h * td[j - 1];
#pragma unroll
            for (int l = 0; l < M; ++l) f[l] += hd * K(1, l) + idt * cs[l];
            sbz_gsolve(c, F, f);
            if constexpr (j >= 2 && j <= 7) {
#pragma unroll
                for (int l = 0; l < M; ++l) kv[((j + 1 - lag) * M + l) * 64] = f[l];
            } else if constexpr (j == 1 || j == 8) {
                if (lag == (j == 8)) {
#pragma unroll
                    for (int l = 0; l < M; ++l) K(j == 1 ? 2 : 8, l) = f[l];
                }
            }
            if constexpr (j == 8) {
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    un[l] = us[l] + f[l];
                    const double au = fabs(un[l]), q = f[l] * sbz_rcp(a.atol + fmax(fabs(u[l]), au) * a.rtol);
                    mx = fmax(mx, au);
                    ss += q * q;
                }
            }
            if constexpr (j == 9) {
#pragma unroll
                for (int l = 0; l < M; ++l) un[l] = sbz_sel(role == 0, un[l], us[l] + f[l]);
            }
            if (role == 0) {
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    S.xv[0][l][threadIdx.x] = us[l];
                    S.xv[1][l][threadIdx.x] = f[l];
                }
            }
            __syncthreads();
        };
        pass(SbzInt<1>{});
        pass(SbzInt<2>{});
        pass(SbzInt<3>{});
        pass(SbzInt<4>{});
        pass(SbzInt<5>{});
        pass(SbzInt<6>{});
        pass(SbzInt<7>{});
        pass(SbzInt<8>{});
        pass(SbzInt<9>{});
        // the error of the primal; both blocks finite
        if (isS) {
            mx = 0.0;
#pragma unroll
            for (int l = 0; l < M; ++l) mx = (un[l] == un[l]) ? fmax(mx, fabs(un[l])) : __builtin_inf();
            ss = 0.0;
        }
        const bool fin_g = group_all((ss == ss) && mx <= 1e300);
        ss = sbz_gsum<GL>(ss);
        if (c.lane == 0 && role <= 1) S.sc[slot][role] = fin_g ? ss : __builtin_inf();
        __syncthreads();
        const double EEst = sqrt((S.sc[slot][0] + S.sc[slot][1]) / SBZ_N);
        const bool acc = live && EEst <= 1.0;
        if (live) st_f += acc ? 8 : 7;
        const double lE = log(EEst);
        const double ex = exp(SBZ_CTL_BETA1 * ((EEst < __builtin_inf()) ? lE : 0.0) - (acc ? SBZ_CTL_BETA2 * lqold : 0.0));
        if (__any(acc)) {
            // f of the tangent block at t + h: the next step's first stage
            sbz_gcoef<double>(c, [&](int i) SBZ_ALWAYS { return gb[5][i]; }, C);
            double f[M];
#pragma unroll
            for (int l = 0; l < M; ++l) x[l] = sbz_sel(role <= 1, un[l], S.xv[0][l][c0]);
            __syncthreads();
            sbz_grhs<false>(c, C, x, f, e0, e1);
            gather(f, true, false, d);
            double tn = t + h;
            if (tn >= t1 - 1e-14 * fabs(t1)) tn = t1;
            if (acc) {
                for (int i = c.lane; i < SBZ_NGB; i += GL) {
                    gb[0][i] = gb[5][i];
                    dgb[0][i] = dgb[1][i];
                }
                const double q = (EEst == 0.0) ? 1.0 / SBZ_CTL_QMAX
                                               : fmax(1.0 / SBZ_CTL_QMAX, fmin(1.0 / SBZ_CTL_QMIN, ex / SBZ_CTL_GAMMA));
                lqold = fmax(lE, lq0);
                t = tn;
                st_acc++;
                dt = h / q;
#pragma unroll
                for (int l = 0; l < M; ++l) {
                    u[l] = un[l];
                    K(0, l) = sbz_sel(isS, f[l] + d[l], f1[l]);
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
