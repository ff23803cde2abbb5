// k_boltsolve: the FP32 solve mode and the tangent-linear solve of the KenCarp4
// integrator (boltsolve, perturbations.jl:25-33), one workgroup of four
// wavefronts per k-mode.  The FP64 solve without tangents is k_solve (solve.hip).
#include "solver_common.h"

// the tangent of stage S after its solve (w̃ = W⁻¹ r̃ banded, y = K⁻¹ D w̃):
// Ż_S = w̃ + hγ(c_S y₀ + c_P y₁ + c_Π y₂), then the next stage's argument
// tangent, or after the last stage u̇ₙ₊₁.  Caller syncs.
template <int S>
__device__ inline void stage_combine_tan(const Geo& G, const WS& W, const WTan& Wt, double hg, const double* y,
                                         const Thr& T) {
    for (int c = T.tid; c < G.n; c += T.nt) {
        const double z = Wt.wd()[c] + hg * (W.cS()[c] * y[0] + W.cP()[c] * y[1] + W.cPi()[c] * y[2]);
        Wt.Zd(S)[c] = z;
        double acc = Wt.ud()[c];
        if constexpr (S < 5) {
#pragma unroll
            for (int j = 0; j < S; ++j) acc += KCT::A[S + 1][j] * Wt.Zd(j)[c];
            Wt.argd()[c] = acc + KCT::A[S + 1][S] * z;
        } else {
#pragma unroll
            for (int j = 0; j < 5; ++j) acc += KCT::A[5][j] * Wt.Zd(j)[c];
            Wt.und()[c] = acc + KC_G * z;
        }
    }
}

// one workgroup of NWAVE wavefronts per k-mode
template <int SR, bool F32, bool TAN = false>
__global__ void __launch_bounds__(NTHR) k_boltsolve(SolveArgs A) {
    // F32: the FP32 solve mode -- factors and substitutions in FP32, each stage
    // value refined against the FP64 residual of its stage equation.
    // TAN: the tangent-linear solve -- u̇ along the primal's steps, each stage's
    // tangent (I − hγL)Ż = h(L ȧrg + L̇(arg + γZ)) solved with the primal's
    // factors and border; outputs and their derivatives
    static_assert(F32 != TAN, "the FP64 solve without tangents is k_solve");
    using P = typename std::conditional<F32, float, double>::type;
    extern __shared__ double lds[];
    __shared__ int s_mode;
    const Thr T = thr_self();
    for (;;) {
        if (T.tid == 0) {
            s_mode = atomicAdd(A.work_counter, 1);
        }
        __syncthreads();
        const int mi = s_mode;
        if (mi >= A.nmodes) return;
#ifdef BOLT_DEBUG_NANFILL
        // debug build: each mode starts from a workspace full of NaNs, so a read
        // of anything this mode has not written itself shows as a wrong value
        for (int i = T.tid; i < A.lds_doubles; i += T.nt) lds[i] = __builtin_nan("");
        __syncthreads();
#endif
        ModeDesc md = A.modes[mi];
        const CosmoDev C = A.cosmos[md.cosmo];
        const CfgDev cf = A.cfgs[md.cfg];
        Geo G = make_geo(cf);
        WS W;
        ws_bind(W, lds, G.n, G.nq);
        const double k = md.k;
        WTan Wt;
        const CosmoDev* Cdp = nullptr;
        if constexpr (TAN) {
            Wt.b = lds + wtan_offset(G.n, G.nq);
            Wt.n = G.n;
            Wt.nq = G.nq;
            Cdp = A.cosmos_dot + md.cosmo;
            if (T.tid < G.nq) {
                Wt.qd()[T.tid] = Cdp->qv[T.tid]; Wt.df0d()[T.tid] = Cdp->df0[T.tid]; Wt.based()[T.tid] = Cdp->base[T.tid];
            }
            for (int c = T.tid; c < G.n; c += T.nt) Wt.ud()[c] = 0.0;
        }
        if (T.tid < G.nq) { W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid]; }
        for (int c = T.tid; c < G.n; c += T.nt) W.u()[c] = 0.0;
        setup_rows(C, G, W, T);
        __syncthreads();
        if constexpr (TAN) initial_conditions_t<D1>(C, Cdp, G, W, &Wt, k, W.u(), Wt.ud(), T);
        else initial_conditions(C, G, W, k, W.u(), T);
        __syncthreads();
        long long nacc = 0, nrej = 0, nrhs = 0, nsol = 0;
        double x = C.x0, xend = C.x1;
        const double rt = cf.reltol, at = cf.abstol;
        const int nref = (cf.flags & BOLT_CFG_REFINE_MASK) ? (cf.flags & BOLT_CFG_REFINE_MASK) >> 4 : 12;
        int status = BOLT_MODE_OK;
        int next = 0;  // next output index
        const int om = A.out_mode;
        const int nout = (om == 0) ? A.nsave : C.nx;
        // outputs at the starting point take the initial condition as saved
        while (next < nout) {
            double xv = (om == 0) ? A.x_save[next] : node_x(C, next);
            if (!(xv <= x)) break;
            if constexpr (TAN)
                emit_tan(C, *Cdp, G, W, Wt, A, md.out, k, x, W.u(), W.u(), Wt.ud(), Wt.ud(), x, W.u(), W.u(), Wt.ud(),
                         Wt.ud(), xv, next, T);
            else
                emit(C, G, W, A, md.out, k, x, W.u(), W.u(), x, W.u(), W.u(), xv, next, T, om, nullptr);
            ++next;
        }
        // FSAL start: f(u0) (the RSA overwrite, if on, persists in u)
        {
            XC X = make_xc(C, k, x);
            qfill(C, G, X, W, T);
            XCd D;
            if constexpr (TAN) {
                D = make_xcd(C, *Cdp, X);
                if (T.tid < G.nq) qfill_one_dot(C, *Cdp, W, Wt, X.a, X.kH, D.kH, W.qe(), Wt.qset_base(5), Wt.ktd(5), T.tid);
                if (T.tid == T.nt - 1) ktab_head_dot(Wt.ktd(5), X, D);
            }
            __syncthreads();
            Fun F = rhs_rows(C, G, X, W, W.qcur(), W.kcur(), W.u(), 1.0, W.f(), false, T);
            ++nrhs;
            Fun Fd;
            if constexpr (TAN) {
                Fd = rhs_rows_tan(C, *Cdp, G, X, D, W, W.qcur(), Wt.qset(5), W.kcur(), Wt.ktd(5), Wt.ud(), W.u(), 1.0,
                                  Wt.fd(), T);
                ++nrhs;
            }
            __syncthreads();
            if constexpr (TAN) {
                if (X.rsa && T.tid == 0) rsa_mutate_t<D1>(G, X, &D, k, W.u(), Wt.ud(), D1{F.P, Fd.P});
            } else {
                if (X.rsa && T.tid == 0) rsa_mutate(G, X, k, W.u(), F.P);
            }
            __syncthreads();
        }
        // Hairer's starting step (order 4)
        double h;
        {
            double d0 = wrms(G, W, W.u(), W.u(), W.u(), rt, at, T);
            double d1 = wrms(G, W, W.f(), W.u(), W.u(), rt, at, T);
            double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
            if (h0 > xend - x) h0 = xend - x;
            for (int c = T.tid; c < G.n; c += T.nt) W.arg()[c] = W.u()[c] + h0 * W.f()[c];
            XC X1 = make_xc(C, k, x + h0);
            qfill(C, G, X1, W, T);
            __syncthreads();
            rhs_rows(C, G, X1, W, W.qcur(), W.kcur(), W.arg(), 1.0, W.w(), false, T);
            ++nrhs;
            __syncthreads();
            for (int c = T.tid; c < G.n; c += T.nt) W.w()[c] -= W.f()[c];
            double d2 = wrms(G, W, W.w(), W.u(), W.u(), rt, at, T) / h0;
            double dm = fmax(d1, d2);
            double h1 = (dm <= 1e-15) ? fmax(1e-6, h0 * 1e-3) : pow(0.01 / dm, 1.0 / 5.0);
            h = fmin(100.0 * h0, h1);
            if (h > xend - x) h = xend - x;
        }
        const int maxsteps = cf.max_steps > 0 ? cf.max_steps : 100000;
        long long nsteps = 0;
        bool take = false;  // the last attempt was accepted
        while (x < xend) {
            if (++nsteps > maxsteps) { status = BOLT_MODE_MAXSTEPS; break; }
            bool last = false;
            if (h >= xend - x) { h = xend - x; last = true; }
            const double hg = h * KC_G;
            // Z₀ = h f(u) and the first stage's argument; after an accepted
            // step this pass also moves u_{n+1}, f_{n+1} into u, f (each thread
            // copies and reads only its own rows)
            for (int c = T.tid; c < G.n; c += T.nt) {
                double uc, fc;
                if (take) {
                    uc = W.un()[c]; fc = W.fn()[c];
                    W.u()[c] = uc; W.f()[c] = fc;
                } else {
                    uc = W.u()[c]; fc = W.f()[c];
                }
                const double z0 = h * fc;
                W.Z(0)[c] = z0;
                W.arg()[c] = uc + KCT::A[1][0] * z0;
                if constexpr (TAN) {
                    double udc, fdc;
                    if (take) {
                        udc = Wt.und()[c]; fdc = Wt.fnd()[c];
                        Wt.ud()[c] = udc; Wt.fd()[c] = fdc;
                    } else {
                        udc = Wt.ud()[c]; fdc = Wt.fd()[c];
                    }
                    const double zd0 = h * fdc;
                    Wt.Zd(0)[c] = zd0;
                    Wt.argd()[c] = udc + KCT::A[1][0] * zd0;
                }
            }
            take = false;
            // the five implicit stage points depend on x and h only: their
            // coefficients, q-quantities, W bands and LU come first, all stages
            // at once
            // lanes 0..4: each stage point's coefficients; wavefronts 1..3 at
            // the same time: the q-sets, from a = e^x and kH = k/ℋ formed
            // exactly as make_xc forms them
            if (T.tid < 5) {
                const XC Xs = make_xc(C, k, x + KC_C[T.tid + 1] * h);
                store_xc(W.xcs(T.tid), Xs);
                ktab_head(W.ktab(T.tid), Xs);
                if constexpr (TAN) {
                    const XCd Ds = make_xcd(C, *Cdp, Xs);
                    store_xcd(Wt.xcd(T.tid), Ds);
                    ktab_head_dot(Wt.ktd(T.tid), Xs, Ds);
                }
            } else if (T.wv > 0) {
                for (int t = T.tid - WAVE; t < 5 * G.nq; t += T.nt - WAVE) {
                    const int st = t / G.nq;
                    const double xs = x + KC_C[st + 1] * h;
                    const double Hs = spl(C, BOLT_T_HC, xs);
                    const double kHs = k * rcp(Hs);
                    const double as = exp(xs);
                    qfill_one(C, W, as, kHs, W.qst_base(st), W.ktab(st), t - st * G.nq);
                    if constexpr (TAN) {
                        const double kHsd = -kHs * (spl(*Cdp, BOLT_T_HC, xs) / Hs);
                        qfill_one_dot(C, *Cdp, W, Wt, as, kHs, kHsd, W.qst_base(st), Wt.qset_base(st), Wt.ktd(st),
                                      t - st * G.nq);
                    }
                }
            }
            __syncthreads();
            stage_bands<P>(G, W, hg, T);
            __syncthreads();
            // the LU of the five stage points on wavefront 0 while the others
            // form stage 1's right-hand side and border columns (which need
            // no factor)
            if (T.wv == 0) {
                chain_factor_all<P>(G, W, T.lane);
            } else {
                Thr Tr = T;
                Tr.tid -= WAVE;
                Tr.nt -= WAVE;
                rhs_rows(C, G, load_xc(W.xcs(0)), W, W.qst(0), W.ktab(0), W.arg(), h, W.w(), true, Tr,
                         F32 ? W.rvec() : nullptr);
            }
            ++nrhs;
            __syncthreads();
            Cap K;
            XC Xs;
            for (int s = 1; s < 6; ++s) {
                Xs = load_xc(W.xcs(s - 1));
                const QSet Qs = W.qst(s - 1);
                // rhs = h f(ψ) and the border columns (stage 1's are formed above)
                if (s > 1) {
                    rhs_rows(C, G, Xs, W, Qs, W.ktab(s - 1), W.arg(), h, W.w(), true, T, F32 ? W.rvec() : nullptr);
                    ++nrhs;
                    __syncthreads();
                }
                chain_solve4<SR, P>(G, W, s - 1, T);
                ++nsol;
                // no barrier: wavefront r's border functionals read only the
                // vector it has just solved (ordered by wave_lds_sync)
                double y[3];
                K = stage_border(C, G, Xs, W, Qs, hg, T, y);
                if constexpr (F32) {
                    // Z_s from the FP32 solve, then sweeps of iterative
                    // refinement: the FP64 residual ρ = r − Z + γ·h·A·Z of the
                    // stage equation (I − hγA)Z = r, its correction through the
                    // same FP32 factors and border, Z += δ
                    for (int c = T.tid; c < G.n; c += T.nt)
                        W.Z(s)[c] = W.w()[c] + hg * (W.cS()[c] * y[0] + W.cP()[c] * y[1] + W.cPi()[c] * y[2]);
                    __syncthreads();
                    for (int it = 0; it < nref; ++it) {
                        // ρ = r − Z + γ·(h·A·Z)
                        rhs_rows(C, G, Xs, W, Qs, W.ktab(s - 1), W.Z(s), h, W.w(), false, T);
                        for (int c = T.tid; c < G.n; c += T.nt)
                            W.w()[c] = (W.rvec()[c] - W.Z(s)[c]) + KC_G * W.w()[c];
                        ++nrhs;
                        __syncthreads();
                        if (T.wv == 0) {
                            wave_subst<SR>(W.bandsT<P>(s - 1), G.n, W.w(), W.dump(), T.lane);
                            const Fun Fc = functionals(C, G, Xs, Qs, W.w(), T);
                            if (T.lane == 0) { W.red()[12] = Fc.S; W.red()[13] = Fc.P; W.red()[14] = Fc.Pi; }
                        }
                        ++nsol;
                        __syncthreads();
                        const double rc[3] = {W.red()[12], W.red()[13], W.red()[14]};
                        double yc[3];
                        solve3(K, rc, yc);
                        // excess of each correction over 1e-14 of its own component
                        double ex = 0.0;
                        for (int c = T.tid; c < G.n; c += T.nt) {
                            const double d = W.w()[c] + hg * (W.cS()[c] * yc[0] + W.cP()[c] * yc[1] +
                                                              W.cPi()[c] * yc[2]);
                            const double z = W.Z(s)[c] + d;
                            W.Z(s)[c] = z;
                            ex = fmax(ex, fabs(d) - 1e-14 * fabs(z));
                        }
                        ex = wave_max(ex);
                        if (T.lane == 0) W.red()[16 + T.wv] = ex;
                        __syncthreads();
                        // converged once every correction is below 1e-14 of its component (every
                        // thread reads the same four maxima, so all leave together; components
                        // below FP32's range get no correction and count as converged).  A
                        // stage still unconverged after the last sweep (the FP32 factors' error
                        // times the stage matrix's condition number near one) is taken as it
                        // stands: its error enters the step's error estimate
                        const double* m = W.red();
                        if (!(fmax(fmax(m[16], m[17]), fmax(m[18], m[19])) > 1e-290)) break;
                    }
                    switch (s) {
                        case 1: stage_combine<1, true>(G, W, hg, y, T); break;
                        case 2: stage_combine<2, true>(G, W, hg, y, T); break;
                        case 3: stage_combine<3, true>(G, W, hg, y, T); break;
                        case 4: stage_combine<4, true>(G, W, hg, y, T); break;
                        default: stage_combine<5, true>(G, W, hg, y, T); break;
                    }
                } else if constexpr (TAN) {
                    // Z_s, and the stage value arg + γZ_s into w (which nothing reads any more)
                    for (int c = T.tid; c < G.n; c += T.nt) {
                        const double z = W.w()[c] + hg * (W.cS()[c] * y[0] + W.cP()[c] * y[1] + W.cPi()[c] * y[2]);
                        W.Z(s)[c] = z;
                        W.w()[c] = W.arg()[c] + KC_G * z;
                    }
                    __syncthreads();
                    // r̃ = h(f(ȧrg) + L̇(arg + γZ_s)) at the stage point
                    rhs_rows_tan(C, *Cdp, G, Xs, load_xcd(Wt.xcd(s - 1)), W, Qs, Wt.qset(s - 1), W.ktab(s - 1),
                                 Wt.ktd(s - 1), Wt.argd(), W.w(), h, Wt.wd(), T);
                    ++nrhs;
                    __syncthreads();
                    // wavefront 0 solves it with the stage's factors while the others
                    // form the primal's next argument
                    if (T.wv == 0) {
                        wave_subst<SR>(W.bandsT<double>(s - 1), G.n, Wt.wd(), W.dump(), T.lane);
                        const Fun Fc = functionals(C, G, Xs, Qs, Wt.wd(), T);
                        if (T.lane == 0) { W.red()[12] = Fc.S; W.red()[13] = Fc.P; W.red()[14] = Fc.Pi; }
                    } else {
                        Thr Tr = T;
                        Tr.tid -= WAVE;
                        Tr.nt -= WAVE;
                        switch (s) {
                            case 1: stage_combine<1, true>(G, W, hg, y, Tr); break;
                            case 2: stage_combine<2, true>(G, W, hg, y, Tr); break;
                            case 3: stage_combine<3, true>(G, W, hg, y, Tr); break;
                            case 4: stage_combine<4, true>(G, W, hg, y, Tr); break;
                            default: stage_combine<5, true>(G, W, hg, y, Tr); break;
                        }
                    }
                    ++nsol;
                    __syncthreads();
                    const double rc[3] = {W.red()[12], W.red()[13], W.red()[14]};
                    double yt[3];
                    solve3(K, rc, yt);
                    switch (s) {
                        case 1: stage_combine_tan<1>(G, W, Wt, hg, yt, T); break;
                        case 2: stage_combine_tan<2>(G, W, Wt, hg, yt, T); break;
                        case 3: stage_combine_tan<3>(G, W, Wt, hg, yt, T); break;
                        case 4: stage_combine_tan<4>(G, W, Wt, hg, yt, T); break;
                        default: stage_combine_tan<5>(G, W, Wt, hg, yt, T); break;
                    }
                }
                __syncthreads();
            }
            // Shampine's smoothed estimate: W⁻¹ e with the last stage's W, on
            // wavefront 0.  Meanwhile the other wavefronts evaluate the FSAL
            // derivative f(u_{n+1}) at x + h, which is the last stage point
            // (abscissa 1): its coefficients, q-set and scalar table serve.
            // It is used only if the step is accepted; a step cut to end on
            // xend evaluates it at xend after acceptance instead.
            const bool spec = !last;
            Fun Fn;
            if (T.wv == 0) {
                chain_solve1<SR, P>(G, W, 4, W.arg(), T);
            } else if (spec) {
                Thr Tf = T;
                Tf.tid -= WAVE;
                Tf.nt -= WAVE;
                Fn = rhs_rows(C, G, load_xc(W.xcs(4)), W, W.qst(4), W.ktab(4), W.un(), 1.0, W.fn(), false, Tf);
            }
            ++nsol;
            if (spec) ++nrhs;
            __syncthreads();
            // the border step of the error solve folded into its norm:
            // e_c = ψ_c + hγ(c_S y₀ + c_P y₁ + c_Π y₂) is formed and weighted
            // row by row, never stored
            double en;
            {
                const Fun Fe = functionals(C, G, Xs, W.qst(4), W.arg(), T);
                double r[3] = {Fe.S, Fe.P, Fe.Pi}, ye[3];
                solve3(K, r, ye);
                double ss = 0.0;
                for (int c = T.tid; c < G.n; c += T.nt) {
                    const double e = W.arg()[c] + hg * (W.cS()[c] * ye[0] + W.cP()[c] * ye[1] + W.cPi()[c] * ye[2]);
                    const double sc = at + rt * fmax(fabs(W.u()[c]), fabs(W.un()[c]));
                    const double q = e / sc;
                    ss += q * q;
                }
                en = sqrt(block_sum(ss, W, T) / G.n);
            }
            if (!isfinite(en)) {
                ++nrej;
                h *= 0.2;
                if (h < 1e-14) { status = BOLT_MODE_NONFINITE; break; }
                continue;
            }
            if (en <= 1.0) {
                double xn = last ? xend : x + h;
                // FSAL at x_{n+1} (already evaluated unless the step ends on xend)
                XC Xn;
                if (spec) {
                    Xn = load_xc(W.xcs(4));
                } else {
                    Xn = make_xc(C, k, xn);
                    qfill(C, G, Xn, W, T);
                    __syncthreads();
                    Fn = rhs_rows(C, G, Xn, W, W.qcur(), W.kcur(), W.un(), 1.0, W.fn(), false, T);
                    ++nrhs;
                    __syncthreads();
                }
                // Fn is held by wavefronts 1.. in both cases
                if constexpr (TAN) {
                    // ḟ(u̇ₙ₊₁) at xₙ₊₁ before the RSA write, from the last stage point's
                    // tangent tables or the current x's
                    XCd Dn;
                    const double *Kn, *Kdn;
                    QSet Qn, Qdn;
                    if (spec) {
                        Dn = load_xcd(Wt.xcd(4));
                        Kn = W.ktab(4); Kdn = Wt.ktd(4); Qn = W.qst(4); Qdn = Wt.qset(4);
                    } else {
                        Dn = make_xcd(C, *Cdp, Xn);
                        if (T.tid < G.nq)
                            qfill_one_dot(C, *Cdp, W, Wt, Xn.a, Xn.kH, Dn.kH, W.qe(), Wt.qset_base(5), Wt.ktd(5), T.tid);
                        if (T.tid == T.nt - 1) ktab_head_dot(Wt.ktd(5), Xn, Dn);
                        __syncthreads();
                        Kn = W.kcur(); Kdn = Wt.ktd(5); Qn = W.qcur(); Qdn = Wt.qset(5);
                    }
                    const Fun Fnd = rhs_rows_tan(C, *Cdp, G, Xn, Dn, W, Qn, Qdn, Kn, Kdn, Wt.und(), W.un(), 1.0,
                                                 Wt.fnd(), T);
                    ++nrhs;
                    __syncthreads();
                    if (Xn.rsa && T.wv == 1 && T.lane == 0)
                        rsa_mutate_t<D1>(G, Xn, &Dn, k, W.un(), Wt.und(), D1{Fn.P, Fnd.P});
                } else {
                    if (Xn.rsa && T.wv == 1 && T.lane == 0) rsa_mutate(G, Xn, k, W.un(), Fn.P);
                }
                __syncthreads();
                ++nacc;
                while (next < nout) {
                    double xv = (om == 0) ? A.x_save[next] : node_x(C, next);
                    if (!(xv <= xn)) break;
                    if constexpr (TAN)
                        emit_tan(C, *Cdp, G, W, Wt, A, md.out, k, x, W.u(), W.f(), Wt.ud(), Wt.fd(), xn, W.un(), W.fn(),
                                 Wt.und(), Wt.fnd(), xv, next, T);
                    else
                        emit(C, G, W, A, md.out, k, x, W.u(), W.f(), xn, W.un(), W.fn(), xv, next, T, om, nullptr);
                    ++next;
                }
                take = true;  // u, f <- u_{n+1}, f_{n+1} in the next step's first pass
                x = xn;
                double fac = (en == 0.0) ? 10.0 : 0.9 * pow(en, -0.25);
                fac = fmin(10.0, fmax(0.2, fac));
                h *= fac;
            } else {
                ++nrej;
                double fac = fmin(1.0, fmax(0.2, 0.9 * pow(en, -0.25)));
                h *= fac;
                if (h < 1e-14 * fmax(1.0, fabs(x))) { status = BOLT_MODE_DTMIN; break; }
            }
        }
        if (T.tid == 0) {
            A.status[md.out] = status;
            if (A.counters) {
                long long* cc = A.counters + (size_t)md.out * 4;
                cc[0] = nacc; cc[1] = nrej; cc[2] = nrhs; cc[3] = nsol;
            }
        }
        __syncthreads();
    }
}

// the tangent-linear solve, or the FP32 solve mode
const void* boltsolve_kernel(bool tan) {
    return tan ? (const void*)k_boltsolve<SR_DEFAULT, false, true> : (const void*)k_boltsolve<SR_DEFAULT, true>;
}
