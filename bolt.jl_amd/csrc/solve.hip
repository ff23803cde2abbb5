// k_solve: the FP64 KenCarp4 integrator (boltsolve, perturbations.jl:25-33), one
// workgroup of four wavefronts per k-mode.  It shares row recipes, banded LU and
// source functions with k_boltsolve (the FP32 and tangent-linear solves); the
// arithmetic of every value is that kernel's, operation for operation, so the two
// take the same steps.
//
// What bounds it: one mode's chain of dependent phases.  A step is about twenty
// barrier-separated phases over n rows (n = 197..473 in use), each a few hundred
// cycles of LDS and FP64 latency that no second wavefront on the SIMD hides.
// The design therefore shortens the chain:
//  - a thread owns rows tid, tid + 256 (and, past 512 rows, tid + 512) and keeps their recipe, state and
//    stage values in registers; LDS holds what other threads read (the stage
//    argument, the right-hand sides, u and f for the dense output);
//  - a substitution keeps its rows in registers from the forward scan through
//    the backward one (the backward scan runs toward lower lanes over the same
//    rows), and everything of it that depends on the factors alone -- the
//    multipliers' products along a lane and the scan's multipliers across lanes
//    -- is formed before the barrier its right-hand side waits for;
//  - the border columns' right-hand sides are formed in the registers of the
//    wavefront that substitutes them;
//  - the dense output of a step (source functions or states at the nodes it
//    crossed) is taken one node per wavefront while the next step's factors are
//    being formed, instead of node after node by the whole workgroup, and
//    interpolates only the entries the source functions read;
//  - a phase's uniform scalars are one LDS access per wavefront (StageSc), not
//    one broadcast read each.
// Measured (one MI355X, against the same solve with its vectors and recipes in LDS
// and runtime strides; 10 or 200 modes up to k = 0.25 alike, since the largest k's
// chain is what counts): source grids of n = 197 88.2 to 57.7 ms, of n = 323 87.3 to
// 65.6; P(k) at n = 473, two scan passes with 96 registers spilled, 95.3 to 80.5.

#include "solve_layout.h"

// ---- substitutions
// One pass of 64·SR rows: the parts of both scans that depend on the factors
// alone.  Row i of the lane: l = -l1; backward, from the lane's highest row
// down: r = -d·u1; d the pivots' reciprocals.  la/ra: the lane maps' multipliers
// (the products of l, r along the lane) before each of the six scan steps,
// lf/rf after them.
template <int SR>
struct FacPass {
    double l[SR], r[SR], d[SR], la[6], ra[6], lf, rf, u0, u1;
};

// backward scan steps 4 and 5 (row_bcast 15 and 31 have no mirror image): lanes
// 0..15 take lane 16's value and 32..47 lane 48's; lanes 0..31 take lane 32's
__device__ inline double mirror_bcast15(double v, double id, int lane) {
    const double a = readlane64(v, 16), b = readlane64(v, 48);
    const int row = lane >> 4;
    return row == 0 ? a : row == 2 ? b : id;
}
__device__ inline double mirror_bcast31(double v, double id, int lane) {
    const double a = readlane64(v, 32);
    return lane < 32 ? a : id;
}

template <int SR>
__device__ inline void lane_rows(const double* v, int j0, bool in, double (&r)[SR]) {
#pragma unroll
    for (int i = 0; i < SR; ++i) r[i] = 0.0;
    if (in) {
        if constexpr (SR % 2 == 0) {
            const double2* p = (const double2*)__builtin_assume_aligned(v + j0, 16);
#pragma unroll
            for (int i = 0; i < SR / 2; ++i) { const double2 t = p[i]; r[2 * i] = t.x; r[2 * i + 1] = t.y; }
        } else {
#pragma unroll
            for (int i = 0; i < SR; ++i) r[i] = v[j0 + i];
        }
    }
}
template <int SR>
__device__ inline void store_rows(double* v, int j0, bool in, const double (&r)[SR]) {
    if (in) {
        if constexpr (SR % 2 == 0) {
            double2* p = (double2*)__builtin_assume_aligned(v + j0, 16);
#pragma unroll
            for (int i = 0; i < SR / 2; ++i) p[i] = make_double2(r[2 * i], r[2 * i + 1]);
        } else {
#pragma unroll
            for (int i = 0; i < SR; ++i) v[j0 + i] = r[i];
        }
    }
}

template <int SR>
__device__ inline void fac_prep(FacPass<SR>& F, const Bands& B, int j0, bool in, int lane) {
    double l1[SR], u1[SR];
    lane_rows<SR>(B.l1, j0, in, l1);
    lane_rows<SR>(B.d, j0, in, F.d);
    lane_rows<SR>(B.u1, j0, in, u1);
    F.u0 = u1[0]; F.u1 = u1[1];
#pragma unroll
    for (int i = 0; i < SR; ++i) {
        F.l[i] = -l1[i];
        F.r[i] = -F.d[SR - 1 - i] * u1[SR - 1 - i];
    }
    double a = F.l[0], b = F.r[0];
#pragma unroll
    for (int i = 1; i < SR; ++i) { a = F.l[i] * a; b = F.r[i] * b; }
    F.la[0] = a; a *= dppk<0x111, 0xF>(a, 1.0);
    F.ra[0] = b; b *= dppk<0x101, 0xF>(b, 1.0);
    F.la[1] = a; a *= dppk<0x112, 0xF>(a, 1.0);
    F.ra[1] = b; b *= dppk<0x102, 0xF>(b, 1.0);
    F.la[2] = a; a *= dppk<0x114, 0xF>(a, 1.0);
    F.ra[2] = b; b *= dppk<0x104, 0xF>(b, 1.0);
    F.la[3] = a; a *= dppk<0x118, 0xF>(a, 1.0);
    F.ra[3] = b; b *= dppk<0x108, 0xF>(b, 1.0);
    F.la[4] = a; a *= dppk<0x142, 0xA>(a, 1.0);
    F.ra[4] = b; b *= mirror_bcast15(b, 1.0, lane);
    F.la[5] = a; a *= dppk<0x143, 0xC>(a, 1.0);
    F.ra[5] = b; b *= mirror_bcast31(b, 1.0, lane);
    F.lf = a; F.rf = b;
}

// forward and back substitution of one right-hand side held in registers, row
// p·64·SR + SR·lane + i in v[p][i]; l2 and u2 are the second band's entries
// (Θ₁ from v_b, v_b from Θ₁), whose rows 0..3 sit in lane 0
template <int SR, int NP>
__device__ inline void subst_regs(const FacPass<SR> (&F)[NP], double (&v)[NP][SR], double l2, double u2, int lane) {
    double carry = 0.0;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        double be[SR];
#pragma unroll
        for (int i = 0; i < SR; ++i) be[i] = v[p][i];
        if (p == 0) {
            const double corr = l2 * fmaT(F[0].l[1], be[0], be[1]);
            be[3] -= lane == 0 ? corr : 0.0;
        }
#pragma unroll
        for (int i = 1; i < SR; ++i) be[i] = fmaT(F[p].l[i], be[i - 1], be[i]);
        double B = be[SR - 1];
        B = fmaT(F[p].la[0], dppz<0x111>(B), B);
        B = fmaT(F[p].la[1], dppz<0x112>(B), B);
        B = fmaT(F[p].la[2], dppz<0x114>(B), B);
        B = fmaT(F[p].la[3], dppz<0x118>(B), B);
        B = fmaT(F[p].la[4], dppk<0x142, 0xA>(B, 0.0), B);
        B = fmaT(F[p].la[5], dppk<0x143, 0xC>(B, 0.0), B);
        if (p > 0) B = fmaT(F[p].lf, carry, B);
        const double tin = dppk<0x138, 0xF>(B, carry);  // wave_shr 1; lane 0 keeps carry
        if (p + 1 < NP) carry = readlane64(B, WAVE - 1);
        double m = 0.0;
#pragma unroll
        for (int i = 0; i < SR; ++i) {
            m = i == 0 ? F[p].l[0] : F[p].l[i] * m;
            v[p][i] = fmaT(m, tin, be[i]);
        }
    }
    carry = 0.0;
#pragma unroll
    for (int p = NP - 1; p >= 0; --p) {
        double be[SR];
#pragma unroll
        for (int i = 0; i < SR; ++i) be[i] = F[p].d[SR - 1 - i] * v[p][SR - 1 - i];
        const double y0 = v[0][0], y1 = v[0][1];
#pragma unroll
        for (int i = 1; i < SR; ++i) be[i] = fmaT(F[p].r[i], be[i - 1], be[i]);
        double B = be[SR - 1];
        B = fmaT(F[p].ra[0], dppz<0x101>(B), B);
        B = fmaT(F[p].ra[1], dppz<0x102>(B), B);
        B = fmaT(F[p].ra[2], dppz<0x104>(B), B);
        B = fmaT(F[p].ra[3], dppz<0x108>(B), B);
        B = fmaT(F[p].ra[4], mirror_bcast15(B, 0.0, lane), B);
        B = fmaT(F[p].ra[5], mirror_bcast31(B, 0.0, lane), B);
        if (p < NP - 1) B = fmaT(F[p].rf, carry, B);
        const double tin = dppk<0x130, 0xF>(B, carry);  // wave_shl 1; lane 63 keeps carry
        if (p > 0) carry = readlane64(B, 0);
        double m = 0.0;
#pragma unroll
        for (int i = 0; i < SR; ++i) {
            m = i == 0 ? F[p].r[0] : F[p].r[i] * m;
            v[p][SR - 1 - i] = fmaT(m, tin, be[i]);
        }
        if (p == 0) {
            const double x1 = ((y1 - u2 * v[0][3]) - F[0].u1 * v[0][2]) * F[0].d[1];
            const double x0 = (y0 - F[0].u0 * x1) * F[0].d[0];
            v[0][1] = lane == 0 ? x1 : v[0][1];
            v[0][0] = lane == 0 ? x0 : v[0][0];
        }
    }
}

// ---- stage coefficients
// A stage point's scalars, 16 doubles: the border functionals' coefficients,
// the scalar table's leading entries, and what else the RSA write reads.  A
// wavefront loads them with one LDS access, an entry per lane, and takes them
// to scalars with v_readlane: every wavefront needs all of them in every phase,
// and as broadcast reads they kept the CU's one LDS pipe busy (four wavefronts
// times some twenty reads a phase) for longer than the phase's arithmetic.
enum { XS_C12 = 0, XS_FS2, XS_K23, XS_FP0, XS_FP1, XS_FP2, XS_FP3, XS_FP4, XS_TP, XS_IHETA, XS_TPR, XS_RSA, XS_HC,
       XS_TPP, XS_CSB2, XS_N = 16 };
__device__ inline void store_xs(double* p, const XC& X) {
    p[XS_C12] = X.c12; p[XS_FS2] = X.fs2; p[XS_K23] = X.k23; p[XS_FP0] = X.fp0; p[XS_FP1] = X.fp1;
    p[XS_FP2] = X.fp2; p[XS_FP3] = X.fp3; p[XS_FP4] = X.fp4;
    p[XS_TP] = X.tp; p[XS_IHETA] = X.iHeta; p[XS_TPR] = X.tp * X.R; p[XS_RSA] = X.rsa ? 0.0 : 1.0;
    p[XS_HC] = X.Hc; p[XS_TPP] = X.tpp; p[XS_CSB2] = X.csb2;
}
struct KHead {
    double tp, iHeta, tpr, rsa;
};
struct StageSc {
    double g;  // lane's entry
    __device__ double at(int i) const { return readlane64(g, i); }
    __device__ KHead head() const {
        KHead h;
        h.tp = at(XS_TP); h.iHeta = at(XS_IHETA); h.tpr = at(XS_TPR); h.rsa = at(XS_RSA);
        return h;
    }
};
__device__ inline StageSc load_sc(const double* xs, int lane) {
    StageSc s;
    s.g = xs[lane & (XS_N - 1)];
    return s;
}
// what rsa_mutate reads
__device__ inline XC rsa_xc(const double* xs) {
    XC X;
    X.Hc = xs[XS_HC]; X.tp = xs[XS_TP]; X.tpp = xs[XS_TPP]; X.csb2 = xs[XS_CSB2];
    return X;
}

// Ψ, Φ′, Π of a vector by one wavefront (functionals' arithmetic) with one
// gather of the vector and one of the q weights: lanes 0..15 hold the bins of
// Σ sw ℳ₂, lanes 16..31 those of Σ rw ℳ₀ (both sums run at once, in their rows
// of 16 lanes; bins 16 and 32 further on come in later turns for nq > 16), lanes
// 32..40 the nine single rows
struct QLane {
    int row, wt, step;  // the lane's row of the state, its weight's place in a q-set, rows per 16 bins
    int left;           // bins of this lane
};
__device__ inline QLane make_qlane(const Geo& G, int lane) {
    QLane q;
    const int i = lane & 15;
    const int fixed[9] = {G.cE, 4, G.cC + 2, G.cD, 0, 2, G.cC, G.cB + 2, G.cB};
    q.left = lane < 32 && i < G.nq ? (G.nq - i + 15) / 16 : 0;
    q.row = q.left ? G.cM + i * (G.nm + 1) + (lane < 16 ? 2 : 0) : 0;
    q.wt = q.left ? (lane < 16 ? 2 : 3) * G.nq + i : 0;
    q.step = 16 * (G.nm + 1);
#pragma unroll
    for (int j = 0; j < 9; ++j) q.row = lane == 32 + j ? fixed[j] : q.row;
    return q;
}
__device__ inline Fun fun_wave(double Or, double Onu, int nq, const StageSc& X, const double* qset, const QLane& ql,
                               const double* v) {
    const double g = v[ql.row];
    double a = qset[ql.wt] * g;
    a = ql.left > 0 ? a : 0.0;
    if (nq > 16) {
        for (int j = 1; 16 * j < nq; ++j) {
            const bool in = j < ql.left;
            const double t = fmaT(qset[in ? ql.wt + 16 * j : 0], v[in ? ql.row + ql.step * j : 0], a);
            a = in ? t : a;
        }
    }
    const double e = readlane64(g, 32), t2 = readlane64(g, 33), n2 = readlane64(g, 34), dl = readlane64(g, 35),
                 db = readlane64(g, 36), t0 = readlane64(g, 37), n0 = readlane64(g, 38), p2 = readlane64(g, 39),
                 p0 = readlane64(g, 40);
    a += dpp64<0x111>(a);
    a += dpp64<0x112>(a);
    a += dpp64<0x114>(a);
    a += dpp64<0x118>(a);
    const double s2 = readlane64(a, 15), s0 = readlane64(a, 31);
    Fun F;
    F.S = fmaT(-X.at(XS_FS2), s2, fmaT(-X.at(XS_C12), fmaT(Or, t2, Onu * n2), -e));
    F.P = fmaT(-X.at(XS_K23), e, F.S) +
          fmaT(X.at(XS_FP4), s0, fmaT(X.at(XS_FP3), n0, fmaT(X.at(XS_FP2), t0, fmaT(X.at(XS_FP0), dl, X.at(XS_FP1) * db))));
    F.Pi = t2 + p2 + p0;
    return F;
}

// ---- row passes from registers
// One owned row: its recipe (row_recipe), the table scalar its two couplings
// share (a coupling absent from a row has a zero constant, so either index
// serves), which diagonal terms it takes (d_coef) and whether the RSA factor
// applies
struct RowReg {
    double al, au, di, cs, cp, cpi, dc;
    int kx, kcs;  // scalar-table indices
    bool tau, vb, rsa;
};
template <class WS_>
__device__ inline RowReg load_row(const Geo& G, const WS_& W, int c) {
    RowReg R;
    const int kd = W.kinds()[c];
    R.al = W.rcp_(RC_AL)[c]; R.au = W.rcp_(RC_AU)[c]; R.di = W.rcp_(RC_DI)[c];
    R.cs = W.rcp_(RC_CS)[c]; R.cp = W.rcp_(RC_CP)[c]; R.cpi = W.rcp_(RC_CPI)[c];
    R.dc = (c == 1 || c == G.cD + 1) ? -1.0 : 0.0;
    R.kx = R.al != 0.0 ? (kd & 255) : ((kd >> 8) & 255);
    R.kcs = (kd >> 16) & 255;
    R.rsa = (kd >> 24) == K_RSA;
    R.tau = c >= 3 && c < G.cC;
    R.vb = c == 1;
    return R;
}
__device__ inline double row_diag(const RowReg& R, const KHead& H) {
    return fmaT(R.di, H.iHeta, R.dc + (R.tau ? H.tp : 0.0)) + (R.vb ? H.tpr : 0.0);
}
// row c of f(v) from its own and neighbouring entries; first: the wavefront
// holding rows 1 and 3, whose second-band terms read v[3] and v[1]
__device__ inline double row_eval_reg(const RowReg& R, const KHead& H, double kx, double kcs, int c, bool first,
                                      double vc, double vm, double vp, const double* v, const Fun& F) {
    double acc = fmaT(R.au * kx, vp, fmaT(row_diag(R, H), vc, (R.al * kx) * vm));
    if (first) {
        const double w = v[c == 1 ? 3 : 1];
        const double e = (c == 1 ? 3.0 * H.tpr : H.tp * (1.0 / 3.0)) * w;
        acc += c == 1 || c == 3 ? e : 0.0;
    }
    acc += fmaT(R.cpi * H.tp, F.Pi, fmaT(R.cs * kcs, F.S, R.cp * F.P));
    return R.rsa ? H.rsa * acc : acc;
}
// the neighbouring rows' values: from the neighbouring lanes' registers, and
// for the wavefront's first and last rows from the vector itself
__device__ inline void row_neighbours(double vc, const double* v, int c, int cm, int cp, int lane, double& vm,
                                      double& vp) {
    const double edge = v[lane == 0 ? cm : lane == WAVE - 1 ? cp : c];
    vm = dppk<0x138, 0xF>(vc, edge);  // wave_shr 1
    vp = dppk<0x130, 0xF>(vc, edge);  // wave_shl 1
}
// W = I - hγL at the five stage points, the owned rows (stage_bands)
template <int NR, class WS_>
__device__ inline void bands_reg(const Geo& G, const WS_& W, const RowReg (&R)[NR], const int (&rc)[NR],
                                 const bool (&in)[NR], double hg, int lane) {
    // every load before the first store: the compiler must assume that a store
    // to LDS changes what a later load reads
    StageSc X[5];
    double kx[5][NR];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        X[s] = load_sc(W.xcs(s), lane);
#pragma unroll
        for (int i = 0; i < NR; ++i) kx[s][i] = W.ktab(s)[R[i].kx];
    }
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const KHead H = X[s].head();
        const Bands B = W.template bandsT<double>(s);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const double mh = R[i].rsa ? H.rsa * hg : hg;
            const double L = -mh * (R[i].al * kx[s][i]), D = fmaT(-mh, row_diag(R[i], H), 1.0),
                         U = -mh * (R[i].au * kx[s][i]);
            if (in[i]) { B.l1[rc[i]] = L; B.d[rc[i]] = D; B.u1[rc[i]] = U; }
            if (i == 0 && rc[0] < CB) {
                B.l2c[rc[0]] = rc[0] == 3 ? -mh * (H.tp * (1.0 / 3.0)) : 0.0;
                B.u2c[rc[0]] = rc[0] == 1 ? -mh * (3.0 * H.tpr) : 0.0;
            }
        }
    }
}

// out = scale·f(v) on all rows by wavefronts 1..3, beside work of wavefront 0's:
// each takes its own rows (v's values there in a), wavefront 1 also wavefront
// 0's, from the recipes in LDS.  Returns v's functionals.
template <int NR, class WS_>
__device__ inline Fun rows_beside(const Geo& G, const WS_& W, const RowReg (&R)[NR], const int (&rc)[NR],
                                  const int (&rm)[NR], const int (&rp)[NR], const bool (&in)[NR], const double (&a)[NR],
                                  int st, const QLane& ql, double Or, double Onu, const double* v, double scale,
                                  double* out, int wv, int lane) {
    const StageSc X = load_sc(W.xcs(st), lane);
    const Fun F = fun_wave(Or, Onu, W.nq, X, W.qst_base(st), ql, v);
    const KHead H = X.head();
    const double* K = W.ktab(st);
    double r[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        double vm, vp;
        row_neighbours(a[i], v, rc[i], rm[i], rp[i], lane, vm, vp);
        r[i] = scale * row_eval_reg(R[i], H, K[R[i].kx], K[R[i].kcs], rc[i], false, a[i], vm, vp, v, F);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
        if (in[i]) out[rc[i]] = r[i];
    if (wv == 1)
        for (int c = lane; c < W.n; c += NTHR) out[c] = scale * row_eval(G, W, K, v, c, W.n, F.S, F.P, F.Pi);
    return F;
}

// ---- banded LU (chain_factor_seg's arithmetic): one lane per (stage point,
// segment), the next block's rows loaded while a block is factored.  A block's
// loads would otherwise complete behind the previous block's stores, LDS
// operations of a wavefront completing in issue order.
struct LuRows {
    double L[CB], D[CB], U[CB];
};
__device__ inline void lu_load(LuRows& r, const double* l1, const double* d, const double* u1, int j) {
#pragma unroll
    for (int i = 0; i < CB; ++i) { r.L[i] = l1[j + i]; r.D[i] = d[j + i]; r.U[i] = u1[j + i]; }
}
// rows j..j+CB-1 of a tridiagonal stretch: the products P stay off the pivot
// chain inv_i = 1/(D_i - P_i·inv_{i-1})
__device__ inline void lu_block(LuRows& r, double* l1, double* d, int j, int m, double& ip1, double& u1p1) {
    double P[CB];
#pragma unroll
    for (int i = 0; i < CB; ++i) { P[i] = r.L[i] * u1p1; u1p1 = r.U[i]; }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        r.L[i] *= ip1;
        ip1 = rcp_piv(fmaT(-P[i], ip1, r.D[i]));
        r.D[i] = ip1;
    }
    if (__all(j + CB <= m)) {  // no lane's segment ends inside the block
#pragma unroll
        for (int i = 0; i < CB; ++i) { l1[j + i] = r.L[i]; d[j + i] = r.D[i]; }
    } else {
#pragma unroll
        for (int i = 0; i < CB; ++i)
            if (j + i < m) { l1[j + i] = r.L[i]; d[j + i] = r.D[i]; }
    }
}
template <class WS_>
__device__ inline void lu_segment(const WS_& W, const Bands& B, int c0, int m) {
    double* const l1 = B.l1 + c0;
    double* const d = B.d + c0;
    double* const u1 = B.u1 + c0;
    const bool first = c0 == 0;  // the only segment with a second band
    double ip1 = 0, ip2 = 0, u1p1 = 0, u1p2 = 0, u2p1 = 0, u2p2 = 0;
    LuRows cur, nxt;
    constexpr int FB = 4;  // rows 0..3 run the full bandwidth-2 recurrence
    {
        double L2[FB], L1[FB], D[FB], U1[FB], U2[FB];
#pragma unroll
        for (int i = 0; i < FB; ++i) {
            const double l2 = B.l2c[i], u2 = B.u2c[i];
            L2[i] = first ? l2 : 0.0; U2[i] = first ? u2 : 0.0;
            L1[i] = l1[i]; D[i] = d[i]; U1[i] = u1[i];
        }
        lu_load(cur, l1, d, u1, FB);
#pragma unroll
        for (int i = 0; i < FB; ++i) {
            const double m2 = L2[i] * ip2;
            const double m1 = fmaT(-m2, u1p2, L1[i]) * ip1;
            const double dd = fmaT(-m1, u1p1, fmaT(-m2, u2p2, D[i]));
            const double uu = fmaT(-m1, u2p1, U1[i]);
            const double inv = rcp_piv(dd);
            L2[i] = m2; L1[i] = m1; D[i] = inv; U1[i] = uu;
            ip2 = ip1; ip1 = inv;
            u1p2 = u1p1; u1p1 = uu;
            u2p2 = u2p1; u2p1 = U2[i];
        }
#pragma unroll
        for (int i = 0; i < FB; ++i) {
            if (first && i < m) B.l2c[i] = L2[i];
            if (i < m) { l1[i] = L1[i]; d[i] = D[i]; u1[i] = U1[i]; }
        }
    }
    // (loads past the segment's end read other rows' entries, never used)
    for (int j = FB; j < m;) {
        lu_load(nxt, l1, d, u1, j + CB < W.n - c0 ? j + CB : j);
        lu_block(cur, l1, d, j, m, ip1, u1p1);
        j += CB;
        if (j >= m) break;
        lu_load(cur, l1, d, u1, j + CB < W.n - c0 ? j + CB : j);
        lu_block(nxt, l1, d, j, m, ip1, u1p1);
        j += CB;
    }
}

// ---- dense output of one node by one wavefront
// The cubic Hermite interpolant between two accepted steps, as weights of their
// states and derivatives
struct Hermite {
    double a, b, fa, fb;
};
__device__ inline Hermite hermite(double xa, double xb, double xv) {
    const double h = xb - xa;
    Hermite w = {1.0, 0.0, 0.0, 0.0};
    if (h != 0.0) {
        const double t = (xv - xa) / h, s = 1.0 - t, c = t * s, e = c * (1.0 - 2.0 * t);
        w.a = s + e;
        w.b = t - e;
        w.fa = c * s * h;
        w.fb = -c * t * h;
        if (t == 1.0) w = {0.0, 1.0, 0.0, 0.0};
    }
    return w;
}
struct DenseIn {
    const double *ua, *ub, *fa, *fb;
    Hermite w;
    __device__ double at(int c) const {
        return fmaT(w.fb, fb[c], fmaT(w.fa, fa[c], fmaT(w.b, ub[c], w.a * ua[c])));
    }
};

// The saved state at xv, or source_function (perturbations.jl:343-383) and
// source_function_P (385-404) there: hierarchy! on the rows they read, with its
// RSA write to the state (spectra.jl:16, 36).  A lane interpolates only what it
// needs: one entry for the functionals (QLane) and a source row with its two
// neighbours; es holds the node's scalar table and q-set.
template <class WS_>
__device__ inline void emit_wave(const CosmoDev& C, const Geo& G, const WS_& W, const SolveArgs& A, int out, double k,
                                 const DenseIn& I, double xv, int idx, int lane, int om, double* obase,
                                 const QLane& ql, double* es) {
    if (om == 0) {
        double* dst = obase ? obase + (size_t)idx * G.n : A.out + ((size_t)out * A.nsave + idx) * A.n_state_stride;
        for (int c = lane; c < G.n; c += WAVE) dst[W.place()[c]] = I.at(c);
        return;
    }
    // the tables at xv, one per lane (lane 11: η at the last node)
    static constexpr int NT = 12;
    const int tabs[NT] = {BOLT_T_HC, BOLT_T_ETA, BOLT_T_TAU_P, BOLT_T_TAU_PP, BOLT_T_CSB2, BOLT_T_HC_P,
                          BOLT_T_HC_PP, BOLT_T_TAU, BOLT_T_G, BOLT_T_G_P, BOLT_T_G_PP, BOLT_T_ETA};
    int tab = BOLT_T_HC;
#pragma unroll
    for (int i = 1; i < NT; ++i) tab = lane == i ? tabs[i] : tab;
    const double tv = spl(C, tab, lane == 11 ? C.x1 : xv);
    // interpolate while the tables load
    double g = I.at(ql.row);
    const int c = source_row(G, lane), cc = c >= 0 ? c : 1;
    const double vm = I.at(cc - 1), vc = I.at(cc), vp = I.at(cc + 1 < G.n ? cc + 1 : cc), v1 = I.at(1), v3 = I.at(3);
    const double Hc = readlane64(tv, 0), eta = readlane64(tv, 1), tp = readlane64(tv, 2), tpp = readlane64(tv, 3),
                 csb2 = readlane64(tv, 4), Hcp = readlane64(tv, 5), Hcpp = readlane64(tv, 6), gv = readlane64(tv, 8),
                 gp = readlane64(tv, 9), gpp = readlane64(tv, 10);
    const XC X = make_xc_at(C, k, xv, exp(xv), Hc, eta, tp, tpp, csb2);
    double* const K = es;
    double* const qp = es + WS_::kt;
    if (lane < G.nq) qfill_one(C, W, X.a, X.kH, qp, K, lane);
    if (lane == WAVE - 1) ktab_head(K, X);
    wave_lds_sync();
    // Ψ, Φ′, Π (fun_wave on interpolated entries)
    double s = qp[ql.wt] * g;
    s = ql.left > 0 ? s : 0.0;
    for (int j = 1; 16 * j < G.nq; ++j) {
        const bool in = j < ql.left;
        const double t = fmaT(qp[in ? ql.wt + 16 * j : 0], I.at(in ? ql.row + ql.step * j : 0), s);
        s = in ? t : s;
    }
    s += dpp64<0x111>(s);
    s += dpp64<0x112>(s);
    s += dpp64<0x114>(s);
    s += dpp64<0x118>(s);
    const double sig = readlane64(s, 15), s0 = readlane64(s, 31);
    FunRows r;
    r.e = readlane64(g, 32); r.t2 = readlane64(g, 33); r.n2 = readlane64(g, 34); r.dl = readlane64(g, 35);
    r.db = readlane64(g, 36); r.t0 = readlane64(g, 37); r.n0 = readlane64(g, 38); r.p2 = readlane64(g, 39);
    r.p0 = readlane64(g, 40);
    const Fun F = fun_finish(C, X, r, sig, s0);
    // the lane's derivative row (source_row's order: 0..2 Θ₁..₃, 3..6 Θᵖ₀..₃,
    // 7 𝒩₂, 8 v_b, 9.. ℳ₂,ᵢ)
    const int kd = W.kinds()[cc];
    double dv = d_coef(G, K, cc, W.rcp_(RC_DI)[cc]) * vc + (W.rcp_(RC_AL)[cc] * K[kd & 255]) * vm +
                (W.rcp_(RC_AU)[cc] * K[(kd >> 8) & 255]) * vp;
    dv += cc == 1 ? (3.0 * X.tp * X.R) * v3 : cc == 3 ? (X.tp * (1.0 / 3.0)) * v1 : 0.0;
    dv += (W.rcp_(RC_CS)[cc] * K[(kd >> 16) & 255]) * F.S + W.rcp_(RC_CP)[cc] * F.P + (W.rcp_(RC_CPI)[cc] * X.tp) * F.Pi;
    dv *= K[kd >> 24];
    // the state after the RSA write (Θ₀, Θ₁ and the ℓ = 2 rows are read below)
    double T0 = r.t0, T1 = readlane64(vc, 0), T2 = r.t2, N2 = r.n2;
    const double T3 = readlane64(vc, 2), vb = readlane64(vc, 8), P0 = r.p0, P1 = readlane64(vc, 4), P2 = r.p2,
                 P3 = readlane64(vc, 6);
    const double ik = 1.0 / k;
    if (X.rsa) {
        const double hk = Hc * ik;
        T0 = r.e - hk * tp * vb;
        T1 = hk * (-2.0 * F.P + tp * (r.e - csb2 * r.db) + hk * (tpp - tp) * vb);
        T2 = 0.0;
        N2 = 0.0;
    }
    const double Pi = T2 + P2 + P0;
    if (om & 1) {
        const bool mrow = lane >= 9 && lane < 9 + G.nq;
        const double sigp = wave_sum(mrow ? qp[2 * G.nq + lane - 9] * dv : 0.0);
        const double dT1 = readlane64(dv, 0), dT2 = readlane64(dv, 1), dT3 = readlane64(dv, 2), dP0 = readlane64(dv, 3),
                     dP1 = readlane64(dv, 4), dP2 = readlane64(dv, 5), dP3 = readlane64(dv, 6), dN2 = readlane64(dv, 7),
                     vbp = readlane64(dv, 8);
        const double iHc = rcp(Hc), q4 = 0.25 / C.rho_crit;
        const double Psi = -r.e - X.c12 * (C.Or * T2 + C.Onu * N2 + sig * q4);
        const double Psip = -F.P - X.c12 * (C.Or * (dT2 - 2.0 * T2) + C.Onu * (dN2 - 2.0 * N2) + (sigp - 2.0 * sig) * q4);
        const double Pip = dT2 + dP2 + dP0, lH = Hcp * iHc;
        const double term1 = gv * (T0 + Psi + 0.25 * Pi) + exp(-readlane64(tv, 7)) * (Psip - F.P);
        const double term2 = -ik * (Hcp * gv * vb + Hc * gp * vb + Hc * gv * vbp);
        const double Pipp = (0.4 * k * iHc) * (dT1 - lH * T1) + 0.3 * (tpp * Pi + tp * Pip) -
                            (0.6 * k * iHc) * ((dT3 + dP1 + dP3) - lH * (T3 + P1 + P3));
        const double term3 = (0.75 * ik * ik) * ((Hcp * Hcp + Hc * Hcpp) * gv * Pi + 3.0 * Hc * Hcp * (gp * Pi + gv * Pip) +
                                                 Hc * Hc * (gpp * Pi + 2.0 * gp * Pip + gv * Pipp));
        if (lane == 0) (obase ? obase + idx : A.out + (size_t)out * C.nx + idx)[0] = term1 + term2 + term3;
    }
    if (om & 2) {
        const double y = k * (readlane64(tv, 11) - eta);
        if (lane == 0) A.out2[(size_t)out * C.nx + idx] = (3.0 / (4.0 * y * y)) * gv * Pi;
    }
    wave_lds_sync();  // es is written again for the next node
}

// ---- the kernel
// w + hγ(c_S y₀ + c_P y₁ + c_Π y₂), the roundings fixed (the compiler's choice
// of which product to fuse would depend on the surrounding code)
__device__ inline double with_border(double w, double hg, double cS, double cP, double cPi, const double* y) {
    return fmaT(hg, fmaT(cPi, y[2], fmaT(cS, y[0], cP * y[1])), w);
}
// KenCarp4's weights of Z_s in the arguments of the stages after s, nearest
// first (row 5: its weight in u_{n+1}, on top of stage 5's argument), and in the
// embedded error.  A stage's argument is accumulated as the stage values come,
// in the order u, Z₀, Z₁, ...
static __constant__ double KC_NEXT[6][4] = {{KCT::A[2][0], KCT::A[3][0], KCT::A[4][0], KCT::A[5][0]},
                                     {KCT::A[2][1], KCT::A[3][1], KCT::A[4][1], KCT::A[5][1]},
                                     {KCT::A[3][2], KCT::A[4][2], KCT::A[5][2], 0},
                                     {KCT::A[4][3], KCT::A[5][3], 0, 0},
                                     {KCT::A[5][4], 0, 0, 0},
                                     {KC_G, 0, 0, 0}};
static __constant__ double KC_ERR[6] = {KCT::A[5][0] - KCT::BH[0], KCT::A[5][1] - KCT::BH[1], KCT::A[5][2] - KCT::BH[2],
                                 KCT::A[5][3] - KCT::BH[3], KCT::A[5][4] - KCT::BH[4], KC_G - KCT::BH[5]};

// SR rows per lane of a scan pass, NP passes; NR rows per thread: n <= 64·SR·NP
// and n <= 256·NR
// (a row block past n is skipped as a whole)
template <int SR, int NP, int NR, class WS_>
__global__ void __launch_bounds__(NTHR) k_solve(SolveArgs A) {
    extern __shared__ __align__(16) double lds[];
    __shared__ int s_mode, s_node;
    const Thr T = thr_self();
    const int wv = __builtin_amdgcn_readfirstlane(T.wv), lane = T.lane;
    // lane 8s + t of wavefront 0 evaluates table t at stage point s; wavefronts
    // 1..3 take (stage point, momentum bin) pairs
    const int xs_s = lane >> 3, xs_t = lane & 7;
    const double xs_c = KC_C[(xs_s < 5 ? xs_s : 4) + 1];
    const int xs_tab = xs_t == 0 ? BOLT_T_HC : xs_t == 1 ? BOLT_T_ETA : xs_t == 2 ? BOLT_T_TAU_P
                     : xs_t == 3 ? BOLT_T_TAU_PP : BOLT_T_CSB2;
    for (;;) {
        if (T.tid == 0) {
            if (A.serve) {
                const int c = serve_claim(A);
                // what the host wrote before publishing (tables, descriptors) is
                // read fresh after this: system-scope acquire
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
                s_mode = c;
            } else {
                s_mode = atomicAdd(A.work_counter, 1);
            }
        }
        __syncthreads();
        const int mi = s_mode;
        if (mi >= A.nmodes) return;
        const ModeDesc md = A.modes[mi];
        const CosmoDev C = A.cosmos[md.cosmo];
        const CfgDev cf = A.cfgs[md.cfg];
        const Geo G = make_geo(cf);
        const int n = G.n, nq = G.nq;
        WS_ W;
        W.b = lds;
        W.n = n;
        W.nq = nq;
        const double k = md.k;
        {
#ifdef BOLT_DEBUG_NANFILL
            // debug build: everything but the vectors' zero padding starts as NaN
            constexpr int NS = WS_::ns;
            for (int i = T.tid; i < A.lds_doubles; i += NTHR) lds[i] = __builtin_nan("");
            __syncthreads();
            for (int i = T.tid; i < WS_::NV * (NS - n); i += NTHR) W.vec(i / (NS - n))[n + i % (NS - n)] = 0.0;
#else
            for (int i = T.tid; i < WS_::T0; i += NTHR) lds[i] = 0.0;
#endif
            __syncthreads();
        }
        if (T.tid < nq) { W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid]; }
        for (int c = T.tid; c < n; c += NTHR) W.u(0)[c] = 0.0;
        setup_rows(C, G, W, T);
        __syncthreads();
        for (int c = n + T.tid; c < WS_::ns; c += NTHR) W.w()[c] = 0.0;  // desc() lay over w
        for (int c = T.tid; c < n; c += NTHR) W.place()[c] = (unsigned short)chain_to_state(G, c);
        initial_conditions(C, G, W, k, W.u(0), T);
        __syncthreads();
        // the outputs at the starting point take the initial condition as saved (f(1)
        // with a weight of zero)
        for (int c = T.tid; c < n; c += NTHR) { W.u(1)[c] = W.u(0)[c]; W.f(1)[c] = 0.0; }
        __syncthreads();
        // owned rows; a row past n is clamped for its loads and never stored
        int rc[NR], rm[NR], rp[NR];
        bool in[NR];
        RowReg R[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            in[i] = T.tid + i * NTHR < n;
            rc[i] = in[i] ? T.tid + i * NTHR : n - 1;
            rm[i] = rc[i] > 0 ? rc[i] - 1 : 0;
            rp[i] = rc[i] + 1 < n ? rc[i] + 1 : rc[i];
            R[i] = load_row(G, W, rc[i]);
        }
        const QLane ql = make_qlane(G, lane);
        const double Or = C.Or, Onu = C.Onu;
        // the border column this wavefront substitutes (1: c_S, 2: c_P, 3: c_Π), in
        // the substitution's layout: constant and scalar-table index per row
        double colc[NP][SR];
        int colk[NP][SR], colp = 0;  // colp: which rows take the RSA factor
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int i = 0; i < SR; ++i) {
                const int c = WAVE * SR * q + SR * lane + i;
                const int kd = c < n ? W.kinds()[c] : 0;
                colc[q][i] = c < n && wv > 0 ? W.rcp_(RC_CS + wv - 1)[c] : 0.0;
                colk[q][i] = (kd >> 16) & 255;
                colp |= (kd >> 24) == K_RSA ? 1 << (SR * q + i) : 0;
            }
        // the LU units of wavefronts 0 and 3: (stage point, segment), one per lane
        const int nseg = W.misc()[0], lu_t = lane + (wv ? WAVE : 0);
        const int lu_st = lu_t / nseg, lu_c0 = lu_t < 5 * nseg ? W.seg()[2 * (lu_t - lu_st * nseg)] : 0,
                  lu_m = lu_t < 5 * nseg ? W.seg()[2 * (lu_t - lu_st * nseg) + 1] : 0;
        const int q_st = (T.tid - WAVE) / nq;
        const double q_c = KC_C[(q_st >= 0 && q_st < 5 ? q_st : 0) + 1];
        long long nacc = 0, nrej = 0, nrhs = 0, nsol = 0;
        double x = C.x0;
        const double xend = C.x1;
        const double rt = cf.reltol, at = cf.abstol;
        int status = BOLT_MODE_OK;
        int next = 0;  // next output index
        const int om = A.serve ? md.pad : A.out_mode;
        double* const obase = A.serve ? A.out + (size_t)(unsigned)md.out : nullptr;
        const int nout = (om == 0) ? A.nsave : C.nx;
        int p = 0;     // u(p), f(p) hold the current state and derivative
        // the dense output still to be taken: nodes pb..pe-1 between xa (u(p^1),
        // f(p^1)) and xb (u(p), f(p))
        int pb = 0, pe = 0;
        double pxa = x, pxb = x;
        auto node = [&](int i) { return om == 0 ? A.x_save[i] : node_x(C, i); };
        double xnext = nout > 0 ? node(0) : 0.0;
        auto crossed = [&](double xn) {
            while (next < nout && xnext <= xn) {
                ++next;
                if (next < nout) xnext = node(next);
            }
        };
        crossed(x);
        pe = next;
        // FSAL start: f(u0) (the RSA overwrite, if on, persists in u)
        {
            const XC X = make_xc(C, k, x);
            qfill(C, G, X, W, T);
            __syncthreads();
            const Fun F = rhs_rows(C, G, X, W, W.qcur(), W.kcur(), W.u(0), 1.0, W.f(0), false, T);
            ++nrhs;
            __syncthreads();
            if (X.rsa && T.tid == 0) rsa_mutate(G, X, k, W.u(0), F.P);
            __syncthreads();
        }
        // Hairer's starting step (order 4)
        double h;
        {
            const double* u = W.u(0);
            const double d0 = wrms(G, W, u, u, u, rt, at, T);
            const double d1 = wrms(G, W, W.f(0), u, u, rt, at, T);
            double h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
            if (h0 > xend - x) h0 = xend - x;
            for (int c = T.tid; c < n; c += NTHR) W.arg()[c] = u[c] + h0 * W.f(0)[c];
            const XC X1 = make_xc(C, k, x + h0);
            qfill(C, G, X1, W, T);
            __syncthreads();
            rhs_rows(C, G, X1, W, W.qcur(), W.kcur(), W.arg(), 1.0, W.w(), false, T);
            ++nrhs;
            __syncthreads();
            for (int c = T.tid; c < n; c += NTHR) W.w()[c] -= W.f(0)[c];
            const double d2 = wrms(G, W, W.w(), u, u, rt, at, T) / h0;
            const double dm = fmax(d1, d2);
            const double h1 = (dm <= 1e-15) ? fmax(1e-6, h0 * 1e-3) : pow(0.01 / dm, 1.0 / 5.0);
            h = fmin(100.0 * h0, h1);
            if (h > xend - x) h = xend - x;
        }
        const int maxsteps = cf.max_steps > 0 ? cf.max_steps : 100000;
        long long nsteps = 0;
        for (;;) {
            // past the end (or a failure) one more turn takes the last step's outputs
            const bool run = status == BOLT_MODE_OK && x < xend && nsteps < maxsteps;
            if (status == BOLT_MODE_OK && x < xend && !run) status = BOLT_MODE_MAXSTEPS;
            if (run) ++nsteps;
            bool last = false;
            if (h >= xend - x) { h = xend - x; last = true; }
            const double hg = h * KC_G;
            if (T.tid == 0) s_node = pb;
            // Z₀ = h f(u) and the first stage's argument
            double a[NR], acc[NR][4], err[NR];
            if (run) {
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    const double u = W.u(p)[rc[i]], z = h * W.f(p)[rc[i]];
                    a[i] = fmaT(KCT::A[1][0], z, u);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = fmaT(KC_NEXT[0][j], z, u);
                    err[i] = KC_ERR[0] * z;
                    if (in[i]) W.arg()[rc[i]] = a[i];
                }
                // the five implicit stage points depend on x and h only: their
                // coefficients, q-quantities, W bands and LU come first, all
                // stages at once.  Wavefront 0: the coefficients, one table per
                // lane, the rest of a point on its first lane; the others: the
                // q-sets, from a = e^x and kH = k/ℋ formed as make_xc forms them
                if (wv == 0) {
                    const double xs = x + xs_c * h;
                    const double tv = spl(C, xs_tab, xs);
                    const double eta = dppz<0x101>(tv), tp = dppz<0x102>(tv), tpp = dppz<0x103>(tv),
                                 csb2 = dppz<0x104>(tv);
                    if (xs_t == 0 && xs_s < 5) {
                        const XC Xs = make_xc_at(C, k, xs, exp(xs), tv, eta, tp, tpp, csb2);
                        store_xs(W.xcs(xs_s), Xs);
                        ktab_head(W.ktab(xs_s), Xs);
                    }
                } else {
                    for (int t = T.tid - WAVE; t < 5 * nq; t += NTHR - WAVE) {
                        const int st = t < NTHR - WAVE ? q_st : t / nq;
                        const double xs = x + (t < NTHR - WAVE ? q_c : KC_C[st + 1]) * h;
                        const double kHs = k * rcp(spl(C, BOLT_T_HC, xs));
                        qfill_one(C, W, exp(xs), kHs, W.qst_base(st), W.ktab(st), t - st * nq);
                    }
                }
                __syncthreads();
                bands_reg<NR>(G, W, R, rc, in, hg, lane);
            }
            __syncthreads();
            // the LU of the five stage points on wavefront 0 while the others
            // form stage 1's right-hand side; the last step's outputs are taken
            // by whichever wavefront is free
            if (run) {
                if (wv > 0)
                    rows_beside<NR>(G, W, R, rc, rm, rp, in, a, 0, ql, Or, Onu, W.arg(), h, W.w(), wv, lane);
                if (wv == 0 || wv == 3) {  // wavefront 3: the units past the first 64
                    for (int t = lu_t, st = lu_st, c0 = lu_c0, m = lu_m; t < 5 * nseg;) {
                        lu_segment(W, W.template bandsT<double>(st), c0, m);
                        t += 2 * WAVE;
                        if (t < 5 * nseg) {
                            st = t / nseg;
                            c0 = W.seg()[2 * (t - st * nseg)];
                            m = W.seg()[2 * (t - st * nseg) + 1];
                        }
                    }
                }
                ++nrhs;
            }
            while (pb < pe) {
                int i = 0;
                if (lane == 0) i = atomicAdd(&s_node, 1);
                i = __builtin_amdgcn_readfirstlane(i);
                if (i >= pe) break;
                const double xv = node(i);
                const DenseIn I = {W.u(p ^ 1), W.u(p), W.f(p ^ 1), W.f(p), hermite(pxa, pxb, xv)};
                emit_wave(C, G, W, A, md.out, k, I, xv, i, lane, om, obase, ql, W.esc(wv));
            }
            pb = pe;
            __syncthreads();
            if (!run) break;
            FacPass<SR> F[NP];
            Cap K;
            double u2 = 0.0;
            for (int s = 1; s < 6; ++s) {
                const double* const Ks = W.ktab(s - 1);
                const Bands B = W.template bandsT<double>(s - 1);
                const StageSc Xs = load_sc(W.xcs(s - 1), lane);
                if (s > 1) {
                    const double* v = W.arg();
                    const Fun Fa = fun_wave(Or, Onu, nq, Xs, W.qst_base(s - 1), ql, v);
                    const KHead H = Xs.head();
                    double r[NR];
#pragma unroll
                    for (int i = 0; i < NR; ++i) {
                        double vm, vp;
                        row_neighbours(a[i], v, rc[i], rm[i], rp[i], lane, vm, vp);
                        r[i] = h * row_eval_reg(R[i], H, Ks[R[i].kx], Ks[R[i].kcs], rc[i], i == 0 && wv == 0, a[i], vm, vp,
                                                v, Fa);
                    }
#pragma unroll
                    for (int i = 0; i < NR; ++i)
                        if (in[i]) W.w()[rc[i]] = r[i];
                    ++nrhs;
                }
                // the factors' part of the substitutions
                double v[NP][SR];
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const int j0 = WAVE * SR * q + SR * lane;
                    fac_prep<SR>(F[q], B, j0, j0 < n, lane);
                    if (wv > 0) {
                        const double rsa = Xs.at(XS_RSA), tp = Xs.at(XS_TP);
                        if (wv == 1) {
#pragma unroll
                            for (int i = 0; i < SR; ++i) v[q][i] = colc[q][i] * Ks[colk[q][i]];
                        } else {
#pragma unroll
                            for (int i = 0; i < SR; ++i) v[q][i] = wv == 2 ? colc[q][i] : colc[q][i] * tp;
                        }
                        if (rsa != 1.0) {
#pragma unroll
                            for (int i = 0; i < SR; ++i) v[q][i] = colp >> (SR * q + i) & 1 ? rsa * v[q][i] : v[q][i];
                        }
                    }
                }
                const double l2 = B.l2c[3];
                u2 = B.u2c[1];
                if (s > 1) __syncthreads();
                double* const bv = wv == 0 ? W.w() : W.c(wv - 1);
                if (wv == 0) {
#pragma unroll
                    for (int q = 0; q < NP; ++q) {
                        const int j0 = WAVE * SR * q + SR * lane;
                        lane_rows<SR>(bv, j0, j0 < n, v[q]);
                    }
                }
                subst_regs<SR, NP>(F, v, l2, u2, lane);
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const int j0 = WAVE * SR * q + SR * lane;
                    store_rows<SR>(bv, j0, j0 < n, v[q]);
                }
                wave_lds_sync();
                ++nsol;
                // the border functionals of the vector this wavefront has solved
                {
                    const Fun Fv = fun_wave(Or, Onu, nq, Xs, W.qst_base(s - 1), ql, bv);
                    if (lane == 0) { W.red()[3 * wv] = Fv.S; W.red()[3 * wv + 1] = Fv.P; W.red()[3 * wv + 2] = Fv.Pi; }
                }
                __syncthreads();
                double y[3];
                {
                    const double* f = W.red();
                    K.m[0][0] = 1.0 - hg * f[3]; K.m[0][1] = -hg * f[6]; K.m[0][2] = -hg * f[9];
                    K.m[1][0] = -hg * f[4]; K.m[1][1] = 1.0 - hg * f[7]; K.m[1][2] = -hg * f[10];
                    K.m[2][0] = -hg * f[5]; K.m[2][1] = -hg * f[8]; K.m[2][2] = 1.0 - hg * f[11];
                    const double rr[3] = {f[0], f[1], f[2]};
                    solve3(K, rr, y);
                }
                double z[NR];
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    const int c = rc[i];
                    z[i] = with_border(W.w()[c], hg, W.c(0)[c], W.c(1)[c], W.c(2)[c], y);
                }
                const double n0 = KC_NEXT[s][0], n1 = KC_NEXT[s][1], n2 = KC_NEXT[s][2], n3 = KC_NEXT[s][3], ke = KC_ERR[s];
                double* const dst = s < 5 ? W.arg() : W.u(p ^ 1);
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    a[i] = fmaT(n0, z[i], acc[i][0]);
                    acc[i][0] = s == 4 ? a[i] : fmaT(n1, z[i], acc[i][1]);  // u_{n+1}: stage 5's argument plus γ Z₅
                    acc[i][1] = fmaT(n2, z[i], acc[i][2]);
                    acc[i][2] = fmaT(n3, z[i], acc[i][3]);
                    err[i] = fmaT(ke, z[i], err[i]);
                    if (in[i]) {
                        dst[rc[i]] = a[i];
                        if (s == 5) W.arg()[rc[i]] = err[i];
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
            if (wv == 0) {
                double v[NP][SR];
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const int j0 = WAVE * SR * q + SR * lane;
                    lane_rows<SR>(W.arg(), j0, j0 < n, v[q]);
                }
                subst_regs<SR, NP>(F, v, W.template bandsT<double>(4).l2c[3], u2, lane);
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const int j0 = WAVE * SR * q + SR * lane;
                    store_rows<SR>(W.arg(), j0, j0 < n, v[q]);
                }
            } else if (spec) {
                Fn = rows_beside<NR>(G, W, R, rc, rm, rp, in, a, 4, ql, Or, Onu, W.u(p ^ 1), 1.0, W.f(p ^ 1), wv, lane);
            }
            ++nsol;
            if (spec) ++nrhs;
            __syncthreads();
            // the border step of the error solve folded into its norm:
            // e_c = ψ_c + hγ(c_S y₀ + c_P y₁ + c_Π y₂) is formed and weighted
            // row by row, never stored
            double en;
            {
                const Fun Fe = fun_wave(Or, Onu, nq, load_sc(W.xcs(4), lane), W.qst_base(4), ql, W.arg());
                const double r[3] = {Fe.S, Fe.P, Fe.Pi};
                double ye[3], ss = 0.0;
                solve3(K, r, ye);
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    if (i > 0 && n <= i * NTHR) continue;
                    const int c = rc[i];
                    const double e = with_border(W.arg()[c], hg, W.c(0)[c], W.c(1)[c], W.c(2)[c], ye);
                    const double sc = fmaT(rt, fmax(fabs(W.u(p)[c]), fabs(a[i])), at);
                    const double q = e / sc;
                    ss = in[i] ? fmaT(q, q, ss) : ss;
                }
                ss = wave_sum(ss);
                if (lane == 0) W.red()[16 + wv] = ss;
                __syncthreads();
                const double* m = W.red() + 16;
                double tot = 0.0;
#pragma unroll
                for (int i = 0; i < NWAVE; ++i) tot += m[i];
                en = sqrt(tot / n);
            }
            if (!isfinite(en)) {
                // the forward scans carried the non-finite values into rows n.. of the
                // two vectors that wavefront 0 solves in place, where the backward
                // scans of the next, shorter step begin: zero again
                for (int c = n + T.tid; c < WS_::ns; c += NTHR) W.w()[c] = W.arg()[c] = 0.0;
                ++nrej;
                h *= 0.2;
                if (h < 1e-14) status = BOLT_MODE_NONFINITE;
                continue;
            }
            if (en <= 1.0) {
                const double xn = last ? xend : x + h;
                // FSAL at x_{n+1} (already evaluated unless the step ends on xend)
                if (spec) {
                    // Fn is held by wavefronts 1..
                    if (wv == 1 && lane == 0 && W.xcs(4)[XS_RSA] == 0.0) rsa_mutate(G, rsa_xc(W.xcs(4)), k, W.u(p ^ 1), Fn.P);
                } else {
                    const XC Xn = make_xc(C, k, xn);
                    qfill(C, G, Xn, W, T);
                    __syncthreads();
                    Fn = rhs_rows(C, G, Xn, W, W.qcur(), W.kcur(), W.u(p ^ 1), 1.0, W.f(p ^ 1), false, T);
                    ++nrhs;
                    __syncthreads();
                    if (Xn.rsa && wv == 1 && lane == 0) rsa_mutate(G, Xn, k, W.u(p ^ 1), Fn.P);
                }
                __syncthreads();
                ++nacc;
                pb = next;
                crossed(xn);
                pe = next;
                pxa = x;
                pxb = xn;
                p ^= 1;
                x = xn;
                double fac = (en == 0.0) ? 10.0 : 0.9 * pow(en, -0.25);
                fac = fmin(10.0, fmax(0.2, fac));
                h *= fac;
            } else {
                ++nrej;
                const double fac = fmin(1.0, fmax(0.2, 0.9 * pow(en, -0.25)));
                h *= fac;
                if (h < 1e-14 * fmax(1.0, fabs(x))) status = BOLT_MODE_DTMIN;
            }
        }
        if (T.tid == 0) {
            const int si = A.serve ? mi : md.out;
            A.status[si] = status;
            if (A.counters) {
                long long* cc = A.counters + (size_t)si * 4;
                cc[0] = nacc; cc[1] = nrej; cc[2] = nrhs; cc[3] = nsol;
            }
            if (A.serve) {
                // the workgroup's outputs (ordered before this thread by the
                // barrier above) reach memory, then the host's flag is raised
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
                __hip_atomic_store(A.done + mi, A.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        __syncthreads();
    }
}

// The instantiations with SOLVE_SR scan rows per lane (this file is compiled once
// for each): one owned row per thread up to 256 rows, two up to 512, and the scan
// passes the layout's rows take.
#define SOLVE_CAT2(a, b) a##b
#define SOLVE_CAT(a, b) SOLVE_CAT2(a, b)
const void* SOLVE_CAT(solver_kernel_sr, SOLVE_SR)(int layout) {
    constexpr int SR = SOLVE_SR;
    constexpr auto passes = [](int n) { return (n + WAVE * SR - 1) / (WAVE * SR); };
    switch (layout) {
        case 0: return (const void*)k_solve<SR, 1, 1, WSN0>;
        case 1: return (const void*)k_solve<SR, passes(WSN1::nmax), 2, WSN1>;
        case 2: return (const void*)k_solve<SR, passes(2 * NTHR), 2, WSN2>;
        default: return (const void*)k_solve<SR, 2, 3, WSN3>;
    }
}
