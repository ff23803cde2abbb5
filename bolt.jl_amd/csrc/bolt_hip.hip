// libbolt_hip: MI355X (gfx950) kernels for Bolt.jl's perturbation hot path and
// the C ABI declared in include/bolt_hip.h.
//
// Integrator design.  hierarchy! (src/perturbations.jl:161-271) is linear in
// the state: du = A(x) u.  Writing A = L + c_S sᵀ + c_P pᵀ + c_Π πᵀ, where L
// couples each hierarchy only to its ℓ±1 neighbours (plus the baryon/photon
// tight-coupling pair) and s, p, π are the Ψ, Φ′ and Π functionals, the
// KenCarp4 stage equation (I - hγA) z = r is solved exactly by
//   * a banded LU (bandwidth <= 2, no pivoting: every chain is a positive
//     diagonal plus a skew-symmetrisable coupling) of I - hγL, one lane per
//     segment of consecutive chains,
//   * a 3x3 capacitance system for the Ψ/Φ′/Π border (Woodbury).
// One workgroup of four wavefronts (one per SIMD) integrates one k-mode: row
// passes spread over its 256 lanes, the four right-hand sides of a stage solve
// run on the four wavefronts at once.  State vectors live in LDS in "chain
// order" (each hierarchy contiguous); a persistent grid pulls modes from an
// atomic work counter, costliest (largest k) first.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <tuple>
#include <climits>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include "../../include/bolt_hip.h"
#include "host_tables.h"

namespace bolt {
int set_error(int code, const std::string& msg);
}
using bolt::set_error;

#include "solve_layout.h"

// hierarchy! parity hook: one wavefront per mode, u/du [n][B]
__global__ void __launch_bounds__(WAVE) k_rhs(const CosmoDev* cosmos, const CfgDev* cfgs, const ModeDesc* modes,
                                               int B, double x, double* u, double* du, int mutate) {
    extern __shared__ double lds[];
    const Thr T = thr_self();
    const int mi = blockIdx.x;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    Geo G = make_geo(cfgs[md.cfg]);
    WS W;
    ws_bind(W, lds, G.n, G.nq);
    if (T.tid < G.nq) { W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid]; }
    for (int c = T.tid; c < G.n; c += T.nt) W.arg()[c] = u[(size_t)chain_to_state(G, c) * B + mi];
    setup_rows(C, G, W, T);
    XC X = make_xc(C, md.k, x);
    qfill(C, G, X, W, T);
    __syncthreads();
    Fun F = rhs_rows(C, G, X, W, W.qcur(), W.kcur(), W.arg(), 1.0, W.w(), false, T);
    __syncthreads();
    if (mutate && X.rsa && T.tid == 0) rsa_mutate(G, X, md.k, W.arg(), F.P);
    __syncthreads();
    for (int c = T.tid; c < G.n; c += T.nt) {
        size_t o = (size_t)chain_to_state(G, c) * B + mi;
        du[o] = W.w()[c];
        if (mutate) u[o] = W.arg()[c];
    }
}

__global__ void __launch_bounds__(WAVE) k_ics(const CosmoDev* cosmos, const CfgDev* cfgs, const ModeDesc* modes,
                                               int B, double* u0) {
    extern __shared__ double lds[];
    const Thr T = thr_self();
    const int mi = blockIdx.x;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    Geo G = make_geo(cfgs[md.cfg]);
    WS W;
    ws_bind(W, lds, G.n, G.nq);
    if (T.tid < G.nq) { W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid]; }
    for (int c = T.tid; c < G.n; c += T.nt) W.u()[c] = 0.0;
    __syncthreads();
    initial_conditions(C, G, W, md.k, W.u(), T);
    __syncthreads();
    for (int c = T.tid; c < G.n; c += T.nt) u0[(size_t)chain_to_state(G, c) * B + mi] = W.u()[c];
}

// tangent of hierarchy! (parity hook): du̇ = f(u̇) + L̇u for every mode at x,
// one wavefront per mode; u, u̇, du̇ [n][B] in Bolt's order
__global__ void __launch_bounds__(WAVE) k_rhs_jvp(const CosmoDev* cosmos, const CosmoDev* cosmos_dot,
                                                   const CfgDev* cfgs, const ModeDesc* modes, int B, double x,
                                                   const double* u, const double* ud, double* dud) {
    extern __shared__ double lds[];
    const Thr T = thr_self();
    const int mi = blockIdx.x;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    const CosmoDev& Cd = cosmos_dot[md.cosmo];
    Geo G = make_geo(cfgs[md.cfg]);
    WS W;
    ws_bind(W, lds, G.n, G.nq);
    WTan Wt;
    Wt.b = lds + wtan_offset(G.n, G.nq);
    Wt.n = G.n;
    Wt.nq = G.nq;
    if (T.tid < G.nq) {
        W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid];
        Wt.qd()[T.tid] = Cd.qv[T.tid]; Wt.df0d()[T.tid] = Cd.df0[T.tid]; Wt.based()[T.tid] = Cd.base[T.tid];
    }
    for (int c = T.tid; c < G.n; c += T.nt) {
        const size_t o = (size_t)chain_to_state(G, c) * B + mi;
        W.arg()[c] = u[o];
        Wt.argd()[c] = ud[o];
    }
    setup_rows(C, G, W, T);
    __syncthreads();
    const XC X = make_xc(C, md.k, x);
    qfill(C, G, X, W, T);
    const XCd D = make_xcd(C, Cd, X);
    if (T.tid < G.nq) qfill_one_dot(C, Cd, W, Wt, X.a, X.kH, D.kH, W.qe(), Wt.qset_base(5), Wt.ktd(5), T.tid);
    if (T.tid == T.nt - 1) ktab_head_dot(Wt.ktd(5), X, D);
    __syncthreads();
    rhs_rows_tan(C, Cd, G, X, D, W, W.qcur(), Wt.qset(5), W.kcur(), Wt.ktd(5), Wt.argd(), W.arg(), 1.0, Wt.wd(), T);
    __syncthreads();
    for (int c = T.tid; c < G.n; c += T.nt) dud[(size_t)chain_to_state(G, c) * B + mi] = Wt.wd()[c];
}

// initial_conditions and their tangent (parity hook); u0, u̇0 [n][B]
__global__ void __launch_bounds__(WAVE) k_ics_jvp(const CosmoDev* cosmos, const CosmoDev* cosmos_dot,
                                                   const CfgDev* cfgs, const ModeDesc* modes, int B, double* u0,
                                                   double* ud0) {
    extern __shared__ double lds[];
    const Thr T = thr_self();
    const int mi = blockIdx.x;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    const CosmoDev& Cd = cosmos_dot[md.cosmo];
    Geo G = make_geo(cfgs[md.cfg]);
    WS W;
    ws_bind(W, lds, G.n, G.nq);
    WTan Wt;
    Wt.b = lds + wtan_offset(G.n, G.nq);
    Wt.n = G.n;
    Wt.nq = G.nq;
    if (T.tid < G.nq) {
        W.q()[T.tid] = C.qv[T.tid]; W.df0()[T.tid] = C.df0[T.tid]; W.base()[T.tid] = C.base[T.tid];
        Wt.qd()[T.tid] = Cd.qv[T.tid]; Wt.df0d()[T.tid] = Cd.df0[T.tid]; Wt.based()[T.tid] = Cd.base[T.tid];
    }
    for (int c = T.tid; c < G.n; c += T.nt) { W.u()[c] = 0.0; Wt.ud()[c] = 0.0; }
    __syncthreads();
    initial_conditions_t<D1>(C, &Cd, G, W, &Wt, md.k, W.u(), Wt.ud(), T);
    __syncthreads();
    for (int c = T.tid; c < G.n; c += T.nt) {
        const size_t o = (size_t)chain_to_state(G, c) * B + mi;
        u0[o] = W.u()[c];
        ud0[o] = Wt.ud()[c];
    }
}

// rsa_perts! after the switch node (perturbations.jl:35-111); one thread per (mode, node)
__global__ void k_rsa_post(const CosmoDev* cosmos, const CfgDev* cfgs, const ModeDesc* modes, int B, double* out) {
    int mi = blockIdx.y;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    const CfgDev cf = cfgs[md.cfg];
    int nx = C.nx, n = cf.n;
    double k = md.k;
    // switch node (identical scan in every thread of the mode)
    int ihor = -1, iod = -1;
    for (int j = 0; j < nx && (ihor < 0 || iod < 0); ++j) {
        double xj = (C.x0 * (nx - 1 - j) + C.x1 * j) / (nx - 1);
        double eta = spl(C, BOLT_T_ETA, xj), Hc = spl(C, BOLT_T_HC, xj), tp = spl(C, BOLT_T_TAU_P, xj);
        if (ihor < 0 && k * eta > 240.0) ihor = j;
        if (iod < 0 && -tp * Hc / eta > 100.0) iod = j;
    }
    if (ihor < 0) ihor = nx - 1;
    if (iod < 0) iod = nx - 1;
    int isw = ihor > iod ? ihor : iod;
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nx) return;
    double xsw = (C.x0 * (nx - 1 - isw) + C.x1 * isw) / (nx - 1);
    double xj = (C.x0 * (nx - 1 - j) + C.x1 * j) / (nx - 1);
    if (!(xj > xsw)) return;
    double* u = out + ((size_t)md.out * nx + j) * n;
    int ng = cf.ng, nn = cf.nn, nm = cf.nm, nq = cf.nq;
    int iN = 2 * (ng + 1), iM = iN + nn + 1, iPhi = iM + (nm + 1) * nq;
    double a = exp(xj), Hc = spl(C, BOLT_T_HC, xj), tp = spl(C, BOLT_T_TAU_P, xj), tpp = spl(C, BOLT_T_TAU_PP, xj);
    double csb2 = spl(C, BOLT_T_CSB2, xj);
    double sr = 0, ss = 0;
    for (int i = 0; i < nq; ++i) {
        double q = C.qv[i], eps = sqrt(q * q + (a * C.mnu) * (a * C.mnu));
        sr += C.base[i] * eps * u[iM + i];
        ss += C.base[i] * (q * q / eps) * u[iM + 2 * nq + i];
    }
    double H02 = C.H0 * C.H0, Phi = u[iPhi];
    double Psi = -Phi - 12.0 * H02 / (k * k) / (a * a) * (C.Or * u[2] + C.Onu * u[iN + 2] + ss / C.rho_crit / 4.0);
    double Phip = Psi - k * k / (3.0 * Hc * Hc) * Phi +
                  H02 / (2.0 * Hc * Hc) * (C.Oc / a * u[iPhi + 1] + C.Ob / a * u[iPhi + 3] + 4.0 * C.Or / (a * a) * u[0] +
                                           4.0 * C.Onu / (a * a) * u[iN] + sr / C.rho_crit / (a * a));
    double db = u[iPhi + 3], vb = u[iPhi + 4];
    double T0 = Phi - Hc / k * tp * vb;
    double T1 = Hc / k * (-2.0 * Phip + tp * (Phi - csb2 * db) + Hc / k * (tpp - tp) * vb);
    u[0] = T0; u[1] = T1; u[2] = 0.0;
    u[iN] = Phi; u[iN + 1] = -2.0 * Hc / k * Phip; u[iN + 2] = 0.0;
    for (int l = 3; l <= ng; ++l) { u[l - 1] = 0.0; u[(ng + 1) + l - 1] = 0.0; }
    for (int l = 3; l <= nn; ++l) u[iN + l - 1] = 0.0;
}

// plin's gauge transform and normalisation (spectra.jl:169-197), one thread per mode
__global__ void k_plin_post(const CosmoDev* cosmos, const CfgDev* cfgs, const ModeDesc* modes, int B, double x,
                            const double* states, double* pk, int stride) {
    // stride: doubles between consecutive modes' states (0: the state length)
    int mi = blockIdx.x * blockDim.x + threadIdx.x;
    if (mi >= B) return;
    ModeDesc md = modes[mi];
    const CosmoDev C = cosmos[md.cosmo];
    const CfgDev cf = cfgs[md.cfg];
    const double* u = states + (size_t)md.out * (stride ? stride : cf.n);
    double k = md.k, a = exp(x);
    int ng = cf.ng, nn = cf.nn, nm = cf.nm, nq = cf.nq;
    int iM = 2 * (ng + 1) + nn + 1, iPhi = iM + (nm + 1) * nq;
    double rho0 = spl(C, BOLT_T_RHO0M, x);
    double sr = 0, th = 0;
    for (int i = 0; i < nq; ++i) {
        double q = C.qv[i], eps = sqrt(q * q + (a * C.mnu) * (a * C.mnu));
        sr += C.base[i] * eps * u[iM + i];
        th += C.thbase[i] * u[iM + nq + i];
    }
    double Mrho = sr / rho0;
    double Mtheta = k * th / rho0;
    double dcN = u[iPhi + 1], vcN = u[iPhi + 2], dbN = u[iPhi + 3], vbN = u[iPhi + 4];
    double vmN = -Mtheta / k;
    double Om = C.Oc + C.Ob + C.Om_nu_nr;
    double Hc = spl(C, BOLT_T_HC, x);
    double dc = dcN - 3.0 * Hc * vcN / k;
    double db = dbN - 3.0 * Hc * vbN / k;
    double dmn = Mrho - 3.0 * Hc * vmN / k;
    double dm = (C.Oc * dc + C.Ob * db + C.Om_nu_nr * dmn) / Om;
    double Pprim = C.Pprim_A * pow(k / 0.05, C.Pprim_n - 1.0);
    pk[md.out] = (2.0 * M_PI * M_PI / (k * k * k)) * dm * dm * Pprim;
}

// ---------------------------------------------------------------- LOS (C_ℓ)
// T_ℓ(k) = Σ_x j_ℓ(k(η₀-η(x))) S(x,k) Δx  (spectra.jl:70-82), all ℓ <= lmax at
// once by the upward recurrence j_{ℓ+1} = (2ℓ+1)/z j_ℓ - j_{ℓ-1}.  Past the
// turning point ((2ℓ+1)/z > 2) the slot ends once |j_ℓ| < 1e-7 max|j| or once
// |j_ℓ| grows (there the true j_ℓ decays monotonically, so growth means the
// recurrence's growing solution has taken over).
// One block per dense-k midpoint at a time; lanes own x nodes (slots of 64
// consecutive nodes); ℓ runs in chunks of 16 reduced across the lanes in registers
// and, every SPAN multipoles, across the wavefronts through LDS.
// NS = 1: one source (C_ℓ^TT, or C_ℓ^EE with the spin factor); NS = 2: the
// temperature and polarization sources share each j_ℓ and give TT, TE, EE.
#define LOS_SLOTS 16   // x slots of 64 nodes (up to 1024 nodes after x = -8)
// blocks of one LOS launch: block b takes the dense-k midpoints b, b + grid,
// b + 2·grid, ... (a spread over k, so blocks cost about the same) and sums
// their C_ℓ contributions into a row of its own.  Fixed, so that the
// summation order, and with it every bit of C_ℓ, does not depend on the device
// Three blocks a CU, which is what k_los<1, 4>'s registers leave room for: the third
// fills the issue slots in which the wavefronts of the other two wait for each other
// (512 blocks at two a CU: 1.7 ms at 2500 ℓ x 4999 k against 1.3; TT/TE/EE, which has
// room for two a CU, the same to 1 %; 1024 blocks: 1.5).
#define LOS_GRID 768
#define LOS_SPW_DEFAULT 4  // x slots per wavefront (LOS_SLOTS/SPW wavefronts per block): 1, 2 or 4
#define LOS_TAU 1e-7
// lanes with z < LOS_ZS take j_ℓ from its ascending series
//   j_ℓ(z) = z^ℓ Σ_m c_{ℓ,m} z^{2m},  c_{ℓ,m} = (-1/2)^m / (m! (2ℓ+2m+1)!!),
// which has no cancellation there (the upward recurrence loses digits for
// z < ℓ), and run until |j_ℓ| < LOS_TAU_SMALL max|j| or ℓ = JSER_L: there the
// polarization source (∝ 1/z²) makes terms far below the cut above count.
#define LOS_ZS 2.0
#define LOS_ZL 32.0  // a wavefront whose live lanes have z >= LOS_ZL takes the short recurrences
// from this ℓ on no lane with z < LOS_ZL is left: the slowest, z = 32, is cut at
// ℓ = 52, and the series ends before JSER_L
#define LOS_LEAN 64
#define LOS_TAU_SMALL 1e-30
#define JSER_L 48
#define JSER_M 14
__device__ double c_jser[JSER_L][JSER_M];  // global, not constant: see jser

static void fill_jser(double* c) {
    for (int l = 0; l < JSER_L; ++l)
        for (int m = 0; m < JSER_M; ++m) {
            long double v = 1.0L;
            for (int i = 1; i <= m; ++i) v /= -2.0L * i;           // (-1/2)^m / m!
            for (int i = 1; i <= 2 * l + 2 * m + 1; i += 2) v /= i;  // / (2ℓ+2m+1)!!
            c[l * JSER_M + m] = (double)v;
        }
}

// inlined; in the unrolled ℓ loop each ℓ's coefficient loads stay behind a
// compiler barrier (los_slot_series), so they are not all hoisted together
__device__ inline double jser(int l, double w, double zl) {
    const double* c = c_jser[l];
    double F = c[JSER_M - 1];
#pragma unroll
    for (int m = JSER_M - 2; m >= 0; --m) F = fma(F, w, c[m]);
    return F * zl;
}

struct LosArgs {
    const CosmoDev* cosmo;
    const double* S;      // [nk_src][nx]
    const double* SP;     // [nk_src][nx] second source (NS = 2)
    const double* k_src;  // [nk_src]
    int nk_src;
    const double* kgrid;  // [nkd]
    int nkd;
    const int* lidx;      // [lmax+1] column of ℓ among the distinct requested ℓ, or -1
    int lmax;
    int nu;               // distinct requested ℓ
    const double* etaj;   // [nxi] η at the integration nodes
    const double* dxj;    // [nxi] x_{j+1}-x_j
    int i0, nxi;
    int spin;             // NS = 1: multiply T_ℓ by ℓð (E modes)
    double* partial;      // [grid][nout][nu] per-block sums over its midpoints; nout = 1 (NS = 1), 3 (NS = 2:
                          // TT, TE, EE) or 2 (NS = 3: TT and its derivative)
    long long* steps;     // executed recurrence steps (per k), may be NULL
    // NS = 3, the derivative along a parameter direction: SP is dS/dp, etajd
    // dη/dp at the integration nodes, eta0d dη₀/dp, dlnA and dns the
    // derivatives of ln A_s and n_s
    const double* etajd = nullptr;
    double eta0d = 0.0, dlnA = 0.0, dns = 0.0;
};

__global__ void k_los_prep(const CosmoDev* cosmo, int i0, int nxi, double* etaj, double* dxj) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nxi) return;
    const CosmoDev C = *cosmo;
    double xa = (C.x0 * (C.nx - 1 - (i0 + j)) + C.x1 * (i0 + j)) / (C.nx - 1);
    double xb = (C.x0 * (C.nx - 1 - (i0 + j + 1)) + C.x1 * (i0 + j + 1)) / (C.nx - 1);
    etaj[j] = spl(C, BOLT_T_ETA, xa);
    dxj[j] = xb - xa;
}

// dη/dp at the integration nodes, from the tangent tables (same x nodes)
__global__ void k_los_prep_dot(const CosmoDev* cosmo_dot, int i0, int nxi, double* etajd) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nxi) return;
    const CosmoDev Cd = *cosmo_dot;
    double xa = (Cd.x0 * (Cd.nx - 1 - (i0 + j)) + Cd.x1 * (i0 + j)) / (Cd.nx - 1);
    etajd[j] = spl(Cd, BOLT_T_ETA, xa);
}

// ℓð = √((ℓ+2)(ℓ+1)ℓ(ℓ−1)) (spectra.jl:101, 119), the product exact in 64 bits
__device__ inline double spin_factor(int l) {
    long long L = l;
    return sqrt((double)((L + 2) * (L + 1) * L * (L - 1)));
}

// one lane's state of one x slot: z = k (η₀ − η), j_{ℓ−2}, j_{ℓ−1}, 1/z, the
// source times Δx and (NS = 2: the second source; NS = 3: its derivative, and
// zs = ż s with ż = k (dη₀/dp − dη/dp)), the largest |j| so far, z^ℓ of the
// series.  A lane past its cut, or without a node, has jp = jc = iz = 0: every
// further j_ℓ is zero.  n: the wavefront's lanes that still count.
struct LosLane {
    double jp, jc, iz, s, sp, zs, M, z, zl;
    int n;
};

// votes as comparisons of a ballot with zero: known to be the same for the whole
// wavefront, so that the compiler branches around a path instead of masking it
__device__ inline bool los_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }
__device__ inline bool los_none(bool p) { return __builtin_amdgcn_ballot_w64(p) == 0; }
// t = (2ℓ−1)/z, which produces j_ℓ: 2ℓ−1 as the low bits of 2⁵² + 2ℓ−1, a scalar
// register pair without a conversion; the fma takes 2⁵²/z off again and rounds once,
// to the same value as the product
__device__ inline double los_t(const LosLane& q, int l) {
    return __builtin_fma(__hiloint2double(0x43300000, 2 * l - 1), q.iz, -0x1p52 * q.iz);
}
// take the lanes past their cut out
__device__ inline void los_drop(LosLane& q, bool live) {
    q.n = __popcll(__builtin_amdgcn_ballot_w64(live));
    q.jp = live ? q.jp : 0.0;
    q.jc = live ? q.jc : 0.0;
    q.iz = live ? q.iz : 0.0;
}
// the terms of one ℓ, v = j_ℓ (zero past the cut), vp = j_{ℓ−1} − (ℓ+1)/z j_ℓ = j′_ℓ
template <int NS>
__device__ inline void los_add(const LosLane& q, double v, double vp, double& acc, double& accp) {
    acc += v * q.s;
    if constexpr (NS == 2) accp += v * q.sp;
    if constexpr (NS == 3) accp += v * q.sp + vp * q.zs;
}

// Advance one x slot through ℓ = L0+I0 .. L0+CH-1, accumulating j_ℓ s (and j_ℓ sp;
// NS = 3: the derivative j_ℓ ṡ + j′_ℓ ż s of the term).  SERIES: the wavefront holds
// live lanes with z < LOS_ZS, which take the series (zl carries z^ℓ).
template <int NS, int CH, int I0, bool SERIES>
__device__ inline void los_slot(LosLane& q, int L0, double* acc, double* accp, int& nstep) {
    bool live = q.iz != 0.0;
    const double w = SERIES ? q.z * q.z : 0.0;
#pragma unroll
    for (int i = I0; i < CH; ++i) {
        const int l = L0 + i;
        const double t = los_t(q, l);
        double jn;
        bool cut;
        if (SERIES) asm volatile("" ::: "memory");  // keeps this ℓ's series coefficients' loads here
        if (SERIES && q.z < LOS_ZS) {
            q.zl *= q.z;
            jn = (live && l < JSER_L) ? jser(l, w, q.zl) : 0.0;
            cut = !(fabs(jn) >= LOS_TAU_SMALL * q.M) || l >= JSER_L;
        } else {
            // past the turning point j_ℓ decays monotonically: a term below
            // LOS_TAU·max or a growing one (the recurrence's error has taken over)
            // ends the slot
            jn = t * q.jc - q.jp;
            cut = t > 2.0 && (fabs(jn) < LOS_TAU * q.M || fabs(jn) > fabs(q.jc));
        }
        live = live && !cut;
        q.jp = q.jc;
        q.jc = jn;
        q.M = fmax(q.M, fabs(jn));
        nstep += __popcll(__builtin_amdgcn_ballot_w64(live));
        los_add<NS>(q, live ? jn : 0.0, NS == 3 && live ? q.jp - (double)(l + 1) * q.iz * jn : 0.0, acc[i], accp[i]);
    }
    los_drop(q, live);
}

// los_slot for a wavefront whose live lanes all have z >= LOS_ZL, with its chunk's
// last t above 1.5.  Up to t = 2 no cut can apply: four instructions a step.  From
// there on a lane is tested in the chunks that begin past its turning point: from
// z = LOS_ZL up j_ℓ is still above 2e-6 of its maximum CH multipoles on, so no cut
// falls into the chunk before, and past t = 2 the maximum stays.
template <int NS, int CH, int I0>
__device__ inline void los_slot_turn(LosLane& q, int L0, double* acc, double* accp, int& nstep) {
    if (los_none(los_t(q, L0 + CH - 1) > 2.0)) {
#pragma unroll
        for (int i = I0; i < CH; ++i) {
            const double jn = los_t(q, L0 + i) * q.jc - q.jp;
            q.jp = q.jc;
            q.jc = jn;
            q.M = fmax(q.M, fabs(jn));
            los_add<NS>(q, jn, q.jp - (double)(L0 + i + 1) * q.iz * jn, acc[i], accp[i]);
        }
        nstep += (CH - I0) * q.n;
        return;
    }
    bool live = q.iz != 0.0;
    const bool past = los_t(q, L0 + I0) > 2.0;
    const double thr = past ? LOS_TAU * q.M : 0.0;
#pragma unroll
    for (int i = I0; i < CH; ++i) {
        const double jn = los_t(q, L0 + i) * q.jc - q.jp;
        if (fabs(jn) < thr || (past && fabs(jn) > fabs(q.jc))) live = false;
        q.jp = q.jc;
        q.jc = jn;
        q.M = fmax(q.M, fabs(jn));
        nstep += __popcll(__builtin_amdgcn_ballot_w64(live));
        los_add<NS>(q, live ? jn : 0.0, NS == 3 && live ? q.jp - (double)(L0 + i + 1) * q.iz * jn : 0.0, acc[i], accp[i]);
    }
    los_drop(q, live);
}

// SPW lanes' states as separate members: an array would be kept as one register
// tuple that every update copies
template <int SPW>
struct LosLanes {
    LosLane q;
    LosLanes<SPW - 1> rest;
    template <int SL = 0, class F>
    __device__ __forceinline__ void each(F&& f) {
        f(q, std::integral_constant<int, SL>{});
        rest.template each<SL + 1>(f);
    }
};
template <>
struct LosLanes<0> {
    template <int SL = 0, class F>
    __device__ __forceinline__ void each(F&&) {}
};

// The first N slots of a wavefront through one chunk with t = (2ℓ−1)/z <= 1.5 up to
// its last ℓ on every lane: neither the cut nor the maximum of |j| falls here.  (At
// fixed z the largest |j_ℓ| is the last one before the turning point, at ℓ ≈ z −
// 0.81 z^{1/3}, the Airy maximum; at z = 32 it is 0.048, against 0.037 for all ℓ up
// to t = 1.5, and the ratio grows with z.)  Three instructions a step, the slots'
// recurrences side by side and without a branch.
template <int NS, int CH, int N, int SPW>
__device__ inline void los_below(LosLanes<SPW>& Q, int L0, double* acc, double* accp, int& nstep) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
        Q.each([&](LosLane& q, auto sl) {
            if constexpr (decltype(sl)::value < N) {
                const double jn = los_t(q, L0 + i) * q.jc - q.jp;
                q.jp = q.jc;
                q.jc = jn;
                los_add<NS>(q, jn, q.jp - (double)(L0 + i + 1) * q.iz * jn, acc[i], accp[i]);
            }
        });
    Q.each([&](LosLane& q, auto sl) { nstep += decltype(sl)::value < N ? CH * q.n : 0; });
}

// the two registers' halves traded so that their sum is a on the lanes whose bit
// 32 (16) is clear and b on the others: v_permlane32_swap, v_permlane16_swap
__device__ inline double fold32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ inline double fold16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
// the same across bit 8 and bit 4 of the lane: DPP moves inside a row of 16, a
// bank (four lanes) masked off keeping its own value
template <int CTRL_UP, int BANKS_UP, int CTRL_DN, int BANKS_DN>
__device__ inline double fold_row(double a, double b) {
    auto mv = [](double old, double v, auto ctrl, auto banks) {
        const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), decltype(ctrl)::value, 0xF,
                                                   decltype(banks)::value, false);
        const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), decltype(ctrl)::value, 0xF,
                                                   decltype(banks)::value, false);
        return __hiloint2double(hi, lo);
    };
    const double t = mv(a, b, std::integral_constant<int, CTRL_UP>{}, std::integral_constant<int, BANKS_UP>{});
    const double u = mv(b, a, std::integral_constant<int, CTRL_DN>{}, std::integral_constant<int, BANKS_DN>{});
    return t + u;
}
// reduce-scatter of acc[16] over the wavefront, in registers: lane l returns
// Σ_lanes acc[l / 4].  57 VALU instructions; through __shfl_xor (LDS) and selects
// it was 170 and six LDS round trips a chunk.
__device__ inline double los_reduce(const double* acc) {
    double a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = fold32(acc[i], acc[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = fold16(a[i], a[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = fold_row<0x128, 0xC, 0x128, 0x3>(a[i], a[i + 2]);  // row_ror 8
    double T = fold_row<0x114, 0xA, 0x104, 0x5>(a[0], a[1]);                              // row_shr 4, row_shl 4
    T += dpp64<0xB1>(T);  // quad_perm 1,0,3,2
    T += dpp64<0x4E>(T);  // quad_perm 2,3,0,1
    return T;
}

// j₀(z), j₁(z): the ascending series below LOS_ZS, sin/cos above.  Out of
// line: inlined, the polynomial constants of sincos stay live across the
// block's whole midpoint loop and crowd out the recurrence's registers.
__device__ __attribute__((noinline)) double2 los_j01(double z) {
    if (z < LOS_ZS) return make_double2(jser(0, z * z, 1.0), jser(1, z * z, z));
    double sn, cs;
    sincos(z, &sn, &cs);
    const double j0 = sn / z;
    return make_double2(j0, (j0 - cs) / z);
}

// A (k/0.05)^(n−1) Δk/k, out of line for the same reason
__device__ __attribute__((noinline)) double los_pw(double A_s, double n_s, double k, double dk) {
    return A_s * pow(k / 0.05, n_s - 1.0) * dk / k;
}

// T_ℓ(k) = Σ_x j_ℓ(k(η₀−η)) S(x, k) Δx for every requested ℓ, and the
// C_ℓ contributions T_ℓ² P(k) Δk/k summed over the block's midpoints.
// A block of LOS_SLOTS/SPW wavefronts; wavefront w owns x slots w, w + W, ...
// (SPW of them).  Each wavefront runs SPAN multipoles on its own, chunk by
// chunk, its partial T_ℓ kept in LDS; then the block adds its wavefronts' partials
// and the row entries (entry ℓ is always read and written by the same thread).
// What bounds it: FP64 issue.  2500 ℓ x 4999 k x 799 x are 5.7e7 wavefront steps, of
// three instructions where nothing can be cut (los_below, 70 % of them), four up to
// the turning point and a dozen past it.  With the cut tested in every step (20
// instructions) and a reduction through LDS with two barriers every 16 ℓ it was
// 5.9 ms (9.0e8 VALU instructions); it is 1.3 ms (4.7e8, of which the reductions
// are a fifth), three quarters of the VALU's issue slots; the rest is the wavefronts'
// unequal shares between two exchanges (13 slots over 4).  TT, TE and EE of 1499 ℓ x
// 3000 k: 4.0 -> 1.2 ms.
// SPW: four slots a wavefront share one reduction and four independent chains; two
// take 25 % more instructions, the same time for NS = 1 and 1.2 times as long for
// NS = 2, so four is the default.
template <int NS, int SPW>
__global__ void __launch_bounds__(LOS_SLOTS / SPW * WAVE, SPW == 1 || (SPW == 2 && NS == 1) ? 4 : NS == 1 ? 3 : 2) k_los(LosArgs A) {
    constexpr int CH = 16;  // ℓ per chunk (NA·CH accumulators per lane)
    constexpr int NW = LOS_SLOTS / SPW;
    constexpr int SPAN = SPW == 4 ? 256 : 128;  // multipoles between two exchanges of the block's wavefronts
    constexpr int NA = NS == 1 ? 1 : 2;                    // accumulator sets
    constexpr int NOUT = NS == 1 ? 1 : (NS == 2 ? 3 : 2);  // partial-row outputs
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = threadIdx.x / WAVE;
    __shared__ double part[2][NW][NA][SPAN];  // by turns, so that one barrier a span is enough
    __shared__ int plive[2][NW];
    int turn = 0;
    __shared__ double nsum[NW];
    const double eta0 = A.cosmo->eta0;
    const int nx = A.cosmo->nx;
    const int nkm = A.nkd - 1;
    double* row = A.partial + (size_t)blockIdx.x * NOUT * A.nu;
    bool first = true;  // the block's first midpoint stores, later ones add
    for (int ik = blockIdx.x; ik < nkm; ik += gridDim.x) {
        const double k = (A.kgrid[ik] + A.kgrid[ik + 1]) / 2.0;
        const double dk = A.kgrid[ik + 1] - A.kgrid[ik];
        // Gridded-linear interpolation in k with Line extrapolation
        int lo = 0, hi = A.nk_src - 2;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (A.k_src[mid] <= k) lo = mid; else hi = mid - 1;
        }
        const int ia = lo;
        const double tt = (k - A.k_src[ia]) / (A.k_src[ia + 1] - A.k_src[ia]);
        const double* Sa = A.S + (size_t)ia * nx + A.i0;
        const double* Sb = A.S + (size_t)(ia + 1) * nx + A.i0;
        const double* Pa = NA == 2 ? A.SP + (size_t)ia * nx + A.i0 : nullptr;
        const double* Pb = NA == 2 ? A.SP + (size_t)(ia + 1) * nx + A.i0 : nullptr;

        // the wavefronts' turns at the longest slots (the earliest x) move on with ik: by
        // three from one midpoint of a block to its next, which lies LOS_GRID further on
        const int own = (wv + (ik >> 8)) & (NW - 1);
        LosLanes<SPW> Q;
        Q.each([&](LosLane& q, auto sl) {
            const int j = (own + NW * decltype(sl)::value) * WAVE + lane;
            q.sp = q.zs = 0.0;
            if (j < A.nxi) {
                const double z = k * (eta0 - A.etaj[j]);
                q.s = ((1.0 - tt) * Sa[j] + tt * Sb[j]) * A.dxj[j];
                if constexpr (NA == 2) q.sp = ((1.0 - tt) * Pa[j] + tt * Pb[j]) * A.dxj[j];
                if constexpr (NS == 3) q.zs = k * (A.eta0d - A.etajd[j]) * q.s;
                const double2 j01 = los_j01(z);
                q.z = q.zl = z;
                q.jp = j01.x;
                q.jc = j01.y;
                q.iz = 1.0 / z;
                q.M = fmax(fabs(q.jp), fabs(q.jc));
            } else {
                q.jp = q.jc = q.iz = q.s = q.M = 0.0;
                q.z = q.zl = LOS_ZS;
            }
            q.n = __popcll(__builtin_amdgcn_ballot_w64(j < A.nxi));
        });
        int nstep = 0;  // wave-uniform
        const double Pw = los_pw(A.cosmo->Pprim_A, A.cosmo->Pprim_n, k, dk);
        const double Pwd = NS == 3 ? Pw * (A.dlnA + A.dns * log(k / 0.05)) : 0.0;
        // ℓ = L0 .. L0+CH-1 of this wavefront into part[]; form 0: the chunk that begins
        // with j₀ and j₁, 1: below LOS_LEAN, 2: above
        auto chunk = [&](int L0, int at, auto form) {
            constexpr int FORM = decltype(form)::value, I0 = FORM == 0 ? 2 : 0;
            double acc[CH], accp[CH];  // accp: NA = 2
#pragma unroll
            for (int i = 0; i < CH; ++i) acc[i] = accp[i] = 0.0;
            int live = 0;
            Q.each([&](LosLane& q, auto) { live += q.n; });
            if (live) {
                int nb = 0;  // leading slots below t = 1.5
                if constexpr (FORM == 2) {
                    bool go = true;
                    Q.each([&](LosLane& q, auto) {
                        go = go && q.n && los_none(los_t(q, L0 + CH - 1) > 1.5);
                        nb += go;
                    });
                    if (nb == 1) los_below<NS, CH, 1>(Q, L0, acc, accp, nstep);
                    if constexpr (SPW >= 2)
                        if (nb == 2) los_below<NS, CH, 2>(Q, L0, acc, accp, nstep);
                    if constexpr (SPW >= 4) {
                        if (nb == 3) los_below<NS, CH, 3>(Q, L0, acc, accp, nstep);
                        if (nb == 4) los_below<NS, CH, 4>(Q, L0, acc, accp, nstep);
                    }
                }
                Q.each([&](LosLane& q, auto sl) {
                    if constexpr (FORM == 0) {
                        acc[0] += q.jp * q.s;
                        acc[1] += q.jc * q.s;
                        if constexpr (NS == 2) { accp[0] += q.jp * q.sp; accp[1] += q.jc * q.sp; }
                        if constexpr (NS == 3) {  // j₀′ = −j₁, j₁′ = j₀ − 2j₁/z
                            accp[0] += q.jp * q.sp - q.jc * q.zs;
                            accp[1] += q.jc * q.sp + (q.jp - 2.0 * q.iz * q.jc) * q.zs;
                        }
                    }
                    if (q.n == 0 || decltype(sl)::value < nb) return;
                    // 1/z outside [0, 1/LOS_ZL]; z < 0 (η > η₀) takes the series
                    if (FORM == 2 || los_none(fabs(q.iz - 0.5 / LOS_ZL) > 0.5 / LOS_ZL))
                        los_slot_turn<NS, CH, I0>(q, L0, acc, accp, nstep);
                    else if (los_any(q.iz != 0.0 && q.z < LOS_ZS))
                        los_slot<NS, CH, I0, true>(q, L0, acc, accp, nstep);
                    else
                        los_slot<NS, CH, I0, false>(q, L0, acc, accp, nstep);
                });
            }
            double Tv = 0.0, Ev = 0.0;
            if (live) {
                Tv = los_reduce(acc);
                if constexpr (NA == 2) Ev = los_reduce(accp);
            }
            if ((lane & 3) == 0) {
                part[turn][own][0][at + (lane >> 2)] = Tv;
                if (NA == 2) part[turn][own][NA - 1][at + (lane >> 2)] = Ev;
            }
            return live;
        };
        // Thread i < SPAN owns ℓ = span + i.  What it adds to is read before the span's
        // recurrences: read after them, 20 spans x 10 midpoints waited for it in turn.
        const int li = threadIdx.x;
        int u = -1;
        double r0 = 0.0, r1 = 0.0, r2 = 0.0;
        auto fetch = [&](int span) {
            const int l = span + li;
            u = li < SPAN && l <= A.lmax ? A.lidx[l] : -1;
            if (u >= 0 && !first) {
                r0 = row[u];
                if (NOUT >= 2) r1 = row[A.nu + u];
                if (NOUT >= 3) r2 = row[2 * A.nu + u];
            }
        };
        // the wavefronts' sums of ℓ = span .. span+SPAN-1 to the block's row; false
        // when every term was past its cut
        auto exchange = [&](int span, int live) {
            if (lane == 0) plive[turn][own] = live;
            __syncthreads();
            int live_block = plive[turn][0];
#pragma unroll
            for (int w = 1; w < NW; ++w) live_block |= plive[turn][w];
            if (u >= 0) {
                const int l = span + li;
                double Tt = part[turn][0][0][li], Et = NA == 2 ? part[turn][0][NA - 1][li] : 0.0;
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    Tt += part[turn][w][0][li];
                    if (NA == 2) Et += part[turn][w][NA - 1][li];
                }
                if (NS == 1) {
                    const double v = A.spin ? Tt * spin_factor(l) : Tt;
                    const double c = v * v * Pw;
                    row[u] = first ? c : r0 + c;
                } else if (NS == 3) {  // T² P and its derivative 2TṪP + T²Ṗ
                    const double c0 = Tt * Tt * Pw, c1 = 2.0 * Tt * Et * Pw + Tt * Tt * Pwd;
                    row[u] = first ? c0 : r0 + c0;
                    row[A.nu + u] = first ? c1 : r1 + c1;
                } else {
                    const double ep = Et * spin_factor(l);
                    const double c0 = Tt * Tt * Pw, c1 = Tt * ep * Pw, c2 = ep * ep * Pw;
                    row[u] = first ? c0 : r0 + c0;
                    row[A.nu + u] = first ? c1 : r1 + c1;
                    row[2 * A.nu + u] = first ? c2 : r2 + c2;
                }
            }
            // the remaining T_ℓ are zero, so the block's first midpoint stores
            // zeros for them (same thread ownership) and later midpoints add
            // nothing
            if (!live_block && first && li < SPAN)
                for (int l2 = span + SPAN + li; l2 <= A.lmax; l2 += SPAN) {
                    const int u2 = A.lidx[l2];
                    if (u2 < 0) continue;
                    for (int o = 0; o < NOUT; ++o) row[o * A.nu + u2] = 0.0;
                }
            turn ^= 1;
            return live_block != 0;
        };
        for (int span = 0; span <= A.lmax; span += SPAN) {
            int live = 0, L0 = span;
            fetch(span);
            if (span == 0) {
                live = chunk(0, 0, std::integral_constant<int, 0>{});
                for (L0 = CH; L0 < LOS_LEAN && L0 <= A.lmax; L0 += CH)
                    live |= chunk(L0, L0, std::integral_constant<int, 1>{});
            }
            for (; L0 < span + SPAN && L0 <= A.lmax; L0 += CH)
                live |= chunk(L0, L0 - span, std::integral_constant<int, 2>{});
            if (!exchange(span, live)) break;
        }
        if (A.steps) {
            const double ns = (double)nstep;
            if (lane == 0) nsum[wv] = ns;
            __syncthreads();
            if (threadIdx.x == 0) {
                double t = 0;
                for (int w = 0; w < NW; ++w) t += nsum[w];
                A.steps[ik] = (long long)t;
            }
            __syncthreads();
        }
        first = false;
    }
}

// ------------------------------------------- Bolt's spline j_ℓ (bessel_mode 1)
// bessel_interpolator (spectra.jl:49-58): j_ℓ on the 5001 nodes 0:Δ:z_max
// (Δ = z_max/5000), interpolated by the natural cubic B-spline of util.jl:11.
// The spline is linear in its coefficients c_m(ℓ), so the sum over the x nodes
// (spectra.jl:70-96) is a matrix product:
//   T_ℓ(k) = Σ_x s_x Σ_p w_p(z_x) c_{i(z_x)+p}(ℓ) = Σ_m W_m(k) c_m(ℓ),
// W_m(k) the sources times basis weights that fall on coefficient m.  W does not
// depend on ℓ: k_spline_weights builds it once per k, and k_spline_cl multiplies
// (FP64 MFMA).  Summed term by term, four gathered coefficients for each (ℓ, k, x),
// a call was 7.6 ms for 120 ℓ x 4999 k x 799 x and 150 ms for 2499 ℓ, bound by the
// gathers; it is 0.47 and 2.9 ms.
// Coefficients are node-major, c[m·nu + u] for requested ℓ column u, with the
// spline's padding rows 0 and BES_N + 1, then zeros up to BES_LD.
#define BES_N 5001
#define BES_LD 5008      // rows of c, columns of W: a multiple of 16
#define BES_ROWS 6144    // midpoints whose W is kept at once (246 MB per source)

// a node's table values, up to the factors that are only known at the recurrence's
// end: j_ℓ = v · scale · 2^(−600·#{q: ℓ > e_q}), zero for ℓ > e[2]
struct BesNode {
    double scale;
    int e[3];
};
// j_ℓ(z_m) for every requested ℓ at node m (one thread per node).  From z = ℓ_max up
// the recurrence runs upward, which is stable for ℓ <= z.  Below, Miller's downward
// recurrence f_{l-1} = (2l+1)/z f_l - f_{l+1} from f_N = 2^-1000, N = ℓ_max + 60 +
// 12·ℓ_max^(1/3), rescaled by 2^-600 whenever |f| is found above 2^600, normalised
// to the exact j₀ or j₁ (whichever is larger).  Each value is stored as it comes: the rescalings that follow it and the normalisation are applied where
// the prefilter reads it.
// One wavefront per SIMD at most (79 wavefronts): what counts is the chain.  Downward
// from N for all nodes and twice (the first pass counted the rescalings) was 10 100
// steps at z = 4800; it is 1200 up or 1390 down for ℓ_max = 1200, in 59 us.  Against 80-bit arithmetic the upward values are off by 5e-14 of the
// largest |j_ℓ|, the downward ones from z = 4800 were by 4e-13.
__global__ void __launch_bounds__(WAVE) k_bessel_nodes(double zmax, const int* ulist, int nu, double* raw, BesNode* node) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= BES_N) return;
    const int lmax = ulist[nu - 1];
    const double z = m * (zmax / (BES_N - 1));
    double* row = raw + (size_t)m * nu;
    BesNode nd = {1.0, {INT_MAX, INT_MAX, INT_MAX}};
    if (z == 0.0) {
        for (int u = 0; u < nu; ++u) row[u] = ulist[u] == 0 ? 1.0 : 0.0;
        node[m] = nd;
        return;
    }
    double j0, j1;
    if (z < 1e-3) {
        const double z2 = z * z;
        j0 = 1.0 - z2 / 6.0 + z2 * z2 / 120.0;
        j1 = z / 3.0 - z * z2 / 30.0 + z * z2 * z2 / 840.0;
    } else {
        double sn, cs;
        sincos(z, &sn, &cs);
        j0 = sn / z;
        j1 = (sn / z - cs) / z;
    }
    const double inv = 1.0 / z;
    if (z >= lmax && z >= 1.0) {
        double fp = j0, fc = j1;  // j_{l-1}, j_l
        int l = 1;
        double a = 3.0;  // 2l + 1
        auto step = [&] {
            const double fn = a * inv * fc - fp;
            fp = fc;
            fc = fn;
            a += 2.0;
            ++l;
        };
        int next = ulist[0];
        for (int u = 0; u < nu; ++u) {
            const int lt = next;
            next = u + 1 < nu ? ulist[u + 1] : lt;
            while (l + 4 <= lt) { step(); step(); step(); step(); }
            while (l < lt) step();
            row[u] = lt == 0 ? j0 : fc;
        }
        node[m] = nd;
        return;
    }
    const double zm = fmax((double)lmax, 1.0);  // z < zm: the same N for the wavefront
    const int N = (int)(zm + 60.0 + 12.0 * cbrt(zm));
    double fp = 0.0, fc = 0x1p-1000;
    int l = N;
    double a = 2 * N + 1;
    auto step = [&] {
        const double fm = a * inv * fc - fp;
        fp = fc;
        fc = fm;
        a -= 2.0;
        --l;
    };
    auto look = [&] {
        if (fabs(fc) > 0x1p600) {
            fc *= 0x1p-600;
            fp *= 0x1p-600;
            nd.e[2] = nd.e[1];
            nd.e[1] = nd.e[0];
            nd.e[0] = l;  // counts for every ℓ above
        }
    };
    // 15 steps grow |f| by at most ((2N+1)/z)^15, less than 2^390 from z = 4e-5 up at
    // ℓ_max = 1200: |f| is looked at after 8 to 15 of them
    const bool eight = __all(a * inv < 0x1p26);
    int next = ulist[nu - 1], since = 0;
    for (int u = nu - 1; u >= -1; --u) {
        const int lt = next;
        next = u > 0 ? ulist[u - 1] : 0;  // the last turn runs on to ℓ = 0
        if (eight) {
            for (; l - lt >= 8; since = 0) {
                step(); step(); step(); step(); step(); step(); step(); step();
                look();
            }
            since += l - lt;
            while (l > lt) step();
            if (since >= 8) {
                look();
                since = 0;
            }
        } else {
            while (l > lt) { step(); look(); }
        }
        if (u >= 0) row[u] = fc;
    }
    nd.scale = fabs(j0) >= fabs(j1) ? j0 / fc : j1 / fp;
    node[m] = nd;
}

// The natural cubic B-spline prefilter, one lane per column: the tridiagonal solve
// (off-diagonals 1, diagonal 4) by the factors cp_q = 1/(4 − cp_{q−1}), cp_0 = 1/4,
// for BES_PC coefficients a block.  Both sweeps forget their start by 0.268 a step:
// BES_WARM steps ahead leave 4e-28 of it, so that the chunks are independent.  (In one
// piece, 10 000 steps with a division and a load each, it was 2 ms on two wavefronts
// for 120 ℓ; it is 32 µs.)
#define BES_PC 32
#define BES_WARM 48
__global__ void __launch_bounds__(WAVE) k_bessel_prefilter(const int* ulist, int nu, const double* raw,
                                                           const BesNode* node, double* c) {
    __shared__ double d[BES_PC + BES_WARM + 1][WAVE];
    __shared__ double cps[BES_PC + 2 * BES_WARM];
    const int lane = threadIdx.x;
    const int u0 = blockIdx.x * WAVE + lane, u = u0 < nu ? u0 : nu - 1;
    const int ell = ulist[u];
    constexpr int n = BES_N, mm = n - 2;
    const int q0 = blockIdx.y * BES_PC, q1 = q0 + BES_PC < mm ? q0 + BES_PC : mm;
    const int qs = q0 > BES_WARM ? q0 - BES_WARM : 0, qe = q1 + BES_WARM < mm ? q1 + BES_WARM : mm;
    auto y = [&](int m) {
        const BesNode nd = node[m];
        double v = raw[(size_t)m * nu + u];
        if (ell > nd.e[0]) v *= 0x1p-600;
        if (ell > nd.e[1]) v *= 0x1p-600;
        return ell > nd.e[2] ? 0.0 : v * nd.scale;
    };
    // cp_qs .. cp_{qe-1}; from cp_40 on they are the same to the last bit
    if (lane == 0) {
        double cp = 0.25;
        for (int q = 0; q < (qs < 40 ? qs : 40); ++q) cp = 1.0 / (4.0 - cp);
        for (int q = qs; q < qe; ++q) {
            cps[q - qs] = cp;
            if (q < 40) cp = 1.0 / (4.0 - cp);
        }
    }
    __syncthreads();
    const double y0 = y(0), yn = y(n - 1);
    double dp = 0.0;
#pragma unroll 16
    for (int q = qs; q < qe; ++q) {
        const double r = 6.0 * y(q + 1) - (q == 0 ? y0 : q == mm - 1 ? yn : 0.0);
        dp = (r - dp) * cps[q - qs];
        d[q >= q0 ? q - q0 : qe - q0][lane] = dp;  // the steps before q0 into a spare row
    }
    double xn = 0.0;  // c_{q+3}
#pragma unroll 16
    for (int q = qe - 1; q >= q0; --q) {
        xn = d[q - q0][lane] - cps[q - qs] * xn;
        if (q < q1 && u0 < nu) c[(size_t)(q + 2) * nu + u] = xn;
    }
    const double c2 = xn, cl = d[qe - 1 - q0][lane];  // c_2 of the first chunk, c_{n−1} of the last
    if (u0 >= nu) return;
    if (q0 == 0) {
        c[(size_t)1 * nu + u] = y0;
        c[u] = 2.0 * y0 - c2;
    }
    if (q1 == mm) {
        c[(size_t)n * nu + u] = yn;
        c[(size_t)(n + 1) * nu + u] = 2.0 * yn - cl;
        for (int m = n + 2; m < BES_LD; ++m) c[(size_t)m * nu + u] = 0.0;
    }
}

struct LosSplArgs {
    const CosmoDev* cosmo;
    const double* S;
    const double* SP;
    const double* k_src;
    int nk_src;
    const double* kgrid;
    int nkd;
    const int* ulist;   // [nu] the distinct requested ℓ, ascending
    int nu;
    const double* c;    // [BES_LD][nu]
    double izd;         // 1/Δ
    const double* etaj;
    const double* dxj;
    int i0, nxi;
    int spin;
    double* partial;    // [grid][nout][nu]
    int ik0, rows;      // this launch's midpoints ik0 .. ik0 + rows - 1
    double* W;          // [NS][tiles·16][BES_LD]
    double* Pw;         // [tiles·16]
    double2* kt;        // [tiles·16] k and the weight of the source column ia + 1
    int* ia;            // [tiles·16]
    int* ext;           // [tiles] columns of W in use, a multiple of 16
};
__device__ inline int spline_node(const LosSplArgs& A, double k, double e) {  // e = η₀ − η
    const int i = (int)floor(k * e * A.izd);
    return i < 0 ? 0 : (i > BES_N - 2 ? BES_N - 2 : i);
}

// what k_spline_weights needs of each midpoint before it can start, one lane each
// (read in a chain by every block it was a quarter of that kernel); midpoints beyond
// `rows` fill up the last tile
__global__ void __launch_bounds__(256) k_spline_rows(LosSplArgs A) {
    __shared__ double emax[4];
    const int tid = threadIdx.x, r = blockIdx.x * 256 + tid, tiles = (A.rows + 15) / 16;
    const double eta0 = A.cosmo->eta0;
    double em = 0.0;
    for (int j = tid; j < A.nxi; j += 256) em = fmax(em, eta0 - A.etaj[j]);
    for (int o = WAVE / 2; o; o >>= 1) em = fmax(em, __shfl_xor(em, o));
    if ((tid & (WAVE - 1)) == 0) emax[tid / WAVE] = em;
    __syncthreads();
    em = fmax(fmax(emax[0], emax[1]), fmax(emax[2], emax[3]));
    const bool in = r < A.rows;
    double k = 0.0, Pw = 0.0, tt = 0.0;
    int lo = 0, hi = A.nk_src - 2;
    if (in) {
        const double ka = A.kgrid[A.ik0 + r], kb = A.kgrid[A.ik0 + r + 1];
        k = (ka + kb) / 2.0;
        while (lo < hi) {
            int m = (lo + hi + 1) >> 1;
            if (A.k_src[m] <= k) lo = m; else hi = m - 1;
        }
        tt = (k - A.k_src[lo]) / (A.k_src[lo + 1] - A.k_src[lo]);
        Pw = los_pw(A.cosmo->Pprim_A, A.cosmo->Pprim_n, k, kb - ka);
    }
    double kt = k;  // columns of the tile: up to the largest k of its 16 midpoints
    for (int o = 8; o; o >>= 1) kt = fmax(kt, __shfl_xor(kt, o));
    if (r >= tiles * 16) return;
    A.kt[r] = make_double2(k, tt);
    A.ia[r] = lo;
    A.Pw[r] = Pw;
    if (r % 16 == 0) A.ext[r / 16] = (spline_node(A, kt, em) + 4 + 15) / 16 * 16;
}

// W of one midpoint per block: W_m = Σ_x s_x w_{m−i(z_x)}(z_x), in the order of the x
// nodes (a gather over the nodes that reach m: no atomics, so the same bits every
// time).  z falls with x where η grows: the x nodes that reach m are those between
// start[m], the first with i <= m, and start[m − 4]; for a table in which η does not
// grow, every x node is looked at.  4999 k x 799 x: 90 us, bound by the latency of
// the LDS reads at four blocks to a CU.
template <int NS>
__global__ void __launch_bounds__(256) k_spline_weights(LosSplArgs A) {
    // [NS][4][nxi] weight p times source, [nxi] first node, start[]
    extern __shared__ double ws[];
    const int nxi = A.nxi;
    int* ix = (int*)(ws + (size_t)NS * 4 * nxi);
    unsigned short* start = (unsigned short*)(ix + nxi);
    const int r = blockIdx.x, tid = threadIdx.x, tiles = gridDim.x / 16;
    const bool in = r < A.rows;  // the others' rows of W are zero
    const double k = A.kt[r].x, tt = A.kt[r].y, eta0 = A.cosmo->eta0;
    const int nx = A.cosmo->nx, ext = A.ext[r / 16];
    const double* Sa = A.S + (size_t)A.ia[r] * nx + A.i0;
    const double* Pa = NS == 2 ? A.SP + (size_t)A.ia[r] * nx + A.i0 : nullptr;
    for (int j = tid; j < nxi; j += 256) {
        const double e = eta0 - A.etaj[j];
        const int i = spline_node(A, k, e);
        ix[j] = i;
        const double t = k * e * A.izd, s = t - i, q = 1.0 - s;
        const double w[4] = {q * q * q / 6.0, 2.0 / 3.0 - s * s + 0.5 * s * s * s, 2.0 / 3.0 - q * q + 0.5 * q * q * q,
                             s * s * s / 6.0};
        const double sx = ((1.0 - tt) * Sa[j] + tt * Sa[nx + j]) * A.dxj[j];
        const double sp = NS == 2 ? ((1.0 - tt) * Pa[j] + tt * Pa[nx + j]) * A.dxj[j] : 0.0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            ws[p * nxi + j] = w[p] * sx;
            if constexpr (NS == 2) ws[(4 + p) * nxi + j] = w[p] * sp;
        }
    }
    __syncthreads();
    bool grows = true;
    for (int j = tid; j + 1 < nxi; j += 256) grows = grows && ix[j + 1] <= ix[j];
    grows = !__syncthreads_or(grows ? 0 : 1);
    if (grows)  // x node j begins nodes ix[j] .. ix[j−1] − 1; none begins those below the last
        for (int j = tid; j <= nxi; j += 256) {
            const int a = j < nxi ? ix[j] : 0, b = j ? ix[j - 1] : ext;
            for (int m = a; m < b; ++m) start[m] = j;
        }
    __syncthreads();
    // a node has 4·nxi/ext terms on average, but at the early end, where η hardly
    // grows, up to twenty times as many: that average in lanes share it, every
    // lanes-th x node each
    int lg = 0;
    while (lg < 6 && (ext << lg) < 4 * nxi) ++lg;
    const int lanes = 1 << lg;
    double* W = A.W + (size_t)r * BES_LD;
    for (int m0 = 0; m0 < ext; m0 += 256 >> lg) {
        const int m = m0 + (tid >> lg);
        double w0 = 0.0, w1 = 0.0;
        if (in && m < ext) {
            const int ja = grows ? start[m] : 0, jb = grows && m >= 4 ? start[m - 4] : nxi;
            for (int j = ja + (tid & (lanes - 1)); j < jb; j += lanes) {
                const int p = m - ix[j];
                if (p < 0 || p > 3) continue;  // only where η does not grow
                w0 += ws[p * nxi + j];
                if constexpr (NS == 2) w1 += ws[(4 + p) * nxi + j];
            }
        }
        for (int o = 1; o < lanes; o *= 2) {
            w0 += __shfl_xor(w0, o);
            if constexpr (NS == 2) w1 += __shfl_xor(w1, o);
        }
        if ((tid & (lanes - 1)) == 0 && m < ext) {
            W[m] = w0;
            if constexpr (NS == 2) W[(size_t)tiles * 16 * BES_LD + m] = w1;
        }
    }
}
static size_t spline_weights_lds(int ns, int nxi) {
    return (sizeof(double) * 4 * ns + sizeof(int)) * (size_t)nxi + sizeof(unsigned short) * BES_LD;
}

// T = W c for 16 midpoints x 64 columns a block, each of the four wavefronts over
// every fourth group of 16 coefficients, then the C_ℓ contributions T_ℓ² P(k) Δk/k
// summed over the block's midpoints into a partial row.  Four MFMAs (16x16x4) take 16
// coefficients, lane l the four of its quarter (l / 16) one after the other, so that W
// comes in two 16-byte loads and c in 128-byte lines, from L2, with no LDS.  The tiles
// of the largest k, with the most coefficients, come first.
// What bounds it is the loads' latency and W's way from memory (67 MB at 4999 k up to
// z = k η₀).  120 ℓ x 4999 k, 3 GFLOP: 187 us with one wavefront per 16 columns over
// all coefficients, 136 split four ways, 100 with a tile's column groups on one XCD,
// 88 with four column groups to a wavefront (which is faster from 59 to 2499 ℓ: a
// call at 499 ℓ takes 0.71 ms against 0.89).
typedef double dbl4 __attribute__((ext_vector_type(4)));
template <int NS>
__global__ void __launch_bounds__(256) k_spline_cl(LosSplArgs A, int tiles, int grid, int first) {
    constexpr int NOUT = NS == 1 ? 1 : 3, NW = 4, NC = 4;  // NC column groups of 16
    __shared__ double red[NW][NS][NC][4][WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    const int col = lane & 15, quarter = lane >> 4;
    // the column groups of one tile follow each other on one XCD (block b runs on XCD
    // b % 8), whose L2 then holds the tile's W
    const int ngroup = (A.nu + 16 * NC - 1) / (16 * NC), idx = blockIdx.x / 8;
    const int bx = idx / ngroup * 8 + blockIdx.x % 8;
    if (bx >= grid) return;
    const int u0 = idx % ngroup * 16 * NC;
    int uc[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) uc[n] = u0 + 16 * n + col < A.nu ? u0 + 16 * n + col : A.nu - 1;
    // wavefront n finishes column group n
    double sum[NOUT] = {};
    for (int tile = tiles - 1 - bx; tile >= 0; tile -= grid) {
        const int steps = A.ext[tile] / 16;
        const double* w = A.W + ((size_t)tile * 16 + col) * BES_LD + 4 * quarter;
        const double* wp = w + (size_t)tiles * 16 * BES_LD;
        const double* c = A.c + (size_t)(4 * quarter) * A.nu;
        dbl4 T[NS][NC];
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int o = 0; o < NS; ++o) T[o][n] = (dbl4){0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
        for (int s = wv; s < steps; s += NW) {
            const dbl4 a = *(const dbl4*)(w + 16 * s);
            dbl4 e = a;
            if constexpr (NS == 2) e = *(const dbl4*)(wp + 16 * s);
            double b[NC][4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int n = 0; n < NC; ++n) b[n][q] = c[(size_t)(16 * s + q) * A.nu + uc[n]];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int n = 0; n < NC; ++n) {
                    T[0][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[n][q], T[0][n], 0, 0, 0);
                    if constexpr (NS == 2)
                        T[1][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(e[q], b[n][q], T[1][n], 0, 0, 0);
                }
        }
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int o = 0; o < NS; ++o)
#pragma unroll
                for (int q = 0; q < 4; ++q) red[wv][o][n][q][lane] = T[o][n][q];
        __syncthreads();
        const int l = A.ulist[u0 + 16 * wv + col < A.nu ? u0 + 16 * wv + col : A.nu - 1];
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // register q of lane l: row 4q + l/16, column l%16
            double t[NS];
#pragma unroll
            for (int o = 0; o < NS; ++o) {
                t[o] = red[0][o][wv][q][lane];
#pragma unroll
                for (int w2 = 1; w2 < NW; ++w2) t[o] += red[w2][o][wv][q][lane];
            }
            const double P = A.Pw[tile * 16 + 4 * q + quarter];
            if constexpr (NS == 1) {
                const double v = A.spin ? t[0] * spin_factor(l) : t[0];
                sum[0] += v * v * P;
            } else {
                const double ep = t[1] * spin_factor(l);
                sum[0] += t[0] * t[0] * P;
                sum[1] += t[0] * ep * P;
                sum[2] += ep * ep * P;
            }
        }
        __syncthreads();
    }
    const int u = u0 + 16 * wv + col;
#pragma unroll
    for (int o = 0; o < NOUT; ++o) {
        sum[o] += __shfl_xor(sum[o], 16);
        sum[o] += __shfl_xor(sum[o], 32);
        double* out = A.partial + ((size_t)bx * NOUT + o) * A.nu + u;
        if (quarter == 0 && u < A.nu) *out = first ? sum[o] : *out + sum[o];
    }
}

// C_ℓ = 4π Σ_blocks partial, in a fixed order: output o, positions
// 64·blockIdx.x .. +63 (one lane each, reading column pmap[i]); wavefront w
// sums the blocks w·nb/4 .. (w+1)·nb/4 - 1 in turn, then the four wavefront
// sums are added in order.  Repeated ℓ read the same column and get the same bits.
__global__ void __launch_bounds__(256) k_los_reduce(const double* partial, int nb, int nout, int nu, const int* pmap,
                                                    int nell, double* cl0, double* cl1, double* cl2) {
    __shared__ double red[4][WAVE];
    const int o = blockIdx.y;
    double* cl = o == 0 ? cl0 : o == 1 ? cl1 : cl2;
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    const int i = blockIdx.x * WAVE + lane;
    const int u = i < nell ? pmap[i] : 0;
    const int b0 = (int)((long long)wv * nb / 4), b1 = (int)((long long)(wv + 1) * nb / 4);
    double s = 0.0;
    if (i < nell) {
#pragma unroll 16
        for (int b = b0; b < b1; ++b) s += partial[((size_t)b * nout + o) * nu + u];
    }
    red[wv][lane] = s;
    __syncthreads();
    if (wv == 0 && i < nell && cl) cl[i] = 4.0 * M_PI * (((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
}

// ------------------------------------------ no-allocation C_ℓ^TT work space
// Device work space of bolt_cltt_dev_noalloc, for callers that cannot allocate
// (code under HIP graph capture, serving loops, harnesses that forbid
// hipMalloc): the LOS partial rows for ℓ <= NOALLOC_MAX_L, η and Δx at the
// integration nodes, the ℓ -> column table and the column map.  One copy per
// GPU (a file-scope device array, 18.5 MB), held until the process ends; host
// code reaches it only through the address hipGetSymbolAddress returns.
#define NOALLOC_MAX_L 3000
#define NOALLOC_MAX_NELL 3001
constexpr size_t NOALLOC_PART = (size_t)LOS_GRID * (NOALLOC_MAX_L + 1);  // doubles
constexpr size_t NOALLOC_NODES = (size_t)LOS_SLOTS * WAVE;               // doubles, for each of η and Δx
constexpr size_t NOALLOC_INTS = (size_t)(NOALLOC_MAX_L + 1) + NOALLOC_MAX_NELL;
constexpr size_t NOALLOC_DOUBLES = NOALLOC_PART + 2 * NOALLOC_NODES + (NOALLOC_INTS + 1) / 2;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

// ------------------------------------------------------------------ host side
#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return set_error(BOLT_E_DEVICE, std::string(#expr " failed: ") + hipGetErrorString(e_));    \
    } while (0)

struct CosmoSlot {
    bool used = false;
    CosmoDev host;        // with device pointers
    double* d_coef = nullptr;
    double* d_q = nullptr;  // qv, df0, base, thbase contiguous
    CosmoDev* d_self = nullptr;
    // bolt_cosmo_upload_jvp: the derivative of every field along one parameter
    // direction (tables, scalars, q arrays), in the same layout
    bool has_tan = false;
    CosmoDev host_dot;
    double* d_dcoef = nullptr;
    double* d_dq = nullptr;
    CosmoDev* d_self_dot = nullptr;
};

struct Server;
static void server_stop(Server* sv);
struct QServer;
static void qserver_stop(QServer* sv);

// A device buffer a context keeps between its calls and only ever grows.
// hipFree waits for the whole device, so a call that allocated and freed its
// launch descriptors would wait for other contexts' kernels too; calls that
// fit the cached capacity allocate nothing and their streams can overlap.
struct GBuf {
    void* p = nullptr;
    size_t cap = 0;
    hipError_t ensure(size_t bytes) {
        if (bytes == 0) bytes = 8;
        if (p && bytes <= cap) return hipSuccess;
        const size_t want = std::max(bytes, 2 * cap);
        release();
        hipError_t e = hipMalloc(&p, want);
        if (e == hipSuccess) cap = want;
        else p = nullptr;
        return e;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
    template <class T> T* as() const { return (T*)p; }
};

struct bolt_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    int n_cu = 0;
    int los_spw = 0;    // LOS slots per wavefront pinned for this context (0: tuned or default)
    int solver_sr = 0;  // scan rows per lane pinned for this context (0: tuned or default)

    hipEvent_t ev0 = nullptr, ev1 = nullptr;  // timing of the no-allocation entry points
    int lds_max = 64 * 1024;
    std::deque<CosmoSlot> cosmos;  // stable slot addresses
    std::mutex mu;
    // launch descriptors and LOS work arrays of calls on `stream` (under mu)
    GBuf c_modes, c_cfgs, c_cosmos, c_counter, c_lidx, c_pmap, c_eta, c_dx, c_contrib, c_btab, c_cosmos_dot, c_etad;
    std::shared_ptr<Server> server;    // request server (bolt_serve_start), if running
    std::shared_ptr<QServer> qserver;  // queue server (bolt_serve_start_queue), if running
    std::mutex server_mu;
};

// LDS of one workgroup of the solver: the FP64 kernel's own layout is the
// smaller one except for short states with many momentum bins
static size_t solve_lds(int n, int nq) { return std::max(ws_bytes(n, nq), wsn_bytes(wsn_layout(n, nq))); }

static int check_cfg(const bolt_hier_cfg* c) {
    if (!c) return set_error(BOLT_E_ARG, "cfg is NULL");
    if (c->ell_g < 3 || c->ell_nu < 2 || c->ell_mnu < 2 || c->nq < 1 || c->nq > 48)
        return set_error(BOLT_E_ARG, "hierarchy sizes need ell_g >= 3, ell_nu >= 2, ell_mnu >= 2, 1 <= nq <= 48");
    if (c->ell_g >= LTAB || c->ell_nu >= LTAB || c->ell_mnu >= LTAB)
        return set_error(BOLT_E_ARG, "hierarchy cut-offs must stay below 512");
    if (!(c->reltol > 0) || !(c->abstol > 0)) return set_error(BOLT_E_ARG, "reltol and abstol must be positive");
    if (c->flags & ~(BOLT_CFG_FP32_SOLVE | BOLT_CFG_REFINE_MASK))
        return set_error(BOLT_E_ARG, "unknown bits in cfg.flags");
    return BOLT_OK;
}

static CfgDev to_cfgdev(const bolt_hier_cfg* c) {
    CfgDev d;
    d.ng = c->ell_g; d.nn = c->ell_nu; d.nm = c->ell_mnu; d.nq = c->nq;
    d.n = 2 * (d.ng + 1) + (d.nn + 1) + (d.nm + 1) * d.nq + 5;
    d.reltol = c->reltol; d.abstol = c->abstol; d.max_steps = c->max_steps;
    d.flags = c->flags;
    return d;
}

// device address of `scratch` on each GPU, set once per device with it current
#define SCRATCH_MAX_DEV 64
static std::mutex g_scratch_mu;
static double* g_scratch[SCRATCH_MAX_DEV] = {};

static int scratch_init(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (device < 0 || device >= SCRATCH_MAX_DEV) return set_error(BOLT_E_ARG, "device index beyond the scratch table");
    if (g_scratch[device]) return BOLT_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return set_error(BOLT_E_DEVICE, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch[device] = (double*)p;
    return BOLT_OK;
}

// callers hold ctx->mu: uploads append to ctx->cosmos under it
static int get_cosmo(bolt_ctx* ctx, int id, CosmoSlot** out) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    if (id < 0 || id >= (int)ctx->cosmos.size() || !ctx->cosmos[id].used)
        return set_error(BOLT_E_STATE, "unknown cosmology id");
    *out = &ctx->cosmos[id];
    return BOLT_OK;
}

// device buffer RAII
struct DBuf {
    void* p = nullptr;
    ~DBuf() { if (p) (void)hipFree(p); }
    hipError_t alloc(size_t bytes) { return hipMalloc(&p, bytes ? bytes : 8); }
    template <class T> T* as() { return (T*)p; }
};

extern "C" {

int bolt_ctx_create(int device, bolt_ctx** out) {
    if (!out) return set_error(BOLT_E_ARG, "out is NULL");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return set_error(BOLT_E_DEVICE, "no HIP device present");
    if (device < 0 || device >= ndev) return set_error(BOLT_E_ARG, "device index out of range");
    HIPCHK(hipSetDevice(device));
    bolt_ctx* c = new bolt_ctx();
    c->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete c; return set_error(BOLT_E_DEVICE, "hipGetDeviceProperties failed"); }
    c->n_cu = prop.multiProcessorCount;
    if (const char* e = std::getenv("BOLT_LOS_SPW")) {
        const int v = std::atoi(e);
        if (v == 1 || v == 2 || v == 4) c->los_spw = v;
    }
    if (const char* e = std::getenv("BOLT_SOLVER_SR")) {
        const int v = std::atoi(e);
        if (v >= SR_RUN_MIN && v <= SR_MAX) c->solver_sr = v;
    }
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return set_error(BOLT_E_DEVICE, "hipStreamCreate failed");
    }
    if (hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        (void)hipStreamDestroy(c->stream);
        delete c;
        return set_error(BOLT_E_DEVICE, "hipEventCreate failed");
    }
    {
        const int r = scratch_init(device);
        if (r) {
            (void)hipEventDestroy(c->ev0); (void)hipEventDestroy(c->ev1);
            (void)hipStreamDestroy(c->stream);
            delete c;
            return r;
        }
    }
    {
        // opt in to the device's full LDS for the one-wavefront-per-mode kernels
        int lds_max = (int)prop.sharedMemPerBlockOptin > 0 ? (int)prop.sharedMemPerBlockOptin
                                                            : (int)prop.sharedMemPerBlock;
        c->lds_max = lds_max - 1024;  // headroom for static __shared__
        for (int sr = SR_RUN_MIN; sr <= SR_MAX; ++sr)
            for (int layout = 0; layout < WSN_LAYOUTS; ++layout)
                (void)hipFuncSetAttribute(solver_kernel(sr, layout), hipFuncAttributeMaxDynamicSharedMemorySize,
                                          c->lds_max);
        for (const void* f : {boltsolve_kernel(false), boltsolve_kernel(true),
                              (const void*)k_rhs, (const void*)k_ics, (const void*)k_rhs_jvp, (const void*)k_ics_jvp,
                              (const void*)k_spline_weights<1>, (const void*)k_spline_weights<2>})
            (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, c->lds_max);
        (void)hipGetLastError();  // an unsupported opt-in must not surface at the next launch check
    }
    {
        std::vector<double> cj(JSER_L * JSER_M);
        fill_jser(cj.data());
        if (hipMemcpyToSymbol(HIP_SYMBOL(c_jser), cj.data(), sizeof(double) * cj.size()) != hipSuccess) {
            (void)hipStreamDestroy(c->stream);
            delete c;
            return set_error(BOLT_E_DEVICE, "hipMemcpyToSymbol(series table) failed");
        }
    }
    *out = c;
    return BOLT_OK;
}

int bolt_ctx_destroy(bolt_ctx* ctx) {
    if (!ctx) return BOLT_OK;
    (void)bolt_serve_stop(ctx);
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    for (auto& s : ctx->cosmos) {
        if (s.d_coef) (void)hipFree(s.d_coef);
        if (s.d_q) (void)hipFree(s.d_q);
        if (s.d_self) (void)hipFree(s.d_self);
        if (s.d_dcoef) (void)hipFree(s.d_dcoef);
        if (s.d_dq) (void)hipFree(s.d_dq);
        if (s.d_self_dot) (void)hipFree(s.d_self_dot);
    }
    for (GBuf* g : {&ctx->c_modes, &ctx->c_cfgs, &ctx->c_cosmos, &ctx->c_counter, &ctx->c_lidx, &ctx->c_pmap,
                    &ctx->c_eta, &ctx->c_dx, &ctx->c_contrib, &ctx->c_btab, &ctx->c_cosmos_dot, &ctx->c_etad})
        g->release();
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return BOLT_OK;
}

// The LDS workspace of one k-mode of the solver, laid out on the host by the
// same accessors the kernel uses: every region as a [begin, end) byte range,
// the dump slot (stores of rows past n), the workspace size the launch
// reserves, and the farthest byte the branch-free reads past n (substitution
// scans, banded LU tails) can touch.
int bolt_ws_layout(int n, int nq, int fp32, int cap, long long* regions, int* nregions, long long* dump_off,
                   long long* total_bytes, long long* read_reach) {
    if (n < 1 || nq < 1 || cap < 0 || !regions || !nregions || !dump_off || !total_bytes || !read_reach)
        return set_error(BOLT_E_ARG, "bad workspace layout query");
    const size_t tot = fp32 ? ws_bytes(n, nq) : solve_lds(n, nq);
    std::vector<double> mem(tot / sizeof(double) + 1);
    const char* b0 = (const char*)mem.data();
    int cnt = 0;
    auto add = [&](const void* p, size_t bytes) {
        if (cnt < cap) {
            regions[2 * cnt] = (const char*)p - b0;
            regions[2 * cnt + 1] = (const char*)p - b0 + (long long)bytes;
        }
        ++cnt;
    };
    const size_t vb = sizeof(double) * (size_t)n, qb = sizeof(double) * (size_t)nq;
    if (!fp32) {  // k_solve's layout: every read past n stays in its vector's padding
        auto regions_of = [&](auto N) {
            using L = decltype(N);
            N.b = mem.data();
            N.n = n;
            N.nq = nq;
            for (int i = 0; i < L::NV; ++i) add(N.vec(i), sizeof(double) * L::ns);
            add(N.tail(), sizeof(double) * 10 * CB);
            for (int st = 0; st < 5; ++st) add(N.xcs(st), sizeof(double) * NXC);
            add(N.red(), sizeof(double) * 15); add(N.red() + 16, sizeof(double) * 8);
            for (int st = 0; st < 6; ++st) add(N.ktab(st), sizeof(double) * L::kt);
            add(N.q(), qb); add(N.df0(), qb); add(N.base(), qb); add(N.qe(), 4 * qb);
            for (int st = 0; st < 5; ++st) add(N.qst_base(st), 4 * qb);
            for (int w = 0; w < NWAVE; ++w) add(N.esc(w), sizeof(double) * L::kt + 4 * qb);
            add(N.kinds(), sizeof(int) * (size_t)n);
            add(N.seg(), sizeof(int) * 2 * MAXSEG); add(N.misc(), sizeof(int) * 4);
            add(N.place(), sizeof(unsigned short) * (size_t)n);
            *dump_off = (const char*)N.dump() - b0;
            *read_reach = (const char*)N.tail() - b0;
        };
        const int layout = wsn_layout(n, nq);
        if (layout == 0) regions_of(WSN0{});
        else if (layout == 1) regions_of(WSN1{});
        else if (layout == 2) regions_of(WSN2{});
        else regions_of(WSN3{});
        *nregions = cnt;
        *total_bytes = (long long)tot;
        return cnt <= cap ? BOLT_OK : set_error(BOLT_E_ARG, "region buffer too small");
    }
    WS W;
    ws_bind(W, mem.data(), n, nq);
    add(W.u(), vb); add(W.f(), vb); add(W.un(), vb); add(W.fn(), vb); add(W.arg(), vb); add(W.w(), vb);
    for (int j = 0; j < 6; ++j) add(W.Z(j), vb);
    add(W.cS(), vb); add(W.cP(), vb); add(W.cPi(), vb);
    for (int j = 0; j < RC_N; ++j) add(W.rcp_(j), vb);
    long long reach = 0;
    long long rows = 0;
    for (int sr = SR_MIN; sr <= SR_MAX; ++sr) {
        const long long span = (long long)WAVE * sr;
        rows = std::max(rows, ((n + span - 1) / span) * span);
    }
    auto reach_of = [&](const double* v) {  // scans read whole passes; the LU tail up to n + CB - 1
        const long long r = (const char*)v - b0 + sizeof(double) * std::max<long long>(rows, n + CB);
        reach = std::max(reach, r);
    };
    auto reach_of_f = [&](const float* v) {
        const long long r = (const char*)v - b0 + sizeof(float) * std::max<long long>(rows, n + CB);
        reach = std::max(reach, r);
    };
    for (int st = 0; st < 5; ++st) {  // the FP32 factors, and the copy of the stage right-hand side
        const BandsT<float> B = W.bandsF(st);
        add(B.l1, sizeof(float) * n); add(B.d, sizeof(float) * n); add(B.u1, sizeof(float) * n);
        add(B.l2c, sizeof(float) * CB); add(B.u2c, sizeof(float) * CB);
        reach_of_f(B.l1); reach_of_f(B.d); reach_of_f(B.u1);
    }
    add(W.rvec(), vb);
    reach_of(W.w()); reach_of(W.cS()); reach_of(W.cP()); reach_of(W.cPi()); reach_of(W.arg());
    add(W.q(), qb); add(W.df0(), qb); add(W.base(), qb);
    add(W.qe(), qb); add(W.eqdf(), qb); add(W.sw(), qb); add(W.rw(), qb);
    for (int st = 0; st < 5; ++st) add(W.qst_base(st), 4 * qb);
    for (int st = 0; st < 5; ++st) add(W.xcs(st), sizeof(double) * NXC);
    for (int st = 0; st < 6; ++st) add(W.ktab(st), sizeof(double) * (K_Q0 + 2 * nq));
    add(W.red(), sizeof(double) * 15);  // stage_border's 4 x 3 functionals, the refinement's 3; block_sum uses 4
    add(W.red() + 16, sizeof(double) * 8);  // the refinement's per-wavefront maxima
    add(W.desc(), sizeof(int) * (size_t)n); add(W.kinds(), sizeof(int) * (size_t)n);
    add(W.seg(), sizeof(int) * 2 * MAXSEG); add(W.misc(), sizeof(int) * 4);
    *nregions = cnt;
    *dump_off = (const char*)W.dump() - b0;
    *total_bytes = (long long)tot;
    *read_reach = reach;
    return cnt <= cap ? BOLT_OK : set_error(BOLT_E_ARG, "region buffer too small");
}

int bolt_ctx_sync(bolt_ctx* ctx) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    HIPCHK(hipSetDevice(ctx->device));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return BOLT_OK;
}

}  // extern "C"

// the device-side description of one cosmology (parameters, scalars, q nodes
// and weights); the table pointers are bound by bind_cosmo_device
// The per-cosmology constants the kernels read, generic over the scalar type:
// R = double gives them, R = bolt::Dual also their derivative along a
// parameter direction (ForwardDiff through Bolt's Hierarchy constructor and
// the q grid of perturbations.jl:127-158).  par: the nine CosmoParams fields;
// scal: H0, η₀, ρ_crit.  out: h, Ω_r, Ω_b, Ω_c, A, n, Y_p, N_ν, Σm_ν, H0, η₀,
// ρ_crit, Ω_ν, Ω_ν of plin (spectra.jl:182-186); qbuf: q_i, dlnf0/dlnq,
// 4πq²f0 w/dxdq, 4πq³f0 w/dxdq.
enum { CS_H = 0, CS_OR, CS_OB, CS_OC, CS_A, CS_NS, CS_YP, CS_NNU, CS_MNU, CS_H0, CS_ETA0, CS_RHOC, CS_ONU, CS_OMNR,
       CS_N };
template <class R>
static void cosmo_scalars(const R* par, const R* scal, const bolt_tables& t, R* out, std::vector<R>& qbuf) {
    using std::exp; using std::log10; using std::pow;
    using bolt::exp; using bolt::log10; using bolt::pow;
    for (int i = 0; i < 9; ++i) out[i] = par[i];
    out[CS_H0] = scal[BOLT_S_H0]; out[CS_ETA0] = scal[BOLT_S_ETA0]; out[CS_RHOC] = scal[BOLT_S_RHO_CRIT];
    const R Or = par[1], h = par[0], Nnu = par[7], rho_crit = scal[BOLT_S_RHO_CRIT];
    out[CS_ONU] = 7.0 * (2.0 / 3.0) * Nnu / 8.0 * std::pow(4.0 / 11.0, 4.0 / 3.0) * Or;
    {   // plin's Ω_ν (spectra.jl:182-186)
        R Tg = pow(15.0 / (M_PI * M_PI) * rho_crit * Or, 0.25);
        R nufac = (90.0 * 1.2020569 / (11.0 * std::pow(M_PI, 4))) * (Or * h * h / Tg) * pow(Nnu / 3.0, 0.75);
        out[CS_OMNR] = par[8] * nufac / (h * h);
    }
    // q nodes and weights (perturbations.jl:127-158 with util.jl:24-27)
    const int nq = t.nq;
    qbuf.assign(4 * (size_t)nq, R(0.0));
    R Tnu = pow(Nnu / 3.0, 0.25) * std::pow(4.0 / 11.0, 1.0 / 3.0) * pow(15.0 / (M_PI * M_PI) * rho_crit * Or, 0.25);
    R lo = log10(Tnu / 30.0), hi = log10(Tnu * 30.0);
    for (int i = 0; i < nq; ++i) {
        R q = pow(10.0, lo + (hi - lo) / 2.0 * (t.xq[i] + 1.0));
        R tu = -1.0 + 2.0 / (hi - lo) * (1.0 + lo - lo);
        R dxdq = (1.0 + tu) / (q * std::log(10.0));
        R f0 = 2.0 / std::pow(2.0 * M_PI, 3) / (exp(q / Tnu) + 1.0);
        qbuf[i] = q;
        qbuf[nq + i] = -q / Tnu / (1.0 + exp(-q / Tnu));
        qbuf[2 * nq + i] = 4.0 * M_PI * q * q * f0 / dxdq * t.wq[i];
        qbuf[3 * nq + i] = 4.0 * M_PI * q * q * q * f0 / dxdq * t.wq[i];
    }
}

static void fill_cosmo(const double* v, const bolt_tables& t, CosmoDev& C) {
    C.h = v[CS_H]; C.Or = v[CS_OR]; C.Ob = v[CS_OB]; C.Oc = v[CS_OC]; C.A = v[CS_A]; C.ns = v[CS_NS];
    C.Yp = v[CS_YP]; C.Nnu = v[CS_NNU]; C.mnu = v[CS_MNU];
    C.H0 = v[CS_H0]; C.eta0 = v[CS_ETA0]; C.rho_crit = v[CS_RHOC]; C.Onu = v[CS_ONU];
    C.x0 = t.x0; C.x1 = t.x1; C.dx = (t.x1 - t.x0) / (t.nx - 1); C.idx = 1.0 / C.dx; C.nx = t.nx; C.nq = t.nq;
    C.Pprim_A = v[CS_A]; C.Pprim_n = v[CS_NS];
    C.Om_nu_nr = v[CS_OMNR];
}

static void par_array(const bolt_cosmo_params& p, double* a) {
    const double v[9] = {p.h, p.Omega_r, p.Omega_b, p.Omega_c, p.A, p.n, p.Y_p, p.N_nu, p.Sum_m_nu};
    for (int i = 0; i < 9; ++i) a[i] = v[i];
}

static void make_cosmo_host(const bolt_cosmo_params& par, const bolt_tables& t, CosmoDev& C,
                            std::vector<double>& qbuf) {
    double pv[9], out[CS_N];
    par_array(par, pv);
    cosmo_scalars<double>(pv, t.scal, t, out, qbuf);
    fill_cosmo(out, t, C);
}

// the tangent of make_cosmo_host along dpar, with dscal the tangent of the
// table scalars: every field of Cd is the derivative of the same field of C
// (x grid and sizes are C's; coef will point at the tangent tables)
static void make_cosmo_tangent(const bolt_cosmo_params& par, const bolt_cosmo_params& dpar, const bolt_tables& t,
                               const double* dscal, CosmoDev& Cd, std::vector<double>& dqbuf) {
    using bolt::Dual;
    double pv[9], dv[9];
    par_array(par, pv);
    par_array(dpar, dv);
    Dual pd[9], sd[BOLT_NSCAL], out[CS_N];
    for (int i = 0; i < 9; ++i) { pd[i] = Dual(pv[i]); pd[i].d[0] = dv[i]; }
    for (int i = 0; i < BOLT_NSCAL; ++i) { sd[i] = Dual(t.scal[i]); sd[i].d[0] = dscal[i]; }
    std::vector<Dual> qd;
    cosmo_scalars<Dual>(pd, sd, t, out, qd);
    double o[CS_N];
    for (int i = 0; i < CS_N; ++i) o[i] = out[i].d[0];
    fill_cosmo(o, t, Cd);
    Cd.x0 = t.x0; Cd.x1 = t.x1; Cd.dx = (t.x1 - t.x0) / (t.nx - 1); Cd.idx = 1.0 / Cd.dx;
    dqbuf.resize(qd.size());
    for (size_t i = 0; i < qd.size(); ++i) dqbuf[i] = qd[i].d[0];
}

// point C at device copies of the tables (coef) and the q arrays (qbuf)
static void bind_cosmo_device(CosmoDev& C, double* d_coef, double* d_q) {
    const int nq = C.nq;
    C.coef = d_coef; C.qv = d_q; C.df0 = d_q + nq; C.base = d_q + 2 * nq; C.thbase = d_q + 3 * nq;
}

extern "C" {

int bolt_cosmo_upload(bolt_ctx* ctx, const bolt_cosmo_params* par, const bolt_tables* t, int* cosmo_id) {
    if (!ctx || !par || !t || !cosmo_id || !t->coef || !t->xq || !t->wq)
        return set_error(BOLT_E_ARG, "bolt_cosmo_upload: NULL argument");
    if (t->nx < 4 || t->nq < 1 || t->nq > 64 || !(t->x1 > t->x0))
        return set_error(BOLT_E_ARG, "bolt_cosmo_upload: bad table geometry");
    std::lock_guard<std::mutex> lk(ctx->mu);
    HIPCHK(hipSetDevice(ctx->device));
    CosmoSlot s;
    s.used = true;
    std::vector<double> qbuf;
    make_cosmo_host(*par, *t, s.host, qbuf);
    size_t ncoef = (size_t)BOLT_NTAB * (t->nx + 2);
    if (hipMalloc(&s.d_coef, ncoef * sizeof(double)) != hipSuccess ||
        hipMalloc(&s.d_q, qbuf.size() * sizeof(double)) != hipSuccess ||
        hipMalloc(&s.d_self, sizeof(CosmoDev)) != hipSuccess) {
        if (s.d_coef) (void)hipFree(s.d_coef);
        if (s.d_q) (void)hipFree(s.d_q);
        return set_error(BOLT_E_NOMEM, "bolt_cosmo_upload: hipMalloc failed");
    }
    HIPCHK(hipMemcpy(s.d_coef, t->coef, ncoef * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(s.d_q, qbuf.data(), qbuf.size() * sizeof(double), hipMemcpyHostToDevice));
    bind_cosmo_device(s.host, s.d_coef, s.d_q);
    HIPCHK(hipMemcpy(s.d_self, &s.host, sizeof(CosmoDev), hipMemcpyHostToDevice));
    int id = -1;
    for (size_t i = 0; i < ctx->cosmos.size(); ++i) if (!ctx->cosmos[i].used) { id = (int)i; break; }
    if (id < 0) { id = (int)ctx->cosmos.size(); ctx->cosmos.push_back(s); } else ctx->cosmos[id] = s;
    *cosmo_id = id;
    return BOLT_OK;
}

int bolt_cosmo_release(bolt_ctx* ctx, int cosmo_id) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* s;
    int r = get_cosmo(ctx, cosmo_id, &s);
    if (r) return r;
    HIPCHK(hipSetDevice(ctx->device));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    (void)hipFree(s->d_coef); (void)hipFree(s->d_q); (void)hipFree(s->d_self);
    if (s->has_tan) { (void)hipFree(s->d_dcoef); (void)hipFree(s->d_dq); (void)hipFree(s->d_self_dot); }
    *s = CosmoSlot();
    return BOLT_OK;
}

int bolt_cosmo_upload_jvp(bolt_ctx* ctx, const bolt_cosmo_params* par, const bolt_cosmo_params* dpar,
                          const bolt_tables* t, const double* dcoef, const double* dscal, int* cosmo_id) {
    if (!dpar || !dcoef || !dscal) return set_error(BOLT_E_ARG, "bolt_cosmo_upload_jvp: NULL argument");
    int id = -1;
    int r = bolt_cosmo_upload(ctx, par, t, &id);
    if (r) return r;
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot& s = ctx->cosmos[id];
    std::vector<double> dq;
    make_cosmo_tangent(*par, *dpar, *t, dscal, s.host_dot, dq);
    const size_t ncoef = (size_t)BOLT_NTAB * (t->nx + 2);
    if (hipMalloc(&s.d_dcoef, ncoef * sizeof(double)) != hipSuccess ||
        hipMalloc(&s.d_dq, dq.size() * sizeof(double)) != hipSuccess ||
        hipMalloc(&s.d_self_dot, sizeof(CosmoDev)) != hipSuccess) {
        if (s.d_dcoef) (void)hipFree(s.d_dcoef);
        if (s.d_dq) (void)hipFree(s.d_dq);
        s.d_dcoef = s.d_dq = nullptr;
        return set_error(BOLT_E_NOMEM, "bolt_cosmo_upload_jvp: hipMalloc failed");
    }
    HIPCHK(hipMemcpy(s.d_dcoef, dcoef, ncoef * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(s.d_dq, dq.data(), dq.size() * sizeof(double), hipMemcpyHostToDevice));
    bind_cosmo_device(s.host_dot, s.d_dcoef, s.d_dq);
    HIPCHK(hipMemcpy(s.d_self_dot, &s.host_dot, sizeof(CosmoDev), hipMemcpyHostToDevice));
    s.has_tan = true;
    *cosmo_id = id;
    return BOLT_OK;
}

}  // extern "C"

// device scratch of one solver launch; a caller that must not allocate per
// call (the serving slots) passes its own
struct SolveBufs {
    ModeDesc* modes = nullptr;
    CfgDev* cfgs = nullptr;
    CosmoDev* cosmos = nullptr;
    int* counter = nullptr;
    int cap_modes = 0, cap_cfgs = 0, cap_cosmos = 0;
};

// shapes chosen by bolt_autotune, shared by every context on a device: scan
// rows per lane by (device, state length), LOS slots per wavefront by
// (device, dense k, ℓ_max, two sources)
static std::mutex g_tune_mu;
static std::map<std::pair<int, int>, int> g_tuned_sr;
static std::map<std::tuple<int, int, int, int>, int> g_tuned_spw;

// (the FP32 solve mode runs with SR_DEFAULT rows per lane)
static void launch_solver(int sr, int layout, bool f32, int grid, size_t lds, hipStream_t stream, const SolveArgs& A) {
    void* args[] = {(void*)&A};
    (void)hipLaunchKernel(f32 ? boltsolve_kernel(false) : solver_kernel(sr, layout), dim3(grid), dim3(NTHR), args, lds,
                          stream);
}
// resident workgroups of that kernel per CU
static hipError_t solver_per_cu(int* per_cu, int sr, int layout, bool f32, size_t lds) {
    const void* f = f32 ? boltsolve_kernel(false) : solver_kernel(sr, layout);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, f, NTHR, lds);
}

// rows per lane of the substitution scans for state length n: the value tuned
// for n on this device, else SR_DEFAULT
static int solver_sr(bolt_ctx* ctx, int n) {
    if (!ctx) return SR_DEFAULT;
    if (ctx->solver_sr > 0) return ctx->solver_sr;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned_sr.find(std::make_pair(ctx->device, n));
    return it != g_tuned_sr.end() ? it->second : SR_DEFAULT;
}

// the integrator over a mode list whose modes may differ in cosmology and
// hierarchy; modes are sorted by k, largest (most steps) first.  persistent:
// a grid of at most one resident workgroup per slot pulls modes from the work
// counter; otherwise one workgroup per mode, so that launches from several
// streams interleave on the CUs.
static int launch_modes(bolt_ctx* ctx, hipStream_t stream, const SolveBufs* pre, bool persistent,
                        const std::vector<CosmoDev>& cosmos, const std::vector<CfgDev>& cfgs,
                        std::vector<ModeDesc>& md, int out_mode, const double* d_xsave, int nsave, double* d_out,
                        double* d_out2, int* d_status, long long* d_counters, int n_stride, double* kernel_ms,
                        int force_sr = 0, const std::vector<CosmoDev>* cosmos_dot = nullptr,
                        double* d_out_dot = nullptr) {
    const int B = (int)md.size();
    const bool tan = cosmos_dot != nullptr;
    std::stable_sort(md.begin(), md.end(), [](const ModeDesc& a, const ModeDesc& b) { return a.k > b.k; });
    size_t lds = 0;
    int nmax = 0, layout = 0;
    for (const CfgDev& c : cfgs) {
        layout = std::max(layout, wsn_layout(c.n, c.nq));
        lds = std::max(lds, tan ? sizeof(double) * (wtan_offset(c.n, c.nq) + wtan_doubles(c.n, c.nq))
                                : solve_lds(c.n, c.nq));
        nmax = std::max(nmax, c.n);
    }
    const int sr = force_sr ? force_sr : solver_sr(ctx, nmax);
    const bool f32 = (cfgs[0].flags & BOLT_CFG_FP32_SOLVE) != 0;
    if ((long long)lds > ctx->lds_max)
        return set_error(BOLT_E_ARG, tan ? "hierarchy too large for one workgroup's LDS with its tangent"
                                         : "hierarchy too large for one workgroup's LDS");
    if (tan && (pre || (int)cosmos_dot->size() != (int)cosmos.size() || !d_out_dot))
        return set_error(BOLT_E_ARG, "tangent solve: one tangent cosmology per cosmology and an output");
    if (tan && (cfgs[0].flags & BOLT_CFG_FP32_SOLVE))
        return set_error(BOLT_E_ARG, "the tangent solve runs in FP64 (no BOLT_CFG_FP32_SOLVE)");
    SolveBufs b;
    if (pre) {
        if (B > pre->cap_modes || (int)cfgs.size() > pre->cap_cfgs || (int)cosmos.size() > pre->cap_cosmos)
            return set_error(BOLT_E_ARG, "launch exceeds the preallocated solver buffers");
        b = *pre;
    } else {  // the context's own stream, under its lock: its cached buffers
        HIPCHK(ctx->c_modes.ensure(sizeof(ModeDesc) * B));
        HIPCHK(ctx->c_cfgs.ensure(sizeof(CfgDev) * cfgs.size()));
        HIPCHK(ctx->c_cosmos.ensure(sizeof(CosmoDev) * cosmos.size()));
        HIPCHK(ctx->c_counter.ensure(sizeof(int)));
        b.modes = ctx->c_modes.as<ModeDesc>(); b.cfgs = ctx->c_cfgs.as<CfgDev>();
        b.cosmos = ctx->c_cosmos.as<CosmoDev>(); b.counter = ctx->c_counter.as<int>();
    }
    HIPCHK(hipMemcpyAsync(b.modes, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(b.cfgs, cfgs.data(), sizeof(CfgDev) * cfgs.size(), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(b.cosmos, cosmos.data(), sizeof(CosmoDev) * cosmos.size(), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemsetAsync(b.counter, 0, sizeof(int), stream));
    SolveArgs A;
    A.cosmos = b.cosmos;
    A.cfgs = b.cfgs;
    A.modes = b.modes;
    A.nmodes = B;
    A.work_counter = b.counter;
    A.out_mode = out_mode;
    A.x_save = d_xsave;
    A.nsave = nsave;
    A.out = d_out;
    A.out2 = d_out2;
    A.status = d_status;
    A.counters = d_counters;
    A.n_state_stride = n_stride;
    A.lds_doubles = (int)(lds / sizeof(double));
    if (tan) {
        HIPCHK(ctx->c_cosmos_dot.ensure(sizeof(CosmoDev) * cosmos_dot->size()));
        HIPCHK(hipMemcpyAsync(ctx->c_cosmos_dot.p, cosmos_dot->data(), sizeof(CosmoDev) * cosmos_dot->size(),
                              hipMemcpyHostToDevice, stream));
        A.cosmos_dot = ctx->c_cosmos_dot.as<CosmoDev>();
        A.out_dot = d_out_dot;
    }
    int grid = B;
    if (persistent) {
        int per_cu = 0;
        if (tan)
            HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, boltsolve_kernel(true), NTHR, lds));
        else
            HIPCHK(solver_per_cu(&per_cu, sr, layout, f32, lds));
        if (per_cu < 1) per_cu = 1;
        grid = std::min(B, per_cu * ctx->n_cu);
    }
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, stream));
    for (const CfgDev& c : cfgs) {
        if ((c.flags & BOLT_CFG_FP32_SOLVE) != (cfgs[0].flags & BOLT_CFG_FP32_SOLVE))
            return set_error(BOLT_E_ARG, "one launch cannot mix FP64 and FP32 solve modes");
    }
    if (tan) {
        void* args[] = {(void*)&A};
        HIPCHK(hipLaunchKernel(boltsolve_kernel(true), dim3(grid), dim3(NTHR), args, lds, stream));
    } else {
        launch_solver(sr, layout, f32, grid, lds, stream, A);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e1, stream));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (kernel_ms) *kernel_ms = ms;
    return BOLT_OK;
}

static int read_positive_k(bolt_ctx* ctx, const double* k, int B, bool on_device, std::vector<double>& kh) {
    kh.resize(B);
    if (on_device) {
        HIPCHK(hipMemcpyAsync(kh.data(), k, sizeof(double) * B, hipMemcpyDeviceToHost, ctx->stream));
        HIPCHK(hipStreamSynchronize(ctx->stream));
    } else {
        std::memcpy(kh.data(), k, sizeof(double) * B);
    }
    for (int i = 0; i < B; ++i)
        if (!(kh[i] > 0.0) || !std::isfinite(kh[i])) return set_error(BOLT_E_ARG, "k must be positive and finite");
    return BOLT_OK;
}

// one cosmology, one hierarchy
static int launch_solve(bolt_ctx* ctx, CosmoSlot* cs, const bolt_hier_cfg* cfg, const double* d_k_or_host, int B,
                        bool k_on_device, int out_mode, const double* d_xsave, int nsave, double* d_out,
                        int* d_status, long long* d_counters, int n_stride, double* kernel_ms,
                        double* d_out2 = nullptr, int force_sr = 0, double* d_out_dot = nullptr) {
    std::vector<double> kh;
    int r = read_positive_k(ctx, d_k_or_host, B, k_on_device, kh);
    if (r) return r;
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = kh[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; md[i].pad = 0; }
    if (d_out_dot) {  // the tangent-linear solve
        const std::vector<CosmoDev> cd = {cs->host_dot};
        return launch_modes(ctx, ctx->stream, nullptr, true, {cs->host}, {to_cfgdev(cfg)}, md, out_mode, d_xsave,
                            nsave, d_out, d_out2, d_status, d_counters, n_stride, kernel_ms, force_sr, &cd, d_out_dot);
    }
    return launch_modes(ctx, ctx->stream, nullptr, true, {cs->host}, {to_cfgdev(cfg)}, md, out_mode, d_xsave, nsave,
                        d_out, d_out2, d_status, d_counters, n_stride, kernel_ms, force_sr);
}

static void fill_stats(bolt_stats* st, const std::vector<long long>& ctr, int B, double ms) {
    if (!st) return;
    std::memset(st, 0, sizeof(*st));
    for (int i = 0; i < B; ++i) {
        st->steps_accepted += ctr[4 * i];
        st->steps_rejected += ctr[4 * i + 1];
        st->rhs_evals += ctr[4 * i + 2];
        st->linear_solves += ctr[4 * i + 3];
    }
    st->kernel_ms = ms;
}

extern "C" {

int bolt_rhs_batch(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B, double x,
                   double* u, double* du, int mutate) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || !u || !du || B <= 0) return set_error(BOLT_E_ARG, "bolt_rhs_batch: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    if (!(x >= cs->host.x0 && x <= cs->host.x1)) return set_error(BOLT_E_ARG, "x outside the table grid");
    HIPCHK(hipSetDevice(ctx->device));
    CfgDev cd = to_cfgdev(cfg);
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    DBuf dm, dc, du_, dd;
    size_t nb = sizeof(double) * (size_t)cd.n * B;
    HIPCHK(dm.alloc(sizeof(ModeDesc) * B));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(du_.alloc(nb));
    HIPCHK(dd.alloc(nb));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(du_.p, u, nb, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_rhs, dim3(B), dim3(WAVE), ws_bytes(cd.n, cd.nq), ctx->stream, cs->d_self, dc.as<CfgDev>(),
                       dm.as<ModeDesc>(), B, x, du_.as<double>(), dd.as<double>(), mutate);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(du, dd.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    if (mutate) HIPCHK(hipMemcpyAsync(u, du_.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return BOLT_OK;
}

int bolt_initial_conditions(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B,
                            double* u0) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || !u0 || B <= 0) return set_error(BOLT_E_ARG, "bolt_initial_conditions: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    HIPCHK(hipSetDevice(ctx->device));
    CfgDev cd = to_cfgdev(cfg);
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    DBuf dm, dc, dout;
    size_t nb = sizeof(double) * (size_t)cd.n * B;
    HIPCHK(dm.alloc(sizeof(ModeDesc) * B));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(dout.alloc(nb));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_ics, dim3(B), dim3(WAVE), ws_bytes(cd.n, cd.nq), ctx->stream, cs->d_self, dc.as<CfgDev>(),
                       dm.as<ModeDesc>(), B, dout.as<double>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(u0, dout.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return BOLT_OK;
}

int bolt_boltsolve_batch(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B,
                         const double* x_save, int nsave, double* u_out, int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || !x_save || !u_out || !status || B <= 0 || nsave <= 0)
        return set_error(BOLT_E_ARG, "bolt_boltsolve_batch: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    for (int i = 0; i < nsave; ++i) {
        if (!(x_save[i] >= cs->host.x0 && x_save[i] <= cs->host.x1))
            return set_error(BOLT_E_ARG, "x_save outside [x0, x1]");
        if (i && !(x_save[i] >= x_save[i - 1])) return set_error(BOLT_E_ARG, "x_save must be sorted ascending");
    }
    HIPCHK(hipSetDevice(ctx->device));
    int n = bolt_state_length(cfg);
    DBuf dk, dx, dout, dst, dctr;
    size_t nb = sizeof(double) * (size_t)B * nsave * n;
    HIPCHK(dx.alloc(sizeof(double) * nsave));
    HIPCHK(dout.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * B));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * B));
    HIPCHK(hipMemcpyAsync(dx.p, x_save, sizeof(double) * nsave, hipMemcpyHostToDevice, ctx->stream));
    double ms = 0;
    if ((r = launch_solve(ctx, cs, cfg, k, B, false, 0, dx.as<double>(), nsave, dout.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), n, &ms)))
        return r;
    std::vector<long long> ctr(4 * (size_t)B);
    HIPCHK(hipMemcpyAsync(u_out, dout.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, B, ms);
    for (int i = 0; i < B; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

int bolt_boltsolve_rsa_batch(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B,
                             double* out, int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || !out || !status || B <= 0) return set_error(BOLT_E_ARG, "bolt_boltsolve_rsa_batch: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    HIPCHK(hipSetDevice(ctx->device));
    int n = bolt_state_length(cfg), nx = cs->host.nx;
    std::vector<double> xs(nx);
    for (int j = 0; j < nx; ++j) xs[j] = (cs->host.x0 * (nx - 1 - j) + cs->host.x1 * j) / (nx - 1);
    DBuf dx, dout, dst, dctr, dm, dc;
    size_t nb = sizeof(double) * (size_t)B * nx * n;
    HIPCHK(dx.alloc(sizeof(double) * nx));
    HIPCHK(dout.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * B));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * B));
    HIPCHK(hipMemcpyAsync(dx.p, xs.data(), sizeof(double) * nx, hipMemcpyHostToDevice, ctx->stream));
    double ms = 0;
    if ((r = launch_solve(ctx, cs, cfg, k, B, false, 0, dx.as<double>(), nx, dout.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), n, &ms)))
        return r;
    CfgDev cd = to_cfgdev(cfg);
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    HIPCHK(dm.alloc(sizeof(ModeDesc) * B));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_rsa_post, dim3((nx + 255) / 256, B), dim3(256), 0, ctx->stream, cs->d_self, dc.as<CfgDev>(),
                       dm.as<ModeDesc>(), B, dout.as<double>());
    HIPCHK(hipGetLastError());
    std::vector<long long> ctr(4 * (size_t)B);
    HIPCHK(hipMemcpyAsync(out, dout.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, B, ms);
    for (int i = 0; i < B; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

int bolt_source_grid_tp_dev(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* d_k, int nk,
                            double* d_ST, double* d_SP, int* d_status, int64_t* d_counters, float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!d_k || (!d_ST && !d_SP) || !d_status || nk <= 0)
        return set_error(BOLT_E_ARG, "bolt_source_grid_tp_dev: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    HIPCHK(hipSetDevice(ctx->device));
    double dms = 0;
    const int mode = (d_ST ? 1 : 0) | (d_SP ? 2 : 0);
    r = launch_solve(ctx, cs, cfg, d_k, nk, true, mode, nullptr, 0, d_ST, d_status, (long long*)d_counters, 0, &dms,
                     d_SP);
    if (ms) *ms = (float)dms;
    return r;
}

int bolt_source_grid_dev(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* d_k, int nk,
                         double* d_S, int* d_status, int64_t* d_counters, float* ms) {
    if (!d_S) return set_error(BOLT_E_ARG, "bolt_source_grid_dev: bad argument");
    return bolt_source_grid_tp_dev(ctx, cosmo_id, cfg, d_k, nk, d_S, nullptr, d_status, d_counters, ms);
}

int bolt_source_grid_tp(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk, double* S_T,
                        double* S_P, int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || (!S_T && !S_P) || !status || nk <= 0) return set_error(BOLT_E_ARG, "bolt_source_grid: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    HIPCHK(hipSetDevice(ctx->device));
    int nx = cs->host.nx;
    DBuf dS, dP, dst, dctr;
    size_t nb = sizeof(double) * (size_t)nk * nx;
    if (S_T) HIPCHK(dS.alloc(nb));
    if (S_P) HIPCHK(dP.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * nk));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * nk));
    double ms = 0;
    const int mode = (S_T ? 1 : 0) | (S_P ? 2 : 0);
    if ((r = launch_solve(ctx, cs, cfg, k, nk, false, mode, nullptr, 0, dS.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), 0, &ms, dP.as<double>())))
        return r;
    std::vector<long long> ctr(4 * (size_t)nk);
    if (S_T) HIPCHK(hipMemcpyAsync(S_T, dS.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    if (S_P) HIPCHK(hipMemcpyAsync(S_P, dP.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, nk, ms);
    for (int i = 0; i < nk; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

int bolt_source_grid(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk, double* S,
                     int* status, bolt_stats* stats) {
    if (!S) return set_error(BOLT_E_ARG, "bolt_source_grid: bad argument");
    return bolt_source_grid_tp(ctx, cosmo_id, cfg, k, nk, S, nullptr, status, stats);
}

int bolt_source_grid_P(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk, double* S_P,
                       int* status, bolt_stats* stats) {
    if (!S_P) return set_error(BOLT_E_ARG, "bolt_source_grid_P: bad argument");
    return bolt_source_grid_tp(ctx, cosmo_id, cfg, k, nk, nullptr, S_P, status, stats);
}

// ------------------------------------------------------- tangent-linear entry points
static int tan_prologue(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, CosmoSlot** cs) {
    int r = get_cosmo(ctx, cosmo_id, cs);
    if (r) return r;
    if (!(*cs)->has_tan) return set_error(BOLT_E_STATE, "the cosmology has no tangent: upload it with bolt_cosmo_upload_jvp");
    if ((r = check_cfg(cfg))) return r;
    if (cfg->flags & BOLT_CFG_FP32_SOLVE) return set_error(BOLT_E_ARG, "the tangent solve runs in FP64");
    if (cfg->nq != (*cs)->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    return BOLT_OK;
}

int bolt_rhs_jvp_batch(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B, double x,
                       const double* u, const double* ud, double* dud) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = tan_prologue(ctx, cosmo_id, cfg, &cs);
    if (r) return r;
    if (!k || !u || !ud || !dud || B <= 0) return set_error(BOLT_E_ARG, "bolt_rhs_jvp_batch: bad argument");
    if (!(x >= cs->host.x0 && x <= cs->host.x1)) return set_error(BOLT_E_ARG, "x outside the table grid");
    HIPCHK(hipSetDevice(ctx->device));
    CfgDev cd = to_cfgdev(cfg);
    const size_t lds = sizeof(double) * (wtan_offset(cd.n, cd.nq) + wtan_doubles(cd.n, cd.nq));
    if ((long long)lds > ctx->lds_max) return set_error(BOLT_E_ARG, "hierarchy too large for one workgroup's LDS with its tangent");
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    DBuf dm, dc, du_, dud_, dd;
    size_t nb = sizeof(double) * (size_t)cd.n * B;
    HIPCHK(dm.alloc(sizeof(ModeDesc) * B));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(du_.alloc(nb));
    HIPCHK(dud_.alloc(nb));
    HIPCHK(dd.alloc(nb));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(du_.p, u, nb, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dud_.p, ud, nb, hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_rhs_jvp, dim3(B), dim3(WAVE), lds, ctx->stream, cs->d_self, cs->d_self_dot,
                       dc.as<CfgDev>(), dm.as<ModeDesc>(), B, x, du_.as<double>(), dud_.as<double>(),
                       dd.as<double>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(dud, dd.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return BOLT_OK;
}

int bolt_initial_conditions_jvp(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B,
                                double* u0, double* ud0) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = tan_prologue(ctx, cosmo_id, cfg, &cs);
    if (r) return r;
    if (!k || !u0 || !ud0 || B <= 0) return set_error(BOLT_E_ARG, "bolt_initial_conditions_jvp: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    CfgDev cd = to_cfgdev(cfg);
    const size_t lds = sizeof(double) * (wtan_offset(cd.n, cd.nq) + wtan_doubles(cd.n, cd.nq));
    if ((long long)lds > ctx->lds_max) return set_error(BOLT_E_ARG, "hierarchy too large for one workgroup's LDS with its tangent");
    std::vector<ModeDesc> md(B);
    for (int i = 0; i < B; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    DBuf dm, dc, d0, d1;
    size_t nb = sizeof(double) * (size_t)cd.n * B;
    HIPCHK(dm.alloc(sizeof(ModeDesc) * B));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(d0.alloc(nb));
    HIPCHK(d1.alloc(nb));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * B, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_ics_jvp, dim3(B), dim3(WAVE), lds, ctx->stream, cs->d_self, cs->d_self_dot, dc.as<CfgDev>(),
                       dm.as<ModeDesc>(), B, d0.as<double>(), d1.as<double>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(u0, d0.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ud0, d1.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return BOLT_OK;
}

int bolt_source_grid_jvp_dev(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* d_k, int nk,
                             double* d_S, double* d_dS, int* d_status, int64_t* d_counters, float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = tan_prologue(ctx, cosmo_id, cfg, &cs);
    if (r) return r;
    if (!d_k || !d_S || !d_dS || !d_status || nk <= 0) return set_error(BOLT_E_ARG, "bolt_source_grid_jvp_dev: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    double dms = 0;
    r = launch_solve(ctx, cs, cfg, d_k, nk, true, 1, nullptr, 0, d_S, d_status, (long long*)d_counters, 0, &dms,
                     nullptr, 0, d_dS);
    if (ms) *ms = (float)dms;
    return r;
}

int bolt_source_grid_jvp(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk, double* S,
                         double* dS, int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = tan_prologue(ctx, cosmo_id, cfg, &cs);
    if (r) return r;
    if (!k || !S || !dS || !status || nk <= 0) return set_error(BOLT_E_ARG, "bolt_source_grid_jvp: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    const int nx = cs->host.nx;
    DBuf d0, d1, dst, dctr;
    const size_t nb = sizeof(double) * (size_t)nk * nx;
    HIPCHK(d0.alloc(nb));
    HIPCHK(d1.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * nk));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * nk));
    double ms = 0;
    if ((r = launch_solve(ctx, cs, cfg, k, nk, false, 1, nullptr, 0, d0.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), 0, &ms, nullptr, 0, d1.as<double>())))
        return r;
    std::vector<long long> ctr(4 * (size_t)nk);
    HIPCHK(hipMemcpyAsync(S, d0.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(dS, d1.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, nk, ms);
    for (int i = 0; i < nk; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

int bolt_boltsolve_jvp_batch(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int B,
                             const double* x_save, int nsave, double* u_out, double* ud_out, int* status,
                             bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = tan_prologue(ctx, cosmo_id, cfg, &cs);
    if (r) return r;
    if (!k || !x_save || !u_out || !ud_out || !status || B <= 0 || nsave <= 0)
        return set_error(BOLT_E_ARG, "bolt_boltsolve_jvp_batch: bad argument");
    for (int i = 0; i < nsave; ++i) {
        if (!(x_save[i] >= cs->host.x0 && x_save[i] <= cs->host.x1))
            return set_error(BOLT_E_ARG, "x_save outside [x0, x1]");
        if (i && !(x_save[i] >= x_save[i - 1])) return set_error(BOLT_E_ARG, "x_save must be sorted ascending");
    }
    HIPCHK(hipSetDevice(ctx->device));
    const int n = bolt_state_length(cfg);
    DBuf dx, d0, d1, dst, dctr;
    const size_t nb = sizeof(double) * (size_t)B * nsave * n;
    HIPCHK(dx.alloc(sizeof(double) * nsave));
    HIPCHK(d0.alloc(nb));
    HIPCHK(d1.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * B));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * B));
    HIPCHK(hipMemcpyAsync(dx.p, x_save, sizeof(double) * nsave, hipMemcpyHostToDevice, ctx->stream));
    double ms = 0;
    if ((r = launch_solve(ctx, cs, cfg, k, B, false, 0, dx.as<double>(), nsave, d0.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), n, &ms, nullptr, 0, d1.as<double>())))
        return r;
    std::vector<long long> ctr(4 * (size_t)B);
    HIPCHK(hipMemcpyAsync(u_out, d0.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ud_out, d1.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, B, ms);
    for (int i = 0; i < B; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

}  // extern "C"

// many cosmologies, each with its own hierarchy and k grid, in one launch
static int source_grid_batch_core(bolt_ctx* ctx, int ncosmo, const int* cosmo_ids, const bolt_hier_cfg* cfgs,
                                  const double* k, int nk, bool k_on_device, double* d_ST, double* d_SP,
                                  int* d_status, long long* d_counters, double* ms) {
    if (ncosmo < 1 || !cosmo_ids || !cfgs || !k || nk < 1 || (!d_ST && !d_SP) || !d_status)
        return set_error(BOLT_E_ARG, "bolt_source_grid_batch: bad argument");
    std::vector<CosmoDev> cos(ncosmo);
    std::vector<CfgDev> cf(ncosmo);
    int nx = -1;
    for (int c = 0; c < ncosmo; ++c) {
        CosmoSlot* cs;
        int r = get_cosmo(ctx, cosmo_ids[c], &cs);
        if (r) return r;
        if ((r = check_cfg(&cfgs[c]))) return r;
        if (cfgs[c].nq != cs->host.nq) return set_error(BOLT_E_ARG, "a cfg's nq differs from its tables' nq");
        if (nx >= 0 && cs->host.nx != nx) return set_error(BOLT_E_ARG, "the cosmologies' x grids differ in length");
        nx = cs->host.nx;
        cos[c] = cs->host;
        cf[c] = to_cfgdev(&cfgs[c]);
    }
    const int B = ncosmo * nk;
    std::vector<double> kh;
    int r = read_positive_k(ctx, k, B, k_on_device, kh);
    if (r) return r;
    std::vector<ModeDesc> md(B);
    for (int c = 0; c < ncosmo; ++c)
        for (int i = 0; i < nk; ++i) {
            ModeDesc& m = md[(size_t)c * nk + i];
            m.k = kh[(size_t)c * nk + i]; m.cosmo = c; m.cfg = c; m.out = c * nk + i; m.pad = 0;
        }
    const int mode = (d_ST ? 1 : 0) | (d_SP ? 2 : 0);
    return launch_modes(ctx, ctx->stream, nullptr, true, cos, cf, md, mode, nullptr, 0, d_ST, d_SP, d_status,
                        d_counters, 0, ms);
}

extern "C" {

int bolt_source_grid_batch(bolt_ctx* ctx, int ncosmo, const int* cosmo_ids, const bolt_hier_cfg* cfgs,
                           const double* k, int nk, double* S_T, double* S_P, int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    if (ncosmo < 1 || nk < 1 || !cosmo_ids || !status || (!S_T && !S_P))
        return set_error(BOLT_E_ARG, "bolt_source_grid_batch: bad argument");
    std::lock_guard<std::mutex> lk(ctx->mu);
    HIPCHK(hipSetDevice(ctx->device));
    CosmoSlot* cs0;
    int r = get_cosmo(ctx, cosmo_ids[0], &cs0);
    if (r) return r;
    const int B = ncosmo * nk, nx = cs0->host.nx;
    DBuf dS, dP, dst, dctr;
    size_t nb = sizeof(double) * (size_t)B * nx;
    if (S_T) HIPCHK(dS.alloc(nb));
    if (S_P) HIPCHK(dP.alloc(nb));
    HIPCHK(dst.alloc(sizeof(int) * B));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * B));
    double ms = 0;
    if ((r = source_grid_batch_core(ctx, ncosmo, cosmo_ids, cfgs, k, nk, false, dS.as<double>(), dP.as<double>(),
                                    dst.as<int>(), dctr.as<long long>(), &ms)))
        return r;
    std::vector<long long> ctr(4 * (size_t)B);
    if (S_T) HIPCHK(hipMemcpyAsync(S_T, dS.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    if (S_P) HIPCHK(hipMemcpyAsync(S_P, dP.p, nb, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * B, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, B, ms);
    for (int i = 0; i < B; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

int bolt_source_grid_batch_dev(bolt_ctx* ctx, int ncosmo, const int* cosmo_ids, const bolt_hier_cfg* cfgs,
                               const double* d_k, int nk, double* d_ST, double* d_SP, int* d_status,
                               int64_t* d_counters, float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    HIPCHK(hipSetDevice(ctx->device));
    double dms = 0;
    int r = source_grid_batch_core(ctx, ncosmo, cosmo_ids, cfgs, d_k, nk, true, d_ST, d_SP, d_status,
                                   (long long*)d_counters, &dms);
    if (ms) *ms = (float)dms;
    return r;
}

int bolt_plin(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk, double x, double* pk,
              int* status, bolt_stats* stats) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || !pk || !status || nk <= 0) return set_error(BOLT_E_ARG, "bolt_plin: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    if (!(x >= cs->host.x0 && x <= cs->host.x1)) return set_error(BOLT_E_ARG, "x outside the table grid");
    HIPCHK(hipSetDevice(ctx->device));
    int n = bolt_state_length(cfg);
    DBuf dx, dout, dst, dctr, dm, dc, dpk;
    HIPCHK(dx.alloc(sizeof(double)));
    HIPCHK(dout.alloc(sizeof(double) * (size_t)nk * n));
    HIPCHK(dst.alloc(sizeof(int) * nk));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * nk));
    HIPCHK(dpk.alloc(sizeof(double) * nk));
    HIPCHK(hipMemcpyAsync(dx.p, &x, sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    double ms = 0;
    if ((r = launch_solve(ctx, cs, cfg, k, nk, false, 0, dx.as<double>(), 1, dout.as<double>(), dst.as<int>(),
                          dctr.as<long long>(), n, &ms)))
        return r;
    CfgDev cd = to_cfgdev(cfg);
    std::vector<ModeDesc> md(nk);
    for (int i = 0; i < nk; ++i) { md[i].k = k[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; }
    HIPCHK(dm.alloc(sizeof(ModeDesc) * nk));
    HIPCHK(dc.alloc(sizeof(CfgDev)));
    HIPCHK(hipMemcpyAsync(dm.p, md.data(), sizeof(ModeDesc) * nk, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dc.p, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_plin_post, dim3((nk + 127) / 128), dim3(128), 0, ctx->stream, cs->d_self, dc.as<CfgDev>(),
                       dm.as<ModeDesc>(), nk, x, dout.as<double>(), dpk.as<double>(), 0);
    HIPCHK(hipGetLastError());
    std::vector<long long> ctr(4 * (size_t)nk);
    HIPCHK(hipMemcpyAsync(pk, dpk.p, sizeof(double) * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipMemcpyAsync(ctr.data(), dctr.p, sizeof(long long) * 4 * nk, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    fill_stats(stats, ctr, nk, ms);
    for (int i = 0; i < nk; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed; see status");
    return BOLT_OK;
}

}  // extern "C"

// C_ℓ core on device buffers; ells given on the host (validated there).
// d_S: temperature source or NULL, d_SP: polarization source or NULL; outputs
// d_tt (needs d_S), d_te (needs both), d_ee (needs d_SP), each may be NULL.
struct LosBufs {
    int* lidx = nullptr;
    int* pmap = nullptr;
    double* etaj = nullptr;
    double* dxj = nullptr;
    double* partial = nullptr;
    size_t cap_lidx = 0, cap_pmap = 0, cap_nxi = 0, cap_partial = 0;
};

template <int NS>
static void launch_los(int spw, int grid, hipStream_t stream, const LosArgs& A) {
    if (spw == 1) hipLaunchKernelGGL((k_los<NS, 1>), dim3(grid), dim3(LOS_SLOTS * WAVE), 0, stream, A);
    else if (spw == 2) hipLaunchKernelGGL((k_los<NS, 2>), dim3(grid), dim3(LOS_SLOTS / 2 * WAVE), 0, stream, A);
    else hipLaunchKernelGGL((k_los<NS, 4>), dim3(grid), dim3(LOS_SLOTS / 4 * WAVE), 0, stream, A);
}

// slots per wavefront of the LOS kernel for this shape: the value pinned on
// the context (BOLT_LOS_SPW at context creation), else the default
static int los_shape(bolt_ctx* ctx, int nkd, int lmax, bool two) {
    if (!ctx) return LOS_SPW_DEFAULT;
    if (ctx->los_spw > 0) return ctx->los_spw;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned_spw.find(std::make_tuple(ctx->device, nkd, lmax, two ? 1 : 0));
    return it != g_tuned_spw.end() ? it->second : LOS_SPW_DEFAULT;
}

// host-side work space of one C_ℓ call that must not allocate: the ℓ -> column
// table and the column map (caller's arrays), and two events for the timing
struct ClHost {
    int* lidx;
    int* pmap;
    int cap_lidx, cap_pmap;
    hipEvent_t ev0, ev1;
};

static int cl_core(bolt_ctx* ctx, hipStream_t stream, const LosBufs* pre, const CosmoDev& host,
                   const CosmoDev* d_cosmo, const double* d_S, const double* d_SP, const double* d_k_src, int nk_src,
                   const double* d_kgrid, int nkd, const int* ells, int nell, int bessel_mode, double* d_tt,
                   double* d_te, double* d_ee, long long* d_steps, float* ms_out, const ClHost* hb = nullptr,
                   int force_spw = 0) {
    if (bessel_mode != 0 && bessel_mode != 1) return set_error(BOLT_E_ARG, "bessel_mode must be 0 or 1");
    if (bessel_mode == 1 && (pre || hb))
        return set_error(BOLT_E_ARG, "bessel_mode 1 (Bolt's spline table) runs on the context's own buffers only");
    if ((d_tt && !d_S) || (d_te && (!d_S || !d_SP)) || (d_ee && !d_SP))
        return set_error(BOLT_E_ARG, "a requested spectrum lacks its source grid");
    if (!d_tt && !d_te && !d_ee) return set_error(BOLT_E_ARG, "no spectrum requested");
    // two sources share the recurrence only when a cross spectrum or both autos are wanted
    const bool two = d_te || (d_tt && d_ee);
    int lmax = 0;
    for (int e = 0; e < nell; ++e) {
        const int l = ells[e];
        if (l < 0 || l > 20000) return set_error(BOLT_E_ARG, "ℓ out of range [0, 20000]");
        lmax = std::max(lmax, l);
    }
    int nx = host.nx;
    int i0 = -1;
    for (int j = 0; j < nx; ++j) {
        double xj = (host.x0 * (nx - 1 - j) + host.x1 * j) / (nx - 1);
        if (xj > -8.0) { i0 = j; break; }
    }
    if (i0 < 0 || i0 >= nx - 1) return set_error(BOLT_E_ARG, "x grid has no node after x = -8");
    int nxi = nx - 1 - i0;
    if (nxi > LOS_SLOTS * WAVE) return set_error(BOLT_E_ARG, "too many integration nodes for the LOS kernel");
    // distinct ℓ, ascending: column u of the partial rows; pmap[i] = column of ells[i]
    std::vector<int> lidx_v, pmap_v;
    if (hb && (lmax + 1 > hb->cap_lidx || nell > hb->cap_pmap))
        return set_error(BOLT_E_ARG, "C_l request exceeds the host work space");
    if (!hb) { lidx_v.resize(lmax + 1); pmap_v.resize(nell); }
    int* lidx = hb ? hb->lidx : lidx_v.data();
    int* pmap = hb ? hb->pmap : pmap_v.data();
    for (int l = 0; l <= lmax; ++l) lidx[l] = -1;
    for (int e = 0; e < nell; ++e) lidx[ells[e]] = 0;
    int nu = 0;
    for (int l = 0; l <= lmax; ++l) if (lidx[l] >= 0) lidx[l] = nu++;
    for (int e = 0; e < nell; ++e) pmap[e] = lidx[ells[e]];
    const int nout = two ? 3 : 1;
    const int nkm = nkd - 1;
    int grid = std::min(LOS_GRID, nkm);
    LosBufs lb;
    const size_t npart = (size_t)grid * nout * nu;
    if (pre) {
        if ((size_t)(lmax + 1) > pre->cap_lidx || (size_t)nell > pre->cap_pmap || (size_t)nxi > pre->cap_nxi ||
            npart > pre->cap_partial)
            return set_error(BOLT_E_ARG, "C_l request exceeds the preallocated LOS buffers");
        lb = *pre;
    } else {  // the context's own stream, under its lock: its cached buffers
        HIPCHK(ctx->c_lidx.ensure(sizeof(int) * (lmax + 1)));
        HIPCHK(ctx->c_pmap.ensure(sizeof(int) * nell));
        HIPCHK(ctx->c_eta.ensure(sizeof(double) * nxi));
        HIPCHK(ctx->c_dx.ensure(sizeof(double) * nxi));
        HIPCHK(ctx->c_contrib.ensure(sizeof(double) * npart));
        lb.lidx = ctx->c_lidx.as<int>(); lb.pmap = ctx->c_pmap.as<int>(); lb.etaj = ctx->c_eta.as<double>();
        lb.dxj = ctx->c_dx.as<double>(); lb.partial = ctx->c_contrib.as<double>();
    }
    HIPCHK(hipMemcpyAsync(lb.lidx, lidx, sizeof(int) * (lmax + 1), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(lb.pmap, pmap, sizeof(int) * nell, hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(k_los_prep, dim3((nxi + 255) / 256), dim3(256), 0, stream, d_cosmo, i0, nxi, lb.etaj, lb.dxj);
    HIPCHK(hipGetLastError());
    LosArgs A;
    A.cosmo = d_cosmo; A.k_src = d_k_src; A.nk_src = nk_src; A.kgrid = d_kgrid; A.nkd = nkd;
    A.S = two ? d_S : (d_tt ? d_S : d_SP);
    A.SP = two ? d_SP : nullptr;
    A.spin = (!two && !d_tt) ? 1 : 0;
    A.lidx = lb.lidx; A.lmax = lmax; A.nu = nu; A.etaj = lb.etaj; A.dxj = lb.dxj;
    A.i0 = i0; A.nxi = nxi; A.partial = lb.partial; A.steps = d_steps;
    hipEvent_t e0, e1;
    if (hb) {
        e0 = hb->ev0; e1 = hb->ev1;
    } else {
        HIPCHK(hipEventCreate(&e0));
        HIPCHK(hipEventCreate(&e1));
    }
    if (bessel_mode == 1) {
        // Bolt's discretisation: the 5001-node spline of j_ℓ on [0, k_max η₀] per requested ℓ
        double kmax = 0;
        HIPCHK(hipMemcpyAsync(&kmax, d_kgrid + nkd - 1, sizeof(double), hipMemcpyDeviceToHost, stream));
        HIPCHK(hipStreamSynchronize(stream));
        const double zmax = kmax * host.eta0;
        std::vector<int> ul(nu);
        for (int l = 0; l <= lmax; ++l) if (lidx[l] >= 0) ul[lidx[l]] = l;
        // one scratch block: W and Pw of up to BES_ROWS midpoints, the two tables, the rest
        const int nsrc = two ? 2 : 1, batch = std::min(nkm, BES_ROWS);
        const int tiles = (batch + 15) / 16;
        const size_t nrow = (size_t)tiles * 16;
        const size_t nW = nsrc * nrow * BES_LD, nc = (size_t)BES_LD * nu, nraw = (size_t)BES_N * nu;
        HIPCHK(ctx->c_btab.ensure(sizeof(double) * (nW + 3 * nrow + nc + nraw) + sizeof(BesNode) * BES_N +
                                  sizeof(int) * (nu + nrow + tiles)));
        LosSplArgs B;
        B.W = ctx->c_btab.as<double>();
        B.kt = (double2*)(B.W + nW);
        B.Pw = (double*)(B.kt + nrow);
        double* c = B.Pw + nrow;
        double* raw = c + nc;
        BesNode* node = (BesNode*)(raw + nraw);
        int* d_ul = (int*)(node + BES_N);
        B.ia = d_ul + nu;
        B.ext = B.ia + nrow;
        HIPCHK(hipMemcpyAsync(d_ul, ul.data(), sizeof(int) * nu, hipMemcpyHostToDevice, stream));
        hipLaunchKernelGGL(k_bessel_nodes, dim3((BES_N + WAVE - 1) / WAVE), dim3(WAVE), 0, stream, zmax, d_ul, nu, raw,
                           node);
        hipLaunchKernelGGL(k_bessel_prefilter, dim3((nu + WAVE - 1) / WAVE, (BES_N - 2 + BES_PC - 1) / BES_PC), dim3(WAVE),
                           0, stream, d_ul, nu, raw, node, c);
        HIPCHK(hipGetLastError());
        B.cosmo = A.cosmo; B.S = A.S; B.SP = A.SP; B.k_src = A.k_src; B.nk_src = A.nk_src; B.kgrid = A.kgrid;
        B.nkd = A.nkd; B.ulist = d_ul; B.nu = nu; B.c = c; B.izd = (BES_N - 1) / zmax; B.etaj = A.etaj;
        B.dxj = A.dxj; B.i0 = A.i0; B.nxi = A.nxi; B.spin = A.spin; B.partial = A.partial;
        grid = std::min(LOS_GRID, tiles);
        HIPCHK(hipEventRecord(e0, stream));
        for (int ik0 = 0; ik0 < nkm; ik0 += batch) {
            B.ik0 = ik0;
            B.rows = std::min(batch, nkm - ik0);
            const int nt = (B.rows + 15) / 16;
            const dim3 gr((nt * 16 + 255) / 256), gw(nt * 16), gc((grid + 7) / 8 * 8 * ((nu + 63) / 64)), b(256);
            const size_t lds = spline_weights_lds(nsrc, nxi);
            hipLaunchKernelGGL(k_spline_rows, gr, b, 0, stream, B);
            if (two) {
                hipLaunchKernelGGL(k_spline_weights<2>, gw, b, lds, stream, B);
                hipLaunchKernelGGL(k_spline_cl<2>, gc, b, 0, stream, B, nt, grid, ik0 == 0);
            } else {
                hipLaunchKernelGGL(k_spline_weights<1>, gw, b, lds, stream, B);
                hipLaunchKernelGGL(k_spline_cl<1>, gc, b, 0, stream, B, nt, grid, ik0 == 0);
            }
        }
    } else {
        HIPCHK(hipEventRecord(e0, stream));
        const int spw = force_spw ? force_spw : los_shape(ctx, nkd, lmax, two);
        if (two) launch_los<2>(spw, grid, stream, A);
        else launch_los<1>(spw, grid, stream, A);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e1, stream));
    hipLaunchKernelGGL(k_los_reduce, dim3((nell + WAVE - 1) / WAVE, nout), dim3(256), 0, stream, lb.partial, grid, nout,
                       nu, lb.pmap, nell, two ? d_tt : (d_tt ? d_tt : d_ee), two ? d_te : (double*)nullptr,
                       two ? d_ee : (double*)nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    if (!hb) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
    if (ms_out) *ms_out = ms;
    HIPCHK(hipStreamSynchronize(stream));
    return BOLT_OK;
}

// C_ℓ^TT and its derivative along the cosmology's tangent direction (cltt,
// spectra.jl:84-96, under Duals): from S and dS/dp, with the Bessel argument's
// derivative k(dη₀/dp − dη/dp) and the primordial spectrum's; exact j_ℓ, on the
// context's own stream and buffers
static int cltt_jvp_core(bolt_ctx* ctx, const CosmoSlot* cs, const double* d_S, const double* d_dS,
                         const double* d_k_src, int nk_src, const double* d_kgrid, int nkd, const int* ells, int nell,
                         double* d_cl, double* d_dcl, float* ms_out) {
    const CosmoDev& host = cs->host;
    hipStream_t stream = ctx->stream;
    int lmax = 0;
    for (int e = 0; e < nell; ++e) {
        if (ells[e] < 0 || ells[e] > 20000) return set_error(BOLT_E_ARG, "ℓ out of range [0, 20000]");
        lmax = std::max(lmax, ells[e]);
    }
    const int nx = host.nx;
    int i0 = -1;
    for (int j = 0; j < nx; ++j) {
        double xj = (host.x0 * (nx - 1 - j) + host.x1 * j) / (nx - 1);
        if (xj > -8.0) { i0 = j; break; }
    }
    if (i0 < 0 || i0 >= nx - 1) return set_error(BOLT_E_ARG, "x grid has no node after x = -8");
    const int nxi = nx - 1 - i0;
    if (nxi > LOS_SLOTS * WAVE) return set_error(BOLT_E_ARG, "too many integration nodes for the LOS kernel");
    std::vector<int> lidx(lmax + 1, -1), pmap(nell);
    for (int e = 0; e < nell; ++e) lidx[ells[e]] = 0;
    int nu = 0;
    for (int l = 0; l <= lmax; ++l) if (lidx[l] >= 0) lidx[l] = nu++;
    for (int e = 0; e < nell; ++e) pmap[e] = lidx[ells[e]];
    const int nout = 2, grid = std::min(LOS_GRID, nkd - 1);
    HIPCHK(ctx->c_lidx.ensure(sizeof(int) * (lmax + 1)));
    HIPCHK(ctx->c_pmap.ensure(sizeof(int) * nell));
    HIPCHK(ctx->c_eta.ensure(sizeof(double) * nxi));
    HIPCHK(ctx->c_dx.ensure(sizeof(double) * nxi));
    HIPCHK(ctx->c_etad.ensure(sizeof(double) * nxi));
    HIPCHK(ctx->c_contrib.ensure(sizeof(double) * (size_t)grid * nout * nu));
    HIPCHK(hipMemcpyAsync(ctx->c_lidx.p, lidx.data(), sizeof(int) * (lmax + 1), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(ctx->c_pmap.p, pmap.data(), sizeof(int) * nell, hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(k_los_prep, dim3((nxi + 255) / 256), dim3(256), 0, stream, cs->d_self, i0, nxi,
                       ctx->c_eta.as<double>(), ctx->c_dx.as<double>());
    hipLaunchKernelGGL(k_los_prep_dot, dim3((nxi + 255) / 256), dim3(256), 0, stream, cs->d_self_dot, i0, nxi,
                       ctx->c_etad.as<double>());
    HIPCHK(hipGetLastError());
    LosArgs A;
    A.cosmo = cs->d_self; A.S = d_S; A.SP = d_dS; A.k_src = d_k_src; A.nk_src = nk_src; A.kgrid = d_kgrid;
    A.nkd = nkd; A.lidx = ctx->c_lidx.as<int>(); A.lmax = lmax; A.nu = nu; A.etaj = ctx->c_eta.as<double>();
    A.dxj = ctx->c_dx.as<double>(); A.i0 = i0; A.nxi = nxi; A.spin = 0; A.partial = ctx->c_contrib.as<double>();
    A.steps = nullptr;
    A.etajd = ctx->c_etad.as<double>();
    A.eta0d = cs->host_dot.eta0;
    A.dlnA = cs->host_dot.Pprim_A / host.Pprim_A;
    A.dns = cs->host_dot.Pprim_n;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, stream));
    launch_los<3>(los_shape(ctx, nkd, lmax, true), grid, stream, A);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e1, stream));
    hipLaunchKernelGGL(k_los_reduce, dim3((nell + WAVE - 1) / WAVE, nout), dim3(256), 0, stream,
                       ctx->c_contrib.as<double>(), grid, nout, nu, ctx->c_pmap.as<int>(), nell, d_cl, d_dcl,
                       (double*)nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (ms_out) *ms_out = ms;
    HIPCHK(hipStreamSynchronize(stream));
    return BOLT_OK;
}

extern "C" {

int bolt_cltt(bolt_ctx* ctx, int cosmo_id, const double* S, const double* k_src, int nk_src, const double* kgrid,
              int nkd, const int* ells, int nell, int bessel_mode, double* cl) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if (!S || !k_src || !kgrid || !ells || !cl || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cltt: bad argument");
    for (int i = 1; i < nk_src; ++i) if (!(k_src[i] > k_src[i - 1])) return set_error(BOLT_E_ARG, "k_src must increase");
    for (int i = 1; i < nkd; ++i) if (!(kgrid[i] > kgrid[i - 1])) return set_error(BOLT_E_ARG, "kgrid must increase");
    HIPCHK(hipSetDevice(ctx->device));
    int nx = cs->host.nx;
    DBuf dS, dks, dkg, dcl;
    HIPCHK(dS.alloc(sizeof(double) * (size_t)nk_src * nx));
    HIPCHK(dks.alloc(sizeof(double) * nk_src));
    HIPCHK(dkg.alloc(sizeof(double) * nkd));
    HIPCHK(dcl.alloc(sizeof(double) * nell));
    HIPCHK(hipMemcpyAsync(dS.p, S, sizeof(double) * (size_t)nk_src * nx, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dks.p, k_src, sizeof(double) * nk_src, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dkg.p, kgrid, sizeof(double) * nkd, hipMemcpyHostToDevice, ctx->stream));
    std::vector<int> ev(ells, ells + nell);
    if ((r = cl_core(ctx, ctx->stream, nullptr, cs->host, cs->d_self, dS.as<double>(), nullptr, dks.as<double>(),
                     nk_src, dkg.as<double>(), nkd, ev.data(), (int)ev.size(),
                     bessel_mode, dcl.as<double>(), nullptr, nullptr, nullptr, nullptr)))
        return r;
    HIPCHK(hipMemcpy(cl, dcl.p, sizeof(double) * nell, hipMemcpyDeviceToHost));
    return BOLT_OK;
}

int bolt_cltt_jvp_dev(bolt_ctx* ctx, int cosmo_id, const double* d_S, const double* d_dS, const double* d_k_src,
                      int nk_src, const double* d_kgrid, int nkd, const int* ells, int nell, double* d_cl,
                      double* d_dcl, float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if (!cs->has_tan) return set_error(BOLT_E_STATE, "the cosmology has no tangent: upload it with bolt_cosmo_upload_jvp");
    if (!d_S || !d_dS || !d_k_src || !d_kgrid || !ells || !d_cl || !d_dcl || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cltt_jvp_dev: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    return cltt_jvp_core(ctx, cs, d_S, d_dS, d_k_src, nk_src, d_kgrid, nkd, ells, nell, d_cl, d_dcl, ms);
}

int bolt_cltt_jvp(bolt_ctx* ctx, int cosmo_id, const double* S, const double* dS, const double* k_src, int nk_src,
                  const double* kgrid, int nkd, const int* ells, int nell, double* cl, double* dcl) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if (!cs->has_tan) return set_error(BOLT_E_STATE, "the cosmology has no tangent: upload it with bolt_cosmo_upload_jvp");
    if (!S || !dS || !k_src || !kgrid || !ells || !cl || !dcl || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cltt_jvp: bad argument");
    for (int i = 1; i < nk_src; ++i) if (!(k_src[i] > k_src[i - 1])) return set_error(BOLT_E_ARG, "k_src must increase");
    for (int i = 1; i < nkd; ++i) if (!(kgrid[i] > kgrid[i - 1])) return set_error(BOLT_E_ARG, "kgrid must increase");
    HIPCHK(hipSetDevice(ctx->device));
    const int nx = cs->host.nx;
    const size_t ns = sizeof(double) * (size_t)nk_src * nx;
    DBuf d0, d1, dks, dkg, dcl0, dcl1;
    HIPCHK(d0.alloc(ns));
    HIPCHK(d1.alloc(ns));
    HIPCHK(dks.alloc(sizeof(double) * nk_src));
    HIPCHK(dkg.alloc(sizeof(double) * nkd));
    HIPCHK(dcl0.alloc(sizeof(double) * nell));
    HIPCHK(dcl1.alloc(sizeof(double) * nell));
    HIPCHK(hipMemcpyAsync(d0.p, S, ns, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(d1.p, dS, ns, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dks.p, k_src, sizeof(double) * nk_src, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dkg.p, kgrid, sizeof(double) * nkd, hipMemcpyHostToDevice, ctx->stream));
    if ((r = cltt_jvp_core(ctx, cs, d0.as<double>(), d1.as<double>(), dks.as<double>(), nk_src, dkg.as<double>(), nkd,
                           ells, nell, dcl0.as<double>(), dcl1.as<double>(), nullptr)))
        return r;
    HIPCHK(hipMemcpy(cl, dcl0.p, sizeof(double) * nell, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(dcl, dcl1.p, sizeof(double) * nell, hipMemcpyDeviceToHost));
    return BOLT_OK;
}

// device-resident variant used by the serving loop and the benchmark: ℓ list on
// the host, everything else on the device; returns the k_los time in *ms.
int bolt_cltt_dev(bolt_ctx* ctx, int cosmo_id, const double* d_S, const double* d_k_src, int nk_src,
                       const double* d_kgrid, int nkd, const int* ells, int nell, double* d_cl, int64_t* d_steps,
                       float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if (!d_S || !d_k_src || !d_kgrid || !ells || !d_cl || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cltt_dev: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    std::vector<int> ev(ells, ells + nell);
    return cl_core(ctx, ctx->stream, nullptr, cs->host, cs->d_self, d_S, nullptr, d_k_src, nk_src, d_kgrid, nkd,
                   ev.data(), (int)ev.size(), 0, d_cl, nullptr, nullptr,
                   (long long*)d_steps, ms);
}

// The project's autotuner: times every solver shape (rows per lane of the
// substitution scans, SR = 5..8) on the caller's k grid and hierarchy, and
// every LOS shape (x slots per wavefront, 1/2/4) on the resulting source grid,
// dense k grid and ℓ range; keeps the fastest of each on the context for that
// state length and that (dense k, ℓ_max).  Each shape gives bitwise
// reproducible results; different shapes add in different orders.
int bolt_autotune(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* k, int nk,
                  const double* kgrid, int nkd, int lmax, bolt_tune_report* rep) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!k || nk < 2 || !rep || (kgrid && (nkd < 2 || lmax < 2 || lmax > 20000)))
        return set_error(BOLT_E_ARG, "bolt_autotune: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    for (int i = 1; i < nk; ++i) if (!(k[i] > k[i - 1])) return set_error(BOLT_E_ARG, "k must increase");
    HIPCHK(hipSetDevice(ctx->device));
    std::memset(rep, 0, sizeof(*rep));
    const int nx = cs->host.nx;
    DBuf dk, dS, dst, dctr;
    HIPCHK(dk.alloc(sizeof(double) * nk));
    HIPCHK(dS.alloc(sizeof(double) * (size_t)nk * nx));
    HIPCHK(dst.alloc(sizeof(int) * nk));
    HIPCHK(dctr.alloc(sizeof(long long) * 4 * nk));
    HIPCHK(hipMemcpyAsync(dk.p, k, sizeof(double) * nk, hipMemcpyHostToDevice, ctx->stream));
    float best = 0;
    for (int sr = SR_RUN_MIN; sr <= SR_MAX; ++sr) {
        double ms = 0;
        for (int rep_i = 0; rep_i < 2; ++rep_i)  // the first launch of a shape loads its code
            if ((r = launch_solve(ctx, cs, cfg, dk.as<double>(), nk, true, 1, nullptr, 0, dS.as<double>(),
                                  dst.as<int>(), dctr.as<long long>(), 0, &ms, nullptr, sr)))
                return r;
        rep->solver_ms[sr - SR_MIN] = (float)ms;
        if (sr == SR_RUN_MIN || ms < best) { best = (float)ms; rep->solver_sr = sr; }
    }
    {
        std::lock_guard<std::mutex> lt(g_tune_mu);
        g_tuned_sr[std::make_pair(ctx->device, bolt_state_length(cfg))] = rep->solver_sr;
    }
    if (kgrid) {
        DBuf dkg, dcl;
        HIPCHK(dkg.alloc(sizeof(double) * nkd));
        HIPCHK(dcl.alloc(sizeof(double) * (lmax - 1)));
        HIPCHK(hipMemcpyAsync(dkg.p, kgrid, sizeof(double) * nkd, hipMemcpyHostToDevice, ctx->stream));
        std::vector<int> ells(lmax - 1);
        for (int l = 2; l <= lmax; ++l) ells[l - 2] = l;
        const int spws[3] = {1, 2, 4};
        for (int c = 0; c < 3; ++c) {
            float ms = 0;
            for (int rep_i = 0; rep_i < 2; ++rep_i)
                if ((r = cl_core(ctx, ctx->stream, nullptr, cs->host, cs->d_self, dS.as<double>(), nullptr,
                                 dk.as<double>(), nk, dkg.as<double>(), nkd, ells.data(), (int)ells.size(), 0,
                                 dcl.as<double>(), nullptr, nullptr, nullptr, &ms, nullptr, spws[c])))
                    return r;
            rep->los_ms[c] = ms;
            if (c == 0 || ms < best) { best = ms; rep->los_spw = spws[c]; }
        }
        std::lock_guard<std::mutex> lt(g_tune_mu);
        g_tuned_spw[std::make_tuple(ctx->device, nkd, lmax, 0)] = rep->los_spw;
    }
    return BOLT_OK;
}

}  // extern "C"

// the solver's work counter, zeroed by a kernel (a graph replays it; memset
// nodes are avoided in captured graphs)
__global__ void k_zero_int(int* p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

// A captured spectrum: source_grid + cltt for one cosmology, hierarchy and pair
// of k grids, with its descriptors and LOS work space owned by the graph
struct bolt_graph {
    bolt_ctx* ctx = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<void*> allocs;
    ~bolt_graph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (void* p : allocs) (void)hipFree(p);
    }
    template <class T>
    hipError_t alloc(T** p, size_t count) {
        hipError_t e = hipMalloc((void**)p, sizeof(T) * (count ? count : 1));
        if (e == hipSuccess) allocs.push_back((void*)*p);
        return e;
    }
};

extern "C" {

int bolt_graph_spectrum_create(bolt_ctx* ctx, int cosmo_id, const bolt_hier_cfg* cfg, const double* d_k, int nk,
                               const double* d_kgrid, int nkd, const int* ells, int nell, double* d_S,
                               int* d_status, int64_t* d_counters, double* d_cl, bolt_graph** out) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((r = check_cfg(cfg))) return r;
    if (!d_k || nk < 2 || !d_kgrid || nkd < 2 || !ells || nell < 1 || !d_S || !d_status || !d_cl || !out)
        return set_error(BOLT_E_ARG, "bolt_graph_spectrum_create: bad argument");
    if (cfg->nq != cs->host.nq) return set_error(BOLT_E_ARG, "cfg.nq differs from the tables' nq");
    HIPCHK(hipSetDevice(ctx->device));
    const CosmoDev& host = cs->host;
    // the solver launch, as launch_modes sets it up
    std::vector<double> kh;
    if ((r = read_positive_k(ctx, d_k, nk, true, kh))) return r;
    std::vector<ModeDesc> md(nk);
    for (int i = 0; i < nk; ++i) { md[i].k = kh[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; md[i].pad = 0; }
    std::stable_sort(md.begin(), md.end(), [](const ModeDesc& a, const ModeDesc& b) { return a.k > b.k; });
    const CfgDev cd = to_cfgdev(cfg);
    const size_t lds = solve_lds(cd.n, cd.nq);
    if ((long long)lds > ctx->lds_max) return set_error(BOLT_E_ARG, "hierarchy too large for one workgroup's LDS");
    // the LOS launch, as cl_core sets it up
    int lmax = 0;
    for (int e = 0; e < nell; ++e) {
        if (ells[e] < 0 || ells[e] > 20000) return set_error(BOLT_E_ARG, "ℓ out of range [0, 20000]");
        lmax = std::max(lmax, ells[e]);
    }
    const int nx = host.nx;
    int i0 = -1;
    for (int j = 0; j < nx; ++j)
        if ((host.x0 * (nx - 1 - j) + host.x1 * j) / (nx - 1) > -8.0) { i0 = j; break; }
    if (i0 < 0 || i0 >= nx - 1) return set_error(BOLT_E_ARG, "x grid has no node after x = -8");
    const int nxi = nx - 1 - i0;
    if (nxi > LOS_SLOTS * WAVE) return set_error(BOLT_E_ARG, "too many integration nodes for the LOS kernel");
    std::vector<int> lidx(lmax + 1, -1), pmap(nell);
    for (int e = 0; e < nell; ++e) lidx[ells[e]] = 0;
    int nu = 0;
    for (int l = 0; l <= lmax; ++l) if (lidx[l] >= 0) lidx[l] = nu++;
    for (int e = 0; e < nell; ++e) pmap[e] = lidx[ells[e]];
    const int nkm = nkd - 1, lgrid = std::min(LOS_GRID, nkm);

    std::unique_ptr<bolt_graph> g(new bolt_graph);
    g->ctx = ctx;
    ModeDesc* d_md; CfgDev* d_cfg; int* d_ctr; int* d_lidx; int* d_pmap; double *d_eta, *d_dx, *d_part;
    HIPCHK(g->alloc(&d_md, nk));
    HIPCHK(g->alloc(&d_cfg, 1));
    HIPCHK(g->alloc(&d_ctr, 1));
    HIPCHK(g->alloc(&d_lidx, lmax + 1));
    HIPCHK(g->alloc(&d_pmap, nell));
    HIPCHK(g->alloc(&d_eta, nxi));
    HIPCHK(g->alloc(&d_dx, nxi));
    HIPCHK(g->alloc(&d_part, (size_t)lgrid * nu));
    HIPCHK(hipMemcpyAsync(d_md, md.data(), sizeof(ModeDesc) * nk, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(d_cfg, &cd, sizeof(CfgDev), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(d_lidx, lidx.data(), sizeof(int) * (lmax + 1), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(d_pmap, pmap.data(), sizeof(int) * nell, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    SolveArgs A;
    A.cosmos = cs->d_self; A.cfgs = d_cfg; A.modes = d_md; A.nmodes = nk; A.work_counter = d_ctr;
    A.out_mode = 1; A.x_save = nullptr; A.nsave = 0; A.out = d_S; A.out2 = nullptr; A.status = d_status;
    A.counters = (long long*)d_counters; A.n_state_stride = 0; A.lds_doubles = (int)(lds / sizeof(double));
    int per_cu = 0;
    const int sr = solver_sr(ctx, cd.n);
    HIPCHK(solver_per_cu(&per_cu, sr, wsn_layout(cd.n, cd.nq), (cd.flags & BOLT_CFG_FP32_SOLVE) != 0, lds));
    const int sgrid = std::min(nk, std::max(per_cu, 1) * ctx->n_cu);
    LosArgs L;
    L.cosmo = cs->d_self; L.S = d_S; L.SP = nullptr; L.k_src = d_k; L.nk_src = nk; L.kgrid = d_kgrid; L.nkd = nkd;
    L.lidx = d_lidx; L.lmax = lmax; L.nu = nu; L.etaj = d_eta; L.dxj = d_dx; L.i0 = i0; L.nxi = nxi; L.spin = 0;
    L.partial = d_part; L.steps = nullptr;
    const int spw = los_shape(ctx, nkd, lmax, false);
    // capture: counter reset, solver, LOS node table, LOS, reduction
    HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, ctx->stream, d_ctr);
    launch_solver(sr, wsn_layout(cd.n, cd.nq), (cd.flags & BOLT_CFG_FP32_SOLVE) != 0, sgrid, lds, ctx->stream, A);
    hipLaunchKernelGGL(k_los_prep, dim3((nxi + 255) / 256), dim3(256), 0, ctx->stream, cs->d_self, i0, nxi, d_eta,
                       d_dx);
    launch_los<1>(spw, lgrid, ctx->stream, L);
    hipLaunchKernelGGL(k_los_reduce, dim3((nell + WAVE - 1) / WAVE, 1), dim3(256), 0, ctx->stream, d_part, lgrid, 1,
                       nu, d_pmap, nell, d_cl, (double*)nullptr, (double*)nullptr);
    const hipError_t le = hipGetLastError();
    const hipError_t ce = hipStreamEndCapture(ctx->stream, &g->graph);
    if (le != hipSuccess || ce != hipSuccess)
        return set_error(BOLT_E_DEVICE, std::string("capturing the spectrum graph failed: ") +
                                            hipGetErrorString(le != hipSuccess ? le : ce));
    HIPCHK(hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0));
    *out = g.release();
    return BOLT_OK;
}

int bolt_graph_launch(bolt_graph* g) {
    if (!g || !g->ctx) return set_error(BOLT_E_ARG, "bolt_graph_launch: NULL graph");
    std::lock_guard<std::mutex> lk(g->ctx->mu);
    HIPCHK(hipSetDevice(g->ctx->device));
    HIPCHK(hipGraphLaunch(g->exec, g->ctx->stream));
    HIPCHK(hipStreamSynchronize(g->ctx->stream));
    return BOLT_OK;
}

int bolt_graph_destroy(bolt_graph* g) {
    if (!g) return BOLT_OK;
    if (g->ctx) {
        std::lock_guard<std::mutex> lk(g->ctx->mu);
        (void)hipSetDevice(g->ctx->device);
        (void)hipStreamSynchronize(g->ctx->stream);
    }
    delete g;
    return BOLT_OK;
}

// bolt_cltt_dev without any allocation: the device work space is this GPU's
// `scratch` array and the host work space sits on the stack; calls that
// overlap on one GPU share the array and race
int bolt_cltt_dev_noalloc(bolt_ctx* ctx, int cosmo_id, const double* d_S, const double* d_k_src, int nk_src,
                          const double* d_kgrid, int nkd, const int* ells, int nell, double* d_cl, int64_t* d_steps,
                          float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if (!d_S || !d_k_src || !d_kgrid || !ells || !d_cl || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cltt_dev_noalloc: bad argument");
    if (nell > NOALLOC_MAX_NELL)
        return set_error(BOLT_E_ARG, "bolt_cltt_dev_noalloc: more than 3001 multipoles requested");
    for (int e = 0; e < nell; ++e)
        if (ells[e] < 0 || ells[e] > NOALLOC_MAX_L)
            return set_error(BOLT_E_ARG, "bolt_cltt_dev_noalloc: ℓ outside [0, 3000]");
    double* base = ctx->device >= 0 && ctx->device < SCRATCH_MAX_DEV ? g_scratch[ctx->device] : nullptr;
    if (!base) return set_error(BOLT_E_STATE, "bolt_cltt_dev_noalloc: no work space on this device");
    LosBufs lb;
    lb.partial = base;
    lb.etaj = base + NOALLOC_PART;
    lb.dxj = lb.etaj + NOALLOC_NODES;
    lb.lidx = (int*)(lb.dxj + NOALLOC_NODES);
    lb.pmap = lb.lidx + NOALLOC_MAX_L + 1;
    lb.cap_partial = NOALLOC_PART; lb.cap_nxi = NOALLOC_NODES;
    lb.cap_lidx = NOALLOC_MAX_L + 1; lb.cap_pmap = NOALLOC_MAX_NELL;
    int h_lidx[NOALLOC_MAX_L + 1], h_pmap[NOALLOC_MAX_NELL];
    const ClHost hb{h_lidx, h_pmap, NOALLOC_MAX_L + 1, NOALLOC_MAX_NELL, ctx->ev0, ctx->ev1};
    HIPCHK(hipSetDevice(ctx->device));
    return cl_core(ctx, ctx->stream, &lb, cs->host, cs->d_self, d_S, nullptr, d_k_src, nk_src, d_kgrid, nkd, ells,
                   nell, 0, d_cl, nullptr, nullptr, (long long*)d_steps, ms, &hb);
}

int bolt_cl(bolt_ctx* ctx, int cosmo_id, const double* S_T, const double* S_P, const double* k_src, int nk_src,
            const double* kgrid, int nkd, const int* ells, int nell, int bessel_mode, double* cltt, double* clte,
            double* clee) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((!S_T && !S_P) || !k_src || !kgrid || !ells || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cl: bad argument");
    for (int i = 1; i < nk_src; ++i) if (!(k_src[i] > k_src[i - 1])) return set_error(BOLT_E_ARG, "k_src must increase");
    for (int i = 1; i < nkd; ++i) if (!(kgrid[i] > kgrid[i - 1])) return set_error(BOLT_E_ARG, "kgrid must increase");
    HIPCHK(hipSetDevice(ctx->device));
    int nx = cs->host.nx;
    size_t sb = sizeof(double) * (size_t)nk_src * nx;
    DBuf dS, dP, dks, dkg, dcl;
    if (S_T) { HIPCHK(dS.alloc(sb)); HIPCHK(hipMemcpyAsync(dS.p, S_T, sb, hipMemcpyHostToDevice, ctx->stream)); }
    if (S_P) { HIPCHK(dP.alloc(sb)); HIPCHK(hipMemcpyAsync(dP.p, S_P, sb, hipMemcpyHostToDevice, ctx->stream)); }
    HIPCHK(dks.alloc(sizeof(double) * nk_src));
    HIPCHK(dkg.alloc(sizeof(double) * nkd));
    HIPCHK(dcl.alloc(sizeof(double) * 3 * nell));
    HIPCHK(hipMemcpyAsync(dks.p, k_src, sizeof(double) * nk_src, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(dkg.p, kgrid, sizeof(double) * nkd, hipMemcpyHostToDevice, ctx->stream));
    std::vector<int> ev(ells, ells + nell);
    double* d = dcl.as<double>();
    if ((r = cl_core(ctx, ctx->stream, nullptr, cs->host, cs->d_self, dS.as<double>(), dP.as<double>(),
                     dks.as<double>(), nk_src, dkg.as<double>(), nkd, ev.data(), (int)ev.size(),
                     bessel_mode, cltt ? d : nullptr, clte ? d + nell : nullptr, clee ? d + 2 * nell : nullptr,
                     nullptr, nullptr)))
        return r;
    if (cltt) HIPCHK(hipMemcpy(cltt, d, sizeof(double) * nell, hipMemcpyDeviceToHost));
    if (clte) HIPCHK(hipMemcpy(clte, d + nell, sizeof(double) * nell, hipMemcpyDeviceToHost));
    if (clee) HIPCHK(hipMemcpy(clee, d + 2 * nell, sizeof(double) * nell, hipMemcpyDeviceToHost));
    return BOLT_OK;
}

int bolt_cl_dev(bolt_ctx* ctx, int cosmo_id, const double* d_ST, const double* d_SP, const double* d_k_src,
                int nk_src, const double* d_kgrid, int nkd, const int* ells, int nell, double* d_tt, double* d_te,
                double* d_ee, int64_t* d_steps, float* ms) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->mu);  // the cosmology table and the device work
    CosmoSlot* cs;
    int r = get_cosmo(ctx, cosmo_id, &cs);
    if (r) return r;
    if ((!d_ST && !d_SP) || !d_k_src || !d_kgrid || !ells || nk_src < 2 || nkd < 2 || nell < 1)
        return set_error(BOLT_E_ARG, "bolt_cl_dev: bad argument");
    HIPCHK(hipSetDevice(ctx->device));
    std::vector<int> ev(ells, ells + nell);
    return cl_core(ctx, ctx->stream, nullptr, cs->host, cs->d_self, d_ST, d_SP, d_k_src, nk_src, d_kgrid, nkd,
                   ev.data(), (int)ev.size(), 0, d_tt, d_te, d_ee, (long long*)d_steps,
                   ms);
}

}  // extern "C"

// ------------------------------------------------------------------ serving
// Continuous batching of spectrum requests.  Each slot owns a HIP stream and
// preallocated device buffers sized for the largest request (no allocation
// per request: hipMalloc/hipFree synchronise the device and would serialise
// the slots).  A worker thread per slot takes the next queued request, builds
// its background/RECFAST tables on the host, uploads them into the slot and
// runs the solver with one workgroup per k-mode, so that the kernels of
// requests on different slots interleave on the CUs as workgroups retire.
// Admission: a request starts as soon as a slot is free; the number of slots
// is bounded by the HBM budget given at start.
namespace {
constexpr int SV_NX = 2001;            // x grid -20:0.01:0 (background.jl:86)
constexpr int SV_MAX_NK = 800;
constexpr int SV_MAX_ELL = 2500;
constexpr int SV_MAX_NKD = 5000;
constexpr int SV_MAX_N = 1024;         // state length
constexpr int SV_MAX_NQ = 48;

double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
}  // namespace

struct ServeSlot {
    hipStream_t stream = nullptr;
    double *d_coef = nullptr, *d_q = nullptr, *d_k = nullptr, *d_S = nullptr, *d_dense = nullptr, *d_cl = nullptr;
    double *d_x = nullptr, *d_states = nullptr, *d_pk = nullptr;
    CosmoDev* d_self = nullptr;
    int* d_status = nullptr;
    long long* d_ctr = nullptr;
    SolveBufs sb;
    LosBufs lb;
    std::vector<void*> allocs;
};

static size_t slot_bytes() {
    size_t b = 0;
    b += sizeof(double) * ((size_t)BOLT_NTAB * (SV_NX + 2) + 4 * SV_MAX_NQ);             // tables, q arrays
    b += sizeof(double) * ((size_t)SV_MAX_NK * SV_NX + SV_MAX_NK + SV_MAX_NKD + SV_MAX_ELL + 1 + SV_MAX_NK);
    b += sizeof(double) * (size_t)SV_MAX_NK * SV_MAX_N;                                  // plin states
    b += sizeof(double) * (size_t)(SV_MAX_ELL - 1) * (SV_MAX_NKD - 1);                   // LOS contributions
    b += sizeof(double) * 2 * (size_t)LOS_SLOTS * WAVE + sizeof(int) * (SV_MAX_ELL + 1);
    b += (sizeof(int) + 4 * sizeof(long long) + sizeof(ModeDesc)) * SV_MAX_NK;
    return b;
}

struct ServeJob {
    uint64_t id;
    bolt_request req;
    double t_submit;
};

struct Server {
    bolt_ctx* ctx = nullptr;
    std::vector<ServeSlot> slots;
    std::vector<std::thread> workers;
    std::mutex mu;
    std::condition_variable cv_job, cv_done;
    std::deque<ServeJob> queue;
    std::unordered_map<uint64_t, bolt_result> results;
    uint64_t next_id = 1;
    bool stopping = false;
};

template <class T>
static hipError_t slot_alloc(ServeSlot& s, T** p, size_t count) {
    hipError_t e = hipMalloc((void**)p, sizeof(T) * (count ? count : 1));
    if (e == hipSuccess) s.allocs.push_back((void*)*p);
    return e;
}

static int slot_create(ServeSlot& s) {
    HIPCHK(hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking));
    HIPCHK(slot_alloc(s, &s.d_coef, (size_t)BOLT_NTAB * (SV_NX + 2)));
    HIPCHK(slot_alloc(s, &s.d_q, 4 * SV_MAX_NQ));
    HIPCHK(slot_alloc(s, &s.d_self, 1));
    HIPCHK(slot_alloc(s, &s.d_k, SV_MAX_NK));
    HIPCHK(slot_alloc(s, &s.d_S, (size_t)SV_MAX_NK * SV_NX));
    HIPCHK(slot_alloc(s, &s.d_dense, SV_MAX_NKD));
    HIPCHK(slot_alloc(s, &s.d_cl, SV_MAX_ELL));
    HIPCHK(slot_alloc(s, &s.d_x, 1));
    HIPCHK(slot_alloc(s, &s.d_states, (size_t)SV_MAX_NK * SV_MAX_N));
    HIPCHK(slot_alloc(s, &s.d_pk, SV_MAX_NK));
    HIPCHK(slot_alloc(s, &s.d_status, SV_MAX_NK));
    HIPCHK(slot_alloc(s, &s.d_ctr, 4 * SV_MAX_NK));
    HIPCHK(slot_alloc(s, &s.sb.modes, SV_MAX_NK));
    HIPCHK(slot_alloc(s, &s.sb.cfgs, 1));
    HIPCHK(slot_alloc(s, &s.sb.cosmos, 1));
    HIPCHK(slot_alloc(s, &s.sb.counter, 1));
    s.sb.cap_modes = SV_MAX_NK; s.sb.cap_cfgs = 1; s.sb.cap_cosmos = 1;
    HIPCHK(slot_alloc(s, &s.lb.lidx, SV_MAX_ELL + 1));
    HIPCHK(slot_alloc(s, &s.lb.pmap, SV_MAX_ELL + 1));
    HIPCHK(slot_alloc(s, &s.lb.etaj, LOS_SLOTS * WAVE));
    HIPCHK(slot_alloc(s, &s.lb.dxj, LOS_SLOTS * WAVE));
    HIPCHK(slot_alloc(s, &s.lb.partial, (size_t)LOS_GRID * (SV_MAX_ELL + 1)));
    s.lb.cap_lidx = SV_MAX_ELL + 1; s.lb.cap_pmap = SV_MAX_ELL + 1; s.lb.cap_nxi = LOS_SLOTS * WAVE;
    s.lb.cap_partial = (size_t)LOS_GRID * (SV_MAX_ELL + 1);
    return BOLT_OK;
}

static void slot_free(ServeSlot& s) {
    if (s.stream) (void)hipStreamSynchronize(s.stream);
    for (void* p : s.allocs) (void)hipFree(p);
    s.allocs.clear();
    if (s.stream) (void)hipStreamDestroy(s.stream);
    s.stream = nullptr;
}

static int validate_request(const bolt_request* r) {
    if (!r || !r->out) return set_error(BOLT_E_ARG, "bolt_submit: NULL request or output");
    if (r->kind != BOLT_REQ_PK && r->kind != BOLT_REQ_CLTT) return set_error(BOLT_E_ARG, "bolt_submit: unknown kind");
    if (r->nk < 2 || r->nk > SV_MAX_NK) return set_error(BOLT_E_ARG, "bolt_submit: nk must be in [2, 800]");
    if (r->k) {
        for (int i = 0; i < r->nk; ++i)
            if (!(r->k[i] > 0) || !std::isfinite(r->k[i]) || (i > 0 && !(r->k[i] > r->k[i - 1])))
                return set_error(BOLT_E_ARG, "bolt_submit: k must be positive, finite and increasing");
    } else if (!(r->kmin > 0) || !(r->kmax > r->kmin) || !std::isfinite(r->kmax)) {
        return set_error(BOLT_E_ARG, "bolt_submit: need 0 < kmin < kmax");
    }
    if (r->kind == BOLT_REQ_CLTT && (r->ell_max < 2 || r->ell_max > SV_MAX_ELL || r->nkd < 2 || r->nkd > SV_MAX_NKD))
        return set_error(BOLT_E_ARG, "bolt_submit: need 2 <= ell_max <= 2500 and 2 <= nkd <= 5000");
    int rc = check_cfg(&r->cfg);
    if (rc) return rc;
    if (r->cfg.nq > SV_MAX_NQ || bolt_state_length(&r->cfg) > SV_MAX_N)
        return set_error(BOLT_E_ARG, "bolt_submit: hierarchy larger than a serving slot holds");
    if (!(r->par.h > 0) || !(r->par.Omega_r > 0) || !(r->par.N_nu > 0))
        return set_error(BOLT_E_ARG, "bolt_submit: Omega_r, N_nu and h must be positive");
    return BOLT_OK;
}

// one request on one slot; returns its status, *host_ms / *device_ms the
// host-table and device times
// a request's Background + RECFAST tables on the host (x grid -20:0.01:0)
static int request_tables(const bolt_request& rq, std::vector<double>& coef, std::vector<double>& scal,
                          std::vector<double>& xq, std::vector<double>& wq) {
    scal.assign(BOLT_NSCAL, 0.0);
    try {
        bolt::Background bg(rq.par, -20.0, 0.0, SV_NX, rq.cfg.nq);
        bg.ionization(-1.0);
        coef = bg.coef;
        scal[BOLT_S_H0] = bg.H0; scal[BOLT_S_ETA0] = bg.eta0; scal[BOLT_S_RHO_CRIT] = bg.rho_crit;
        scal[BOLT_S_OMEGA_L] = bg.Omega_L; scal[BOLT_S_TAU0] = bg.tau0;
        xq.assign(bg.cosmo.xq.begin(), bg.cosmo.xq.end());
        wq.assign(bg.cosmo.wq.begin(), bg.cosmo.wq.end());
    } catch (const std::exception& e) {
        return set_error(BOLT_E_NUMERIC, std::string("host tables: ") + e.what());
    }
    for (double v : coef) if (!std::isfinite(v)) return set_error(BOLT_E_NUMERIC, "host tables: non-finite entry");
    return BOLT_OK;
}

// the request's k grid: given, or log-spaced as the full-CMB workload's
static std::vector<double> request_k(const bolt_request& rq) {
    std::vector<double> kh(rq.nk);
    if (rq.k) {
        std::memcpy(kh.data(), rq.k, sizeof(double) * rq.nk);
    } else {
        const double l0 = std::log10(rq.kmin), l1 = std::log10(rq.kmax);
        for (int i = 0; i < rq.nk; ++i) kh[i] = std::pow(10.0, l0 + (l1 - l0) * i / (rq.nk - 1));
    }
    return kh;
}

// quadratic_k(0.01H₀, 1000H₀, nkd) (spectra.jl:60-63, 133)
static std::vector<double> request_dense(double H0, int nkd) {
    std::vector<double> dense(nkd);
    const double kmin = 0.01 * H0, kmax = 1000.0 * H0;
    for (int i = 1; i <= nkd; ++i) {
        const double f = (double)i / nkd;
        dense[i - 1] = kmin + (kmax - kmin) * (f * f);
    }
    return dense;
}

static int run_request(bolt_ctx* ctx, ServeSlot& sl, const bolt_request& rq, double* host_ms, double* device_ms) {
    const double t0 = now_ms();
    std::vector<double> coef, xq, wq, scal;
    int rt = request_tables(rq, coef, scal, xq, wq);
    if (rt) return rt;
    bolt_tables t;
    t.nx = SV_NX; t.nq = rq.cfg.nq; t.x0 = -20.0; t.x1 = 0.0;
    for (int i = 0; i < BOLT_NSCAL; ++i) t.scal[i] = scal[i];
    t.xq = xq.data(); t.wq = wq.data(); t.coef = coef.data();
    CosmoDev C;
    std::vector<double> qbuf;
    make_cosmo_host(rq.par, t, C, qbuf);
    bind_cosmo_device(C, sl.d_coef, sl.d_q);
    const double t1 = now_ms();
    *host_ms = t1 - t0;
    hipStream_t st = sl.stream;
    HIPCHK(hipMemcpyAsync(sl.d_coef, coef.data(), sizeof(double) * coef.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(sl.d_q, qbuf.data(), sizeof(double) * qbuf.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(sl.d_self, &C, sizeof(CosmoDev), hipMemcpyHostToDevice, st));
    const int nk = rq.nk;
    const std::vector<double> kh = request_k(rq);
    HIPCHK(hipMemcpyAsync(sl.d_k, kh.data(), sizeof(double) * nk, hipMemcpyHostToDevice, st));
    std::vector<ModeDesc> md(nk);
    for (int i = 0; i < nk; ++i) { md[i].k = kh[i]; md[i].cosmo = 0; md[i].cfg = 0; md[i].out = i; md[i].pad = 0; }
    const CfgDev cd = to_cfgdev(&rq.cfg);
    double ms = 0;
    int r;
    std::vector<int> status(nk);
    if (rq.kind == BOLT_REQ_PK) {
        const double x = 0.0;
        HIPCHK(hipMemcpyAsync(sl.d_x, &x, sizeof(double), hipMemcpyHostToDevice, st));
        if ((r = launch_modes(ctx, st, &sl.sb, false, {C}, {cd}, md, 0, sl.d_x, 1, sl.d_states, nullptr, sl.d_status,
                              sl.d_ctr, cd.n, &ms)))
            return r;
        hipLaunchKernelGGL(k_plin_post, dim3((nk + 127) / 128), dim3(128), 0, st, sl.sb.cosmos, sl.sb.cfgs,
                           sl.sb.modes, nk, x, sl.d_states, sl.d_pk, 0);
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(rq.out, sl.d_pk, sizeof(double) * nk, hipMemcpyDeviceToHost, st));
    } else {
        if ((r = launch_modes(ctx, st, &sl.sb, false, {C}, {cd}, md, 1, nullptr, 0, sl.d_S, nullptr, sl.d_status,
                              sl.d_ctr, 0, &ms)))
            return r;
        const int nkd = rq.nkd;
        const std::vector<double> dense = request_dense(C.H0, nkd);
        HIPCHK(hipMemcpyAsync(sl.d_dense, dense.data(), sizeof(double) * nkd, hipMemcpyHostToDevice, st));
        std::vector<int> ells(rq.ell_max - 1);
        for (int l = 2; l <= rq.ell_max; ++l) ells[l - 2] = l;
        float ms2 = 0;
        if ((r = cl_core(ctx, st, &sl.lb, C, sl.d_self, sl.d_S, nullptr, sl.d_k, nk, sl.d_dense, nkd, ells.data(),
                         (int)ells.size(), 0, sl.d_cl,
                         nullptr, nullptr, nullptr, &ms2)))
            return r;
        ms += ms2;
        HIPCHK(hipMemcpyAsync(rq.out, sl.d_cl, sizeof(double) * ells.size(), hipMemcpyDeviceToHost, st));
    }
    HIPCHK(hipMemcpyAsync(status.data(), sl.d_status, sizeof(int) * nk, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    *device_ms = ms;
    for (int i = 0; i < nk; ++i) if (status[i] != BOLT_MODE_OK) return set_error(BOLT_E_NUMERIC, "a mode failed");
    return BOLT_OK;
}

static void worker_loop(Server* sv, int w) {
    (void)hipSetDevice(sv->ctx->device);
    for (;;) {
        ServeJob job;
        {
            std::unique_lock<std::mutex> lk(sv->mu);
            sv->cv_job.wait(lk, [&] { return sv->stopping || !sv->queue.empty(); });
            if (sv->queue.empty()) return;
            job = sv->queue.front();
            sv->queue.pop_front();
            sv->results[job.id].state = BOLT_REQ_RUNNING;
        }
        const double t0 = now_ms();
        double host_ms = 0, dev_ms = 0;
        int st = run_request(sv->ctx, sv->slots[w], job.req, &host_ms, &dev_ms);
        const double t1 = now_ms();
        {
            std::lock_guard<std::mutex> lk(sv->mu);
            bolt_result& r = sv->results[job.id];
            r.state = BOLT_REQ_DONE;
            r.status = st;
            if (st) std::snprintf(r.error, sizeof(r.error), "%s", bolt_last_error());
            r.queue_ms = t0 - job.t_submit;
            r.host_ms = host_ms;
            r.device_ms = dev_ms;
            r.latency_ms = t1 - job.t_submit;
        }
        sv->cv_done.notify_all();
    }
}

// ------------------------------------------------------------ queue serving
// bolt_serve_start_queue: requests join a running solver launch.  Each
// request's device memory (tables, k grids, outputs) comes out of one HBM
// arena, first fit, sized by the request itself; a pool of host threads builds
// the requests' tables; a publisher uploads each request's tables, cosmology
// and k-modes (the work queue, in device memory) and then raises the published
// count in pinned host memory, which the workgroups of the running persistent
// launch poll (serve_claim).  The launcher drains a launch once the server has
// held no request for QS_DRAIN_MS and starts a new one whenever published
// modes are left unclaimed.  A completion thread watches the per-mode done
// flags (pinned host memory), runs the request's C_ℓ or P(k) step on its own
// stream, on CUs the solver's stream is masked off, and copies the result out.
namespace {
constexpr int QS_QCAP = 1 << 19;     // queue positions before the queue is rewound
constexpr int QS_RCAP = 256;         // requests published and not yet done
constexpr double QS_IDLE_US = 2e6;    // ~2 s without work before a workgroup leaves on its own
constexpr double QS_DRAIN_MS = 5.0;    // the launcher drains a launch after this long with no request in the server
constexpr int QS_XCD = 8;           // MI355X: 8 XCDs, each with its own L2
// Polls of a workgroup without work, every 3.4 µs x this.  They delay the scratch
// accesses of the workgroups at work (k_solve's two-pass layouts spill): with 4, 10
// modes of n = 473 took 104 to 179 ms beside 214 idle workgroups (93 with 16, the same
// as alone) and of n = 464 with 48 bins 52 to 79 (33.5); 8, 16, 32 and 64 are alike.
constexpr int QS_POLL_SLEEPS = 16;
constexpr size_t QS_ALIGN = 256;
// Layout of a launch (solve_layout.h): up to 512 rows and 16 momentum bins, unless a
// request needs the one of any size, which is slower for all (10 modes of n = 323: 90
// against 81 ms, n = 473: 93 against 81, n = 197: 85 against 77).
constexpr int QS_LAYOUT = 2;
}  // namespace

struct QArena {
    size_t size = 0;
    std::map<size_t, size_t> free_;  // offset -> bytes
    size_t used = 0, peak = 0;
    void init(size_t bytes) { size = bytes; free_.clear(); free_[0] = bytes; used = peak = 0; }
    bool alloc(size_t bytes, size_t* off) {
        bytes = (bytes + QS_ALIGN - 1) / QS_ALIGN * QS_ALIGN;
        for (auto it = free_.begin(); it != free_.end(); ++it) {
            if (it->second < bytes) continue;
            *off = it->first;
            const size_t rest = it->second - bytes, o2 = it->first + bytes;
            free_.erase(it);
            if (rest) free_[o2] = rest;
            used += bytes;
            peak = std::max(peak, used);
            return true;
        }
        return false;
    }
    void release(size_t off, size_t bytes) {
        bytes = (bytes + QS_ALIGN - 1) / QS_ALIGN * QS_ALIGN;
        used -= bytes;
        auto it = free_.emplace(off, bytes).first;
        auto nx = std::next(it);
        if (nx != free_.end() && it->first + it->second == nx->first) { it->second += nx->second; free_.erase(nx); }
        if (it != free_.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) { pv->second += it->second; free_.erase(it); }
        }
    }
};

struct QReq {
    uint64_t id;
    bolt_request rq;
    double t_submit = 0, t_start = 0, host_ms = 0, t_pub = 0, t_solved = 0;
    std::vector<double> coef, scal, xq, wq, kh;
    size_t off = 0, bytes = 0;
    int slot = -1, q0 = 0, epoch_pub = 0, status = BOLT_OK;
    size_t o_coef = 0, o_q = 0, o_k = 0, o_out = 0, o_dense = 0, o_cl = 0, o_pk = 0, o_md = 0;
    CosmoDev C;
};

struct QServer {
    bolt_ctx* ctx = nullptr;
    char* arena_d = nullptr;
    QArena arena;
    // pinned host memory: staging of the device copies below
    ModeDesc* ring = nullptr;
    CosmoDev* cosmos = nullptr;
    CfgDev* cfgs = nullptr;
    // pinned host memory the device polls and writes
    int* ctl = nullptr;  // [0] published, [1] closed, [2] epoch of the launch to drain
    int* done = nullptr;
    // device memory: the work queue and the request slots' cosmologies and configurations
    ModeDesc* d_ring = nullptr;
    CosmoDev* d_cosmos = nullptr;
    CfgDev* d_cfgs = nullptr;
    int* d_counter = nullptr;
    int* d_leave = nullptr;  // epoch of the last launch a workgroup has left
    int* d_status = nullptr;
    long long* d_ctr = nullptr;
    double* d_xzero = nullptr;
    LosBufs lb;
    std::vector<void*> dallocs;
    hipStream_t s_solve = nullptr, s_copy = nullptr, s_post = nullptr;
    size_t lds = 0;
    int grid = 0;
    int poll_sleeps = QS_POLL_SLEEPS;
    bool cu_mask = true;  // the solver and the post-step streams on disjoint CU masks
    std::mutex mu;  // everything below
    std::condition_variable cv;
    std::deque<std::shared_ptr<QReq>> pending;       // waiting for host tables
    std::deque<std::shared_ptr<QReq>> ready;         // tables built, waiting for memory and publication
    std::vector<std::shared_ptr<QReq>> inflight;     // published, not done
    std::unordered_map<uint64_t, bolt_result> results;
    std::vector<int> free_slots;
    uint64_t next_id = 1;
    int building = 0;       // requests whose host tables are being built
    int unsettled = 0;      // requests holding queue positions and not yet done
    bool failed = false;    // a device error: requests in flight end with it
    int published = 0;
    int epoch = 0;          // launches so far
    bool running = false;   // a solver launch is in flight
    int launched = QS_LAYOUT;  // its layout
    int layout = QS_LAYOUT;    // the next launch's
    bool stopping = false;
    long long launches = 0, joined = 0, served = 0;
    std::vector<std::thread> threads;
};

static size_t qreq_layout(QReq& q) {
    const bolt_request& rq = q.rq;
    size_t b = 0;
    auto take = [&](size_t bytes) {
        const size_t o = b;
        b += (bytes + QS_ALIGN - 1) / QS_ALIGN * QS_ALIGN;
        return o;
    };
    q.o_coef = take(sizeof(double) * (size_t)BOLT_NTAB * (SV_NX + 2));
    q.o_q = take(sizeof(double) * 4 * (size_t)rq.cfg.nq);
    q.o_k = take(sizeof(double) * (size_t)rq.nk);
    if (rq.kind == BOLT_REQ_CLTT) {
        q.o_out = take(sizeof(double) * (size_t)rq.nk * SV_NX);
        q.o_dense = take(sizeof(double) * (size_t)rq.nkd);
        q.o_cl = take(sizeof(double) * (size_t)(rq.ell_max - 1));
    } else {
        q.o_out = take(sizeof(double) * (size_t)rq.nk * bolt_state_length(&rq.cfg));
        q.o_pk = take(sizeof(double) * (size_t)rq.nk);
        q.o_md = take(sizeof(ModeDesc) * (size_t)rq.nk);
    }
    return b;
}

static void qs_finish(QServer* sv, const std::shared_ptr<QReq>& q, int status) {
    bolt_result& r = sv->results[q->id];
    r.state = BOLT_REQ_DONE;
    r.status = status;
    if (status) std::snprintf(r.error, sizeof(r.error), "%s", bolt_last_error());
    r.queue_ms = q->t_start - q->t_submit;
    r.host_ms = q->host_ms;
    r.latency_ms = now_ms() - q->t_submit;
}

// host tables, one request at a time per thread
static void qs_tables_loop(QServer* sv) {
    for (;;) {
        std::shared_ptr<QReq> q;
        {
            std::unique_lock<std::mutex> lk(sv->mu);
            sv->cv.wait(lk, [&] { return sv->stopping || !sv->pending.empty(); });
            if (sv->pending.empty()) return;
            q = sv->pending.front();
            sv->pending.pop_front();
            ++sv->building;
            q->t_start = now_ms();
            sv->results[q->id].state = BOLT_REQ_RUNNING;
        }
        const double t0 = now_ms();
        const int r = request_tables(q->rq, q->coef, q->scal, q->xq, q->wq);
        q->kh = request_k(q->rq);
        q->host_ms = now_ms() - t0;
        std::lock_guard<std::mutex> lk(sv->mu);
        --sv->building;
        if (r) {
            qs_finish(sv, q, r);
        } else {
            sv->ready.push_back(q);
        }
        sv->cv.notify_all();
    }
}

// memory, upload and publication, in arrival order; then the launcher
static int qs_publish(QServer* sv, QReq& q) {
    const bolt_request& rq = q.rq;
    char* base = sv->arena_d + q.off;
    bolt_tables t;
    t.nx = SV_NX; t.nq = rq.cfg.nq; t.x0 = -20.0; t.x1 = 0.0;
    for (int i = 0; i < BOLT_NSCAL; ++i) t.scal[i] = q.scal[i];
    t.xq = q.xq.data(); t.wq = q.wq.data(); t.coef = q.coef.data();
    std::vector<double> qbuf;
    make_cosmo_host(rq.par, t, q.C, qbuf);
    bind_cosmo_device(q.C, (double*)(base + q.o_coef), (double*)(base + q.o_q));
    hipStream_t st = sv->s_copy;
    HIPCHK(hipMemcpyAsync(base + q.o_coef, q.coef.data(), sizeof(double) * q.coef.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(base + q.o_q, qbuf.data(), sizeof(double) * qbuf.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(base + q.o_k, q.kh.data(), sizeof(double) * rq.nk, hipMemcpyHostToDevice, st));
    std::vector<double> dense;
    if (rq.kind == BOLT_REQ_CLTT) {
        dense = request_dense(q.C.H0, rq.nkd);
        HIPCHK(hipMemcpyAsync(base + q.o_dense, dense.data(), sizeof(double) * rq.nkd, hipMemcpyHostToDevice, st));
    } else {
        std::vector<ModeDesc> pm(rq.nk);
        for (int i = 0; i < rq.nk; ++i) { pm[i].k = q.kh[i]; pm[i].cosmo = q.slot; pm[i].cfg = q.slot; pm[i].out = i; pm[i].pad = 0; }
        HIPCHK(hipMemcpyAsync(base + q.o_md, pm.data(), sizeof(ModeDesc) * rq.nk, hipMemcpyHostToDevice, st));
    }
    sv->cosmos[q.slot] = q.C;
    sv->cfgs[q.slot] = to_cfgdev(&rq.cfg);
    // the request's modes, largest k (most steps) first
    const int n = bolt_state_length(&rq.cfg);
    const size_t out0 = (q.off + q.o_out) / sizeof(double);
    for (int j = 0; j < rq.nk; ++j) {
        const int i = rq.nk - 1 - j;
        ModeDesc& m = sv->ring[q.q0 + j];
        m.k = q.kh[i];
        m.cosmo = q.slot;
        m.cfg = q.slot;
        m.out = (int)(out0 + (size_t)i * (rq.kind == BOLT_REQ_CLTT ? SV_NX : n));
        m.pad = rq.kind == BOLT_REQ_CLTT ? 1 : 0;
        sv->done[q.q0 + j] = 0;
    }
    HIPCHK(hipMemcpyAsync(sv->d_cosmos + q.slot, sv->cosmos + q.slot, sizeof(CosmoDev), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(sv->d_cfgs + q.slot, sv->cfgs + q.slot, sizeof(CfgDev), hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(sv->d_ring + q.q0, sv->ring + q.q0, sizeof(ModeDesc) * rq.nk, hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st));
    std::atomic_thread_fence(std::memory_order_seq_cst);
    __atomic_store_n(&sv->ctl[0], q.q0 + rq.nk, __ATOMIC_RELEASE);
    q.t_pub = now_ms();
    return BOLT_OK;
}

static void qs_admit_loop(QServer* sv) {
    (void)hipSetDevice(sv->ctx->device);
    for (;;) {
        std::shared_ptr<QReq> q;
        int running_before = 0;
        {
            std::unique_lock<std::mutex> lk(sv->mu);
            for (;;) {
                if (sv->stopping && sv->ready.empty() && sv->pending.empty() && !sv->building) return;
                if (sv->failed) {
                    for (auto& r : sv->ready) qs_finish(sv, r, set_error(BOLT_E_DEVICE, "serving: device error"));
                    sv->ready.clear();
                }
                if (!sv->ready.empty()) {
                    std::shared_ptr<QReq>& f = sv->ready.front();
                    if (!f->bytes) f->bytes = qreq_layout(*f);
                    const bool room = sv->published + f->rq.nk <= QS_QCAP && !sv->free_slots.empty();
                    if (room && sv->arena.alloc(f->bytes, &f->off)) {
                        q = f;
                        sv->ready.pop_front();
                        q->slot = sv->free_slots.back();
                        sv->free_slots.pop_back();
                        q->q0 = sv->published;
                        sv->published += q->rq.nk;
                        ++sv->unsettled;
                        running_before = sv->running ? sv->epoch : 0;
                        break;
                    }
                }
                sv->cv.wait_for(lk, std::chrono::milliseconds(2));
            }
        }
        const CfgDev cd = to_cfgdev(&q->rq.cfg);
        const int layout = wsn_layout(cd.n, cd.nq);
        {
            // a running launch whose layout does not hold the request ends first; what it
            // leaves unclaimed goes to the next one
            std::unique_lock<std::mutex> lk(sv->mu);
            sv->layout = std::max(sv->layout, layout);
            while (sv->running && sv->launched < layout) {
                __atomic_store_n(&sv->ctl[2], sv->epoch, __ATOMIC_RELEASE);
                sv->cv.wait_for(lk, std::chrono::milliseconds(1));
            }
        }
        const int r = qs_publish(sv, *q);
        std::lock_guard<std::mutex> lk(sv->mu);
        if (r) {  // nothing was published for it: its positions hold no work (status stays 0, done 0)
            sv->arena.release(q->off, q->bytes);
            sv->free_slots.push_back(q->slot);
            --sv->unsettled;
            sv->failed = true;
            qs_finish(sv, q, r);
        } else {
            // admitted into a running launch: the same launch was running before and after publication
            q->epoch_pub = (running_before && sv->running && sv->epoch == running_before) ? running_before : 0;
            sv->inflight.push_back(q);
        }
        sv->cv.notify_all();
    }
}

// solver launches: whenever published modes are left unclaimed; the queue is
// rewound when every published mode is done
static void qs_launch_loop(QServer* sv) {
    (void)hipSetDevice(sv->ctx->device);
    int claimed = 0;
    for (;;) {
        int ep, layout;
        {
            std::unique_lock<std::mutex> lk(sv->mu);
            for (;;) {
                if (sv->failed) return;
                if (__atomic_load_n(&sv->ctl[0], __ATOMIC_ACQUIRE) > claimed) break;
                if (!sv->unsettled && sv->published > 0 && sv->published == claimed) {
                    // rewind: nothing published is pending (ready requests publish afresh from 0)
                    int zero = 0;
                    if (hipMemcpyAsync(sv->d_counter, &zero, sizeof(int), hipMemcpyHostToDevice, sv->s_solve) ==
                            hipSuccess &&
                        hipStreamSynchronize(sv->s_solve) == hipSuccess) {
                        __atomic_store_n(&sv->ctl[0], 0, __ATOMIC_RELEASE);
                        sv->published = 0;
                        sv->layout = QS_LAYOUT;
                        claimed = 0;
                    }
                }
                if (sv->stopping && sv->pending.empty() && sv->ready.empty() && !sv->building && !sv->unsettled)
                    return;
                sv->cv.wait_for(lk, std::chrono::milliseconds(1));
            }
            ep = ++sv->epoch;
            sv->running = true;
            sv->launched = sv->layout;
            layout = sv->layout;
            ++sv->launches;
        }
        SolveArgs A;
        A.cosmos = sv->d_cosmos; A.cfgs = sv->d_cfgs; A.modes = sv->d_ring; A.nmodes = QS_QCAP;
        A.work_counter = sv->d_counter; A.out_mode = 0; A.x_save = sv->d_xzero; A.nsave = 1;
        A.out = (double*)sv->arena_d; A.out2 = nullptr; A.status = sv->d_status; A.counters = sv->d_ctr;
        A.n_state_stride = 0; A.lds_doubles = (int)(sv->lds / sizeof(double));
        A.serve = 1; A.epoch = ep; A.poll_sleeps = sv->poll_sleeps;
        A.idle_limit = (int)std::max(1000.0, QS_IDLE_US / (3.4 * sv->poll_sleeps + 1.0));
        A.published = sv->ctl; A.closed = sv->ctl + 1; A.drain = sv->ctl + 2; A.leave = sv->d_leave;
        A.done = sv->done;
        launch_solver(SR_DEFAULT, layout, false, sv->grid, sv->lds, sv->s_solve, A);
        bool ok = hipGetLastError() == hipSuccess;
        // wait for the launch; drain it once the server has held no request for QS_DRAIN_MS
        double idle_since = -1.0;
        while (ok) {
            const hipError_t e = hipStreamQuery(sv->s_solve);
            if (e == hipSuccess) break;
            if (e != hipErrorNotReady) { ok = false; break; }
            std::unique_lock<std::mutex> lk(sv->mu);
            const bool idle = !sv->unsettled && sv->ready.empty() && sv->pending.empty() && !sv->building;
            if (!idle) {
                idle_since = -1.0;
            } else if (idle_since < 0) {
                idle_since = now_ms();
            } else if (now_ms() - idle_since > QS_DRAIN_MS || sv->stopping) {
                __atomic_store_n(&sv->ctl[2], ep, __ATOMIC_RELEASE);
            }
            sv->cv.wait_for(lk, std::chrono::microseconds(200));
        }
        int c = claimed;
        ok = ok && hipStreamSynchronize(sv->s_solve) == hipSuccess &&
             hipMemcpy(&c, sv->d_counter, sizeof(int), hipMemcpyDeviceToHost) == hipSuccess;
        std::lock_guard<std::mutex> lk(sv->mu);
        sv->running = false;
        if (ok) claimed = c;
        else sv->failed = true;  // a device error: the requests in flight report it
        sv->cv.notify_all();
    }
}

// completion: every mode of a request done -> its C_ℓ or P(k), then the result
static void qs_complete_loop(QServer* sv) {
    (void)hipSetDevice(sv->ctx->device);
    for (;;) {
        std::shared_ptr<QReq> q;
        {
            std::unique_lock<std::mutex> lk(sv->mu);
            for (;;) {
                for (auto it = sv->inflight.begin(); it != sv->inflight.end(); ++it) {
                    QReq& r = **it;
                    bool all = true;
                    for (int j = 0; j < r.rq.nk && all; ++j) all = __atomic_load_n(&sv->done[r.q0 + j], __ATOMIC_ACQUIRE) != 0;
                    if (all) { q = *it; q->t_solved = now_ms(); sv->inflight.erase(it); break; }
                }
                if (q) break;
                if (sv->failed && !sv->running) {
                    for (auto& r : sv->inflight) {
                        qs_finish(sv, r, set_error(BOLT_E_DEVICE, "serving: device error"));
                        sv->arena.release(r->off, r->bytes);
                        sv->free_slots.push_back(r->slot);
                        --sv->unsettled;
                    }
                    sv->inflight.clear();
                }
                if (sv->stopping && sv->pending.empty() && sv->ready.empty() && !sv->building && !sv->unsettled)
                    return;
                sv->cv.wait_for(lk, std::chrono::microseconds(200));
            }
        }
        const bolt_request& rq = q->rq;
        char* base = sv->arena_d + q->off;
        bool joined = q->epoch_pub != 0;
        for (int j = 0; j < rq.nk && joined; ++j) joined = sv->done[q->q0 + j] == q->epoch_pub;
        std::vector<int> status(rq.nk);
        int r = BOLT_OK;
        hipStream_t st = sv->s_post;
        const double tp0 = now_ms();
        if (hipMemcpyAsync(status.data(), sv->d_status + q->q0, sizeof(int) * rq.nk, hipMemcpyDeviceToHost, st) !=
            hipSuccess)
            r = set_error(BOLT_E_DEVICE, "serving: status copy failed");
        if (!r && rq.kind == BOLT_REQ_CLTT) {
            std::vector<int> ells(rq.ell_max - 1);
            for (int l = 2; l <= rq.ell_max; ++l) ells[l - 2] = l;
            float ms = 0;
            r = cl_core(sv->ctx, st, &sv->lb, q->C, sv->d_cosmos + q->slot, (double*)(base + q->o_out), nullptr,
                        (double*)(base + q->o_k), rq.nk, (double*)(base + q->o_dense), rq.nkd, ells.data(),
                        (int)ells.size(), 0, (double*)(base + q->o_cl), nullptr, nullptr, nullptr, &ms);
            if (!r && hipMemcpyAsync(rq.out, base + q->o_cl, sizeof(double) * ells.size(), hipMemcpyDeviceToHost, st) !=
                          hipSuccess)
                r = set_error(BOLT_E_DEVICE, "serving: result copy failed");
        } else if (!r) {
            hipLaunchKernelGGL(k_plin_post, dim3((rq.nk + 127) / 128), dim3(128), 0, st, (const CosmoDev*)sv->d_cosmos,
                               (const CfgDev*)sv->d_cfgs, (const ModeDesc*)(base + q->o_md), rq.nk, 0.0,
                               (const double*)(base + q->o_out), (double*)(base + q->o_pk),
                               bolt_state_length(&rq.cfg));
            if (hipGetLastError() != hipSuccess ||
                hipMemcpyAsync(rq.out, base + q->o_pk, sizeof(double) * rq.nk, hipMemcpyDeviceToHost, st) != hipSuccess)
                r = set_error(BOLT_E_DEVICE, "serving: plin post step failed");
        }
        if (hipStreamSynchronize(st) != hipSuccess && !r) r = set_error(BOLT_E_DEVICE, "serving: stream failed");
        const double dev_ms = now_ms() - tp0;
        for (int i = 0; i < rq.nk && !r; ++i)
            if (status[i] != BOLT_MODE_OK) r = set_error(BOLT_E_NUMERIC, "a mode failed");
        std::lock_guard<std::mutex> lk(sv->mu);
        sv->arena.release(q->off, q->bytes);
        sv->free_slots.push_back(q->slot);
        --sv->unsettled;
        qs_finish(sv, q, r);
        bolt_result& res = sv->results[q->id];
        res.device_ms = dev_ms;
        res.solve_ms = q->t_solved - q->t_pub;
        res.joined_running = joined ? 1 : 0;
        sv->joined += joined ? 1 : 0;
        ++sv->served;
        sv->cv.notify_all();
    }
}

// the server's device and pinned memory and streams (its threads have ended)
static void qserver_free(QServer* sv) {
    if (sv->s_solve) (void)hipStreamSynchronize(sv->s_solve);
    if (sv->s_post) (void)hipStreamSynchronize(sv->s_post);
    for (void* p : sv->dallocs) (void)hipFree(p);
    sv->dallocs.clear();
    for (void** p : {(void**)&sv->ring, (void**)&sv->cosmos, (void**)&sv->cfgs, (void**)&sv->ctl, (void**)&sv->done})
        if (*p) { (void)hipHostFree(*p); *p = nullptr; }
    for (hipStream_t* s : {&sv->s_solve, &sv->s_copy, &sv->s_post})
        if (*s) { (void)hipStreamDestroy(*s); *s = nullptr; }
}

static void qserver_stop(QServer* sv) {
    {
        std::lock_guard<std::mutex> lk(sv->mu);
        sv->stopping = true;
    }
    sv->cv.notify_all();
    // the admitter and table threads finish the queued work first; then the queue closes
    for (size_t i = 0; i < sv->threads.size(); ++i) sv->threads[i].join();
    sv->threads.clear();
    __atomic_store_n(&sv->ctl[1], 1, __ATOMIC_RELEASE);
    qserver_free(sv);
    sv->cv.notify_all();
}

template <class T>
static hipError_t qs_dalloc(QServer* sv, T** p, size_t count) {
    hipError_t e = hipMalloc((void**)p, sizeof(T) * (count ? count : 1));
    if (e == hipSuccess) sv->dallocs.push_back((void*)*p);
    return e;
}

static int qserver_create(bolt_ctx* ctx, double hbm_gib, int host_threads, std::shared_ptr<QServer>* out) {
    auto owner = std::make_shared<QServer>();
    QServer* sv = owner.get();
    sv->ctx = ctx;
    auto fail = [&](int code, const char* msg) {
        qserver_free(sv);
        return set_error(code, msg);
    };
    const size_t fixed = (sizeof(ModeDesc) + sizeof(int) + sizeof(long long) * 4) * QS_QCAP +
                         (sizeof(CosmoDev) + sizeof(CfgDev)) * QS_RCAP +
                         sizeof(double) * ((size_t)LOS_GRID * (SV_MAX_ELL + 1) + 2 * LOS_SLOTS * WAVE) +
                         sizeof(int) * 2 * (SV_MAX_ELL + 1);
    const double want = hbm_gib * 1073741824.0;
    if (want < (double)fixed + 4.0 * 1048576.0) return fail(BOLT_E_NOMEM, "bolt_serve_start_queue: the HBM budget is too small");
    // a mode's output offset is an int count of doubles: the arena stays below 2^31 doubles
    const size_t arena = std::min((size_t)(want - (double)fixed), (size_t)15 << 30);
    const unsigned hf = hipHostMallocMapped | hipHostMallocCoherent;
    if (hipHostMalloc((void**)&sv->ring, sizeof(ModeDesc) * QS_QCAP, hf) != hipSuccess ||
        hipHostMalloc((void**)&sv->cosmos, sizeof(CosmoDev) * QS_RCAP, hf) != hipSuccess ||
        hipHostMalloc((void**)&sv->cfgs, sizeof(CfgDev) * QS_RCAP, hf) != hipSuccess ||
        hipHostMalloc((void**)&sv->ctl, sizeof(int) * 3, hf) != hipSuccess ||
        hipHostMalloc((void**)&sv->done, sizeof(int) * QS_QCAP, hf) != hipSuccess)
        return fail(BOLT_E_NOMEM, "bolt_serve_start_queue: pinned host memory");
    std::memset(sv->ctl, 0, sizeof(int) * 3);
    std::memset(sv->done, 0, sizeof(int) * QS_QCAP);
    if (hipMalloc((void**)&sv->arena_d, arena) != hipSuccess) return fail(BOLT_E_NOMEM, "bolt_serve_start_queue: arena");
    sv->dallocs.push_back(sv->arena_d);
    sv->arena.init(arena);
    if (qs_dalloc(sv, &sv->d_ring, QS_QCAP) || qs_dalloc(sv, &sv->d_cosmos, QS_RCAP) ||
        qs_dalloc(sv, &sv->d_cfgs, QS_RCAP) || qs_dalloc(sv, &sv->d_counter, 1) || qs_dalloc(sv, &sv->d_leave, 1) ||
        qs_dalloc(sv, &sv->d_status, QS_QCAP) ||
        qs_dalloc(sv, &sv->d_ctr, 4 * (size_t)QS_QCAP) || qs_dalloc(sv, &sv->d_xzero, 1) ||
        qs_dalloc(sv, &sv->lb.lidx, SV_MAX_ELL + 1) || qs_dalloc(sv, &sv->lb.pmap, SV_MAX_ELL + 1) ||
        qs_dalloc(sv, &sv->lb.etaj, LOS_SLOTS * WAVE) || qs_dalloc(sv, &sv->lb.dxj, LOS_SLOTS * WAVE) ||
        qs_dalloc(sv, &sv->lb.partial, (size_t)LOS_GRID * (SV_MAX_ELL + 1)))
        return fail(BOLT_E_NOMEM, "bolt_serve_start_queue: work arrays");
    sv->lb.cap_lidx = SV_MAX_ELL + 1; sv->lb.cap_pmap = SV_MAX_ELL + 1; sv->lb.cap_nxi = LOS_SLOTS * WAVE;
    sv->lb.cap_partial = (size_t)LOS_GRID * (SV_MAX_ELL + 1);
    const double zero = 0.0;
    const int izero = 0;
    if (hipMemcpy(sv->d_xzero, &zero, sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(sv->d_counter, &izero, sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(sv->d_leave, &izero, sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
        return fail(BOLT_E_DEVICE, "bolt_serve_start_queue: initialisation");
    // The solver's stream is masked to n_cu - reserve CUs and the copy and
    // post-step streams to the other ones: without the masks, the C_ℓ kernels of
    // a finished request get no CU while the persistent launch is resident, even
    // on CUs it leaves free, and wait for its workgroups to leave.  The reserve
    // is whole XCDs (mask bits 32x .. 32x + 31 are one XCD's CUs): one XCD by
    // default, whose L2 serves the C_ℓ kernels alone.  Splitting an XCD between
    // the two (16 or 48 CUs) gave multi-second latency tails under load.
    // Tunables: BOLT_QS_RESERVE_CU (rounded up to whole XCDs), BOLT_QS_POLL_SLEEPS,
    // BOLT_QS_CU_MASK=0 (plain streams, 16 CUs left free)
    const int per_xcd = std::max(1, ctx->n_cu / QS_XCD);
    int reserve = per_xcd;
    if (const char* e = std::getenv("BOLT_QS_RESERVE_CU"))
        reserve = std::min(ctx->n_cu / 2, (std::max(1, std::atoi(e)) + per_xcd - 1) / per_xcd * per_xcd);
    if (const char* e = std::getenv("BOLT_QS_CU_MASK")) sv->cu_mask = std::atoi(e) != 0;
    if (!sv->cu_mask) reserve = std::min(reserve, 16);
    if (const char* e = std::getenv("BOLT_QS_POLL_SLEEPS")) sv->poll_sleeps = std::max(1, std::min(4096, std::atoi(e)));
    const int nsolve = std::max(1, ctx->n_cu - reserve);
    if (sv->cu_mask) {
        // mask bit i is the i-th CU of the device
        const int words = (ctx->n_cu + 31) / 32;
        std::vector<uint32_t> m_solve(words, 0u), m_post(words, 0u);
        for (int i = 0; i < ctx->n_cu; ++i) (i < nsolve ? m_solve : m_post)[i / 32] |= 1u << (i % 32);
        if (hipExtStreamCreateWithCUMask(&sv->s_solve, words, m_solve.data()) != hipSuccess ||
            hipExtStreamCreateWithCUMask(&sv->s_copy, words, m_post.data()) != hipSuccess ||
            hipExtStreamCreateWithCUMask(&sv->s_post, words, m_post.data()) != hipSuccess)
            return fail(BOLT_E_DEVICE, "bolt_serve_start_queue: hipExtStreamCreateWithCUMask");
    } else {
        for (hipStream_t* s : {&sv->s_solve, &sv->s_copy, &sv->s_post})
            if (hipStreamCreateWithFlags(s, hipStreamNonBlocking) != hipSuccess)
                return fail(BOLT_E_DEVICE, "bolt_serve_start_queue: hipStreamCreate");
    }
    sv->lds = (size_t)ctx->lds_max;
    sv->grid = nsolve;
    for (int i = QS_RCAP - 1; i >= 0; --i) sv->free_slots.push_back(i);
    const int nt = std::max(1, host_threads);
    for (int i = 0; i < nt; ++i) sv->threads.emplace_back(qs_tables_loop, sv);
    sv->threads.emplace_back(qs_admit_loop, sv);
    sv->threads.emplace_back(qs_launch_loop, sv);
    sv->threads.emplace_back(qs_complete_loop, sv);
    *out = owner;
    return BOLT_OK;
}

static void server_stop(Server* sv) {
    {
        std::lock_guard<std::mutex> lk(sv->mu);
        sv->stopping = true;
    }
    sv->cv_job.notify_all();
    for (auto& t : sv->workers) t.join();
    for (auto& s : sv->slots) slot_free(s);
    sv->cv_done.notify_all();
}

// a request's result from either server; wait: block until it is done, then
// drop it from the server's table
template <class S>
static int result_of(const std::shared_ptr<S>& sv, std::condition_variable& cv, uint64_t id, bool wait,
                     bolt_result* res) {
    std::unique_lock<std::mutex> lq(sv->mu);
    auto it = sv->results.find(id);
    if (it == sv->results.end()) return set_error(BOLT_E_ARG, "unknown request id");
    if (wait) {
        cv.wait(lq, [&] { auto f = sv->results.find(id); return f == sv->results.end() || f->second.state == BOLT_REQ_DONE; });
        it = sv->results.find(id);
        if (it == sv->results.end()) return set_error(BOLT_E_ARG, "unknown request id");
    }
    *res = it->second;
    if (wait) sv->results.erase(it);
    return BOLT_OK;
}

extern "C" {

int bolt_serve_start(bolt_ctx* ctx, int slots, double hbm_gib) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    if (slots < 1 || !(hbm_gib > 0)) return set_error(BOLT_E_ARG, "bolt_serve_start: need slots >= 1, hbm_gib > 0");
    std::lock_guard<std::mutex> lk(ctx->server_mu);
    if (ctx->server || ctx->qserver) return set_error(BOLT_E_STATE, "bolt_serve_start: already serving");
    const int by_hbm = (int)(hbm_gib * 1073741824.0 / (double)slot_bytes());
    const int n = std::min(slots, by_hbm);
    if (n < 1) return set_error(BOLT_E_NOMEM, "bolt_serve_start: the HBM budget holds no slot");
    HIPCHK(hipSetDevice(ctx->device));
    auto sv = std::make_shared<Server>();
    sv->ctx = ctx;
    sv->slots.resize(n);
    for (auto& s : sv->slots) {
        int r = slot_create(s);
        if (r) {
            for (auto& q : sv->slots) slot_free(q);
            return r;
        }
    }
    for (int w = 0; w < n; ++w) sv->workers.emplace_back(worker_loop, sv.get(), w);
    ctx->server = sv;
    return BOLT_OK;
}

int bolt_serve_start_queue(bolt_ctx* ctx, double hbm_gib, int host_threads) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    if (!(hbm_gib > 0) || host_threads < 0) return set_error(BOLT_E_ARG, "bolt_serve_start_queue: bad argument");
    std::lock_guard<std::mutex> lk(ctx->server_mu);
    if (ctx->server || ctx->qserver) return set_error(BOLT_E_STATE, "bolt_serve_start_queue: already serving");
    HIPCHK(hipSetDevice(ctx->device));
    return qserver_create(ctx, hbm_gib, host_threads ? host_threads : 4, &ctx->qserver);
}

int bolt_serve_queue_info(bolt_ctx* ctx, bolt_queue_info* info) {
    if (!ctx || !info) return set_error(BOLT_E_ARG, "bolt_serve_queue_info: NULL argument");
    std::shared_ptr<QServer> sv;
    {
        std::lock_guard<std::mutex> lk(ctx->server_mu);
        sv = ctx->qserver;
    }
    if (!sv) return set_error(BOLT_E_STATE, "bolt_serve_queue_info: no queue server");
    std::lock_guard<std::mutex> lq(sv->mu);
    info->launches = sv->launches;
    info->served = sv->served;
    info->joined_running = sv->joined;
    info->arena_bytes = (long long)sv->arena.size;
    info->arena_peak_bytes = (long long)sv->arena.peak;
    info->solver_workgroups = sv->grid;
    return BOLT_OK;
}

int bolt_serve_slots(bolt_ctx* ctx) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::lock_guard<std::mutex> lk(ctx->server_mu);
    return ctx->server ? (int)ctx->server->slots.size() : 0;
}

int bolt_submit(bolt_ctx* ctx, const bolt_request* req, uint64_t* id) {
    if (!ctx || !id) return set_error(BOLT_E_ARG, "bolt_submit: NULL argument");
    int r = validate_request(req);
    if (r) return r;
    std::lock_guard<std::mutex> lk(ctx->server_mu);
    bolt_result res;
    std::memset(&res, 0, sizeof(res));
    res.state = BOLT_REQ_QUEUED;
    if (ctx->qserver) {
        QServer* sv = ctx->qserver.get();
        const CfgDev cd = to_cfgdev(&req->cfg);
        if (solve_lds(cd.n, cd.nq) > (size_t)ctx->lds_max)
            return set_error(BOLT_E_ARG, "bolt_submit: hierarchy too large for one workgroup's LDS");
        auto q = std::make_shared<QReq>();
        q->rq = *req;
        q->t_submit = now_ms();
        q->bytes = qreq_layout(*q);
        if (q->bytes > sv->arena.size) return set_error(BOLT_E_NOMEM, "bolt_submit: the request exceeds the HBM arena");
        {
            std::lock_guard<std::mutex> lq(sv->mu);
            q->id = sv->next_id++;
            sv->results[q->id] = res;
            sv->pending.push_back(q);
            *id = q->id;
        }
        sv->cv.notify_all();
        return BOLT_OK;
    }
    if (!ctx->server) return set_error(BOLT_E_STATE, "bolt_submit: call bolt_serve_start first");
    Server* sv = ctx->server.get();
    {
        std::lock_guard<std::mutex> lq(sv->mu);
        ServeJob j;
        j.id = sv->next_id++;
        j.req = *req;
        j.t_submit = now_ms();
        sv->results[j.id] = res;
        sv->queue.push_back(j);
        *id = j.id;
    }
    sv->cv_job.notify_one();
    return BOLT_OK;
}

int bolt_poll(bolt_ctx* ctx, uint64_t id, bolt_result* res) {
    if (!ctx || !res) return set_error(BOLT_E_ARG, "bolt_poll: NULL argument");
    std::shared_ptr<Server> a;
    std::shared_ptr<QServer> b;
    {
        std::lock_guard<std::mutex> lk(ctx->server_mu);
        a = ctx->server;
        b = ctx->qserver;
    }
    if (b) return result_of(b, b->cv, id, false, res);
    if (a) return result_of(a, a->cv_done, id, false, res);
    return set_error(BOLT_E_STATE, "bolt_poll: not serving");
}

int bolt_wait(bolt_ctx* ctx, uint64_t id, bolt_result* res) {
    if (!ctx || !res) return set_error(BOLT_E_ARG, "bolt_wait: NULL argument");
    std::shared_ptr<Server> a;
    std::shared_ptr<QServer> b;
    {
        std::lock_guard<std::mutex> lk(ctx->server_mu);
        a = ctx->server;
        b = ctx->qserver;
    }
    // the shared pointers keep the server alive while this thread waits, also
    // across a concurrent bolt_serve_stop (which finishes every request first)
    if (b) return result_of(b, b->cv, id, true, res);
    if (a) return result_of(a, a->cv_done, id, true, res);
    return set_error(BOLT_E_STATE, "bolt_wait: not serving");
}

int bolt_serve_stop(bolt_ctx* ctx) {
    if (!ctx) return set_error(BOLT_E_STATE, "ctx is NULL");
    std::shared_ptr<Server> a;
    std::shared_ptr<QServer> b;
    {
        std::lock_guard<std::mutex> lk(ctx->server_mu);
        a = ctx->server;
        b = ctx->qserver;
    }
    if (a) server_stop(a.get());
    if (b) qserver_stop(b.get());
    std::lock_guard<std::mutex> lk(ctx->server_mu);
    ctx->server.reset();
    ctx->qserver.reset();
    return BOLT_OK;
}

}  // extern "C"

// ============================================================================
// Moments of spherical Bessel functions, their tables and the Filon rule
// (src/bessel/moments.jl, interpolator.jl, integrator.jl)
//
// I_m(x) = ∫_0^x t^m j_ν(t) dt.  Three device evaluations:
// - the Lommel-function asymptotic (moments.jl:5-21, 72-86), FP64, with its
//   series truncated as the reference truncates it (at most 21 terms, stop
//   once a term is below 1e-16 of the sum);
// - the Maclaurin series of ₁F₂ in FP64 (moments.jl:97-102, weniger.jl:237-249),
//   used below a table's range;
// - for the table nodes below x = 40, where the reference sums ₁F₂ by Weniger's
//   transformation in Double64 (below 50, moments.jl:89-94):
//   · below x = 20 the same series in double-double arithmetic,
//     I_m = x^{ν+m+1}/(2ν+1)!! Σ_k (−x²/2)^k / (k! (2ν+3)…(2ν+2k+1) (2k+ν+m+1));
//     its terms reach about e^x/√(2πx)·x^{ν+m+1}/(2ν+1)!! against the moment,
//     ~1e12 of it at x = 20 but ~1e20 at 40 for m = 3, too much for 2⁻¹⁰⁶;
//   · from 20 to 40 exact identities: ∫_0^x t^m j_ν = x^m j_{ν+1}(x) −
//     (m−ν−2) ∫_0^x t^{m−1} j_{ν+1} (from d[t^{ν+2} j_{ν+1}] = t^{ν+2} j_ν dt)
//     down to ∫_0^x j_L, and (L+1)∫j_{L+1} = L∫j_{L−1} − (2L+1) j_L(x) up from
//     ∫j_0 = Si(x), ∫j_1 = 1 − j_0(x); Si by its power series in double-double,
//     whose terms reach only ~e^x/x² against Si ≈ π/2.
//   From x = 40 on the asymptotic holds to double precision for ν ≤ 3 (the
//   tables' range of ν, like the reference's).
// A table (interpolator.jl:85-111) holds the moments m = 0..order−1 on
// LinRange(x_min, x_max, N) as cubic B-spline coefficients with Line(OnGrid())
// ends; below x_min it evaluates the FP64 series, above x_max the asymptotic.
// ============================================================================
namespace {
constexpr double MOM_CUT = 40.0;
constexpr double MOM_SQRT_HALF_PI = 1.2533141373155002512078826424055;
// prefilter: unknowns per lane, lanes per block, warm-up (the recurrences contract by
// 0.268 an unknown: 4e-28 of the start is left), and the lanes at a block's end whose
// unknowns only warm the others up
constexpr int MOM_CHUNK = 32, MOM_LANES = 128, MOM_WARM = 48, MOM_HALO = (MOM_WARM + MOM_CHUNK - 1) / MOM_CHUNK;
constexpr int MOM_TILE = (MOM_LANES - MOM_HALO) * MOM_CHUNK;  // unknowns a block delivers
}  // namespace

struct DD {
    double hi, lo;
};
// error-free transformations: no contraction of their additions
__device__ inline DD dd_fast2(double a, double b) {
#pragma clang fp contract(off)
    const double s = a + b;
    return {s, b - (s - a)};
}
__device__ inline DD dd_two(double a, double b) {
#pragma clang fp contract(off)
    const double s = a + b, bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
__device__ inline DD dd_add(DD a, DD b) {
#pragma clang fp contract(off)
    DD s = dd_two(a.hi, b.hi);
    const DD t = dd_two(a.lo, b.lo);
    s.lo += t.hi;
    s = dd_fast2(s.hi, s.lo);
    s.lo += t.lo;
    return dd_fast2(s.hi, s.lo);
}
__device__ inline DD dd_mul(DD a, DD b) {
#pragma clang fp contract(off)
    const double p = a.hi * b.hi;
    double e = fma(a.hi, b.hi, -p);
    e = fma(a.hi, b.lo, e);
    e = fma(a.lo, b.hi, e);
    return dd_fast2(p, e);
}
__device__ inline DD dd_div(DD a, double b) {
#pragma clang fp contract(off)
    const double q1 = a.hi / b;
    const double p = q1 * b;
    const double pe = fma(q1, b, -p);
    const double r = ((a.hi - p) - pe) + a.lo;
    return dd_fast2(q1, r / b);
}

// the series in double-double (see above); x ≥ 0
__device__ double mom_series_dd(double x, int nu, double m) {
#pragma clang fp contract(off)
    if (x == 0.0) return 0.0;
    const double p = x * x, pe = fma(x, x, -p);
    const DD z = dd_fast2(-0.5 * p, -0.5 * pe);  // −x²/2
    const double a = nu + m + 1.0;
    DD t = {1.0, 0.0}, s = {0.0, 0.0};
    for (int k = 0; k < 1000; ++k) {
        const DD term = dd_div(t, a + 2.0 * k);
        s = dd_add(s, term);
        if (k > 2 && fabs(term.hi) < 1e-33 * fabs(s.hi)) break;
        t = dd_div(dd_mul(t, z), (double)(k + 1) * (double)(2 * nu + 2 * k + 3));
    }
    double df = 1.0;
    for (int i = 3; i <= 2 * nu + 1; i += 2) df *= i;
    return pow(x, a) / df * (s.hi + s.lo);
}

// Si(x) = Σ_k (−1)^k x^{2k+1} / ((2k+1)(2k+1)!) in double-double (x ≤ 40)
__device__ double mom_si_dd(double x) {
#pragma clang fp contract(off)
    const double p = x * x, pe = fma(x, x, -p);
    const DD z = dd_fast2(-p, -pe);  // −x²
    DD t = {x, 0.0}, s = {0.0, 0.0};
    for (int k = 0; k < 1000; ++k) {
        const DD term = dd_div(t, 2.0 * k + 1.0);
        s = dd_add(s, term);
        if (k > 2 && fabs(term.hi) < 1e-33 * fabs(s.hi)) break;
        t = dd_div(dd_mul(t, z), (2.0 * k + 2.0) * (2.0 * k + 3.0));
    }
    return s.hi + s.lo;
}

// I_m(x) for integer 0 ≤ m ≤ 3, 1 ≤ ν ≤ 3 and 20 ≤ x < 40 by the identities above
__device__ double mom_closed(double x, int nu, int m) {
    double j[8];  // j_0 .. j_{ν+m+1} by upward recurrence (x > ν + m + 1)
    j[0] = sin(x) / x;
    j[1] = sin(x) / (x * x) - cos(x) / x;
    for (int l = 1; l <= nu + m; ++l) j[l + 1] = (2 * l + 1) / x * j[l] - j[l - 1];
    double a0 = mom_si_dd(x), a1 = 1.0 - j[0];  // ∫j_{L−1}, ∫j_L
    for (int l = 1; l < nu + m; ++l) {
        const double a2 = (l * a0 - (2 * l + 1) * j[l]) / (l + 1);
        a0 = a1;
        a1 = a2;
    }
    double I = nu + m == 0 ? a0 : a1;  // ∫_0^x j_{ν+m}
    double xk = 1.0;
    for (int k = 1; k <= m; ++k) {
        const int mu = nu + m - k;
        xk *= x;
        I = xk * j[mu + 1] - (k - mu - 2) * I;
    }
    return I;
}

__device__ double mom_asymp(double x, int nu, double m, double pref);

// a table node's value: the series below 20, the identities below 40, the asymptotic from 40 on
__device__ inline double mom_node_value(double x, int nu, int m, double pref) {
    return x < 20.0 ? mom_series_dd(x, nu, m) : (x < MOM_CUT ? mom_closed(x, nu, m) : mom_asymp(x, nu, m, pref));
}

// s⁽²⁾(t, α − ½, ν) (moments.jl:5-21)
__device__ inline double mom_s2(double t, double amh, double nu) {
    double s = 1.0, sk = 1.0;
    const double ti = 1.0 / t, ti2 = ti * ti, nu2 = nu * nu, am1 = amh - 0.5;
    for (int j = 0; j <= 20; ++j) {
        const double d = am1 - 2.0 * j;
        sk *= (nu2 - d * d) * ti2;
        s += sk;
        if (fabs(sk) < 1e-16 * fabs(s)) break;
    }
    return s * pow(t, amh) * sqrt(ti);
}

// sph_j_moment_asymp_prefactor (moments.jl:72-73): √(π/2) 2^{m−½} Γ((ν+m+1)/2) / Γ((ν−m+2)/2)
__host__ __device__ inline double mom_asymp_prefactor(int nu, double m) {
    const double nuh = nu + 0.5, al = m - 0.5;
    return exp(log(2.0) * al + lgamma((nuh + al + 1.0) / 2.0) - lgamma((nuh - al + 1.0) / 2.0)) * MOM_SQRT_HALF_PI;
}

// sph_j_moment_asymp (moments.jl:76-86), ν ≥ 1, x > ν: J_{ν±½}(x) = √(2x/π) j_ν, j_{ν−1}
// by upward recurrence from j_0, j_1
__device__ double mom_asymp(double x, int nu, double m, double pref) {
    double jm = sin(x) / x, jc = sin(x) / (x * x) - cos(x) / x;  // j_0, j_1
    for (int l = 1; l < nu; ++l) {
        const double jn = (2 * l + 1) / x * jc - jm;
        jm = jc;
        jc = jn;
    }
    const double c = sqrt(x) / MOM_SQRT_HALF_PI;
    return pref + x * MOM_SQRT_HALF_PI *
                      ((m + nu - 1.0) * (c * jc) * mom_s2(x, m - 2.0, nu - 0.5) - (c * jm) * mom_s2(x, m - 1.0, nu + 0.5));
}

// maclaurin_₁F₂ (weniger.jl:237-249) and sph_j_moment_maclaurin_₁F₂ (moments.jl:97-102), FP64
__device__ double mom_maclaurin64(double x, int nu, double m) {
    const double nup = nu + 1.5, a = (1.0 + m + nu) / 2.0, b1 = (3.0 + m + nu) / 2.0, b2 = nup, z = -x * x / 4.0;
    double S0 = 1.0, S1 = 1.0 + a * z / (b1 * b2);
    for (int j = 1; j < 100000; ++j) {
        const bool more = isfinite(S0) && isfinite(S1) &&
                          fabs(S0 - S1) > fmax(fabs(S0), fabs(S1)) * (10.0 * 2.220446049250313e-16);
        if (!(more || j <= 1)) break;
        double r = 1.0 / (j + 1.0);
        r *= a + j;
        r /= (b1 + j) * (b2 + j);
        const double Sn = S1 + (S1 - S0) * r * z;
        S0 = S1;
        S1 = Sn;
    }
    return (MOM_SQRT_HALF_PI / (m + nu + 1.0)) * exp((m + nu + 1.0) * log(x) - (nup - 1.0) * log(2.0) - lgamma(nup)) *
           S1;
}

struct MomTab {
    int nu, order, n;
    double xmin, xmax, dx;
    double pref[4];
    double* coef;  // [order][n + 2]
};

// node i of LinRange(x_min, x_max, n)
__host__ __device__ inline double mom_node(const MomTab& T, int i) {
    const double t = (double)i / (double)(T.n - 1);
    return (1.0 - t) * T.xmin + t * T.xmax;
}

// node values into rows 1..n of each coefficient column
// a lane per node and moment: the nodes below x = 40 (double-double series, closed
// forms) take a hundred times as long as the others, and with the three moments one
// after the other they alone were 101 us at 400 000 nodes; 57 now
__global__ void __launch_bounds__(256) k_moment_nodes(MomTab T, double* y) {
    const int m = blockIdx.y;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < T.n; i += gridDim.x * blockDim.x)
        y[(size_t)m * T.n + i] = mom_node_value(mom_node(T, i), T.nu, m, T.pref[m]);
}

// Line(OnGrid()) prefilter, the Thomas algorithm of the host tables' prefilter
// (d_q = (r_q − d_{q−1}) cp_q, cp_q = 1/(4 − cp_{q−1}), cp_0 = 1/4, r_q = 6 y_{q+1} −
// [q = 0] y_0 − [q = mm−1] y_{n−1}, then c_{q+2} = d_q − cp_q c_{q+3}).  The unknowns
// are c[2..n−1] (q = 0..mm−1 = n−3); c[1] = y_0 and c[n] = y_{n−1}.  cp_q is bitwise
// constant from q ≈ 20 on.
// A block brings its node values into LDS in whole lines; a lane takes MOM_CHUNK
// unknowns and starts its recurrence MOM_WARM of them early from zero (or at the true
// start), forward in the block's values, backward in its d.  One double of padding
// after every 32 keeps the lanes' strides off one bank.
// What bounds it is the chain of 160 steps, 300 blocks at 400 000 nodes x 3.  As two
// kernels of one lane per 128 unknowns straight from memory, every load and store a
// line of its own, it was 79 + 198 us; it is 27.
__global__ void __launch_bounds__(MOM_LANES) k_moment_prefilter(MomTab T, const double* yall) {
    constexpr int NV = MOM_LANES * MOM_CHUNK;
    __shared__ double v[(MOM_WARM + NV) / 32 * 33 + 33], cps[MOM_WARM];
    auto at = [](int i) { return i + (i >> 5); };
    const int mm = T.n - 2, tid = threadIdx.x, m = blockIdx.y;
    const int Q0 = blockIdx.x * MOM_TILE;          // the block's first unknown
    const double* y = yall + (size_t)m * T.n;
    double* c = T.coef + (size_t)m * (T.n + 2);
    // v[i]: r of unknown Q0 − MOM_WARM + i
    for (int i = tid; i < MOM_WARM + NV; i += MOM_LANES) {
        const int q = Q0 - MOM_WARM + i;
        double r = 0.0;
        if (q >= 0 && q < mm) {
            r = 6.0 * y[q + 1];
            if (q == 0) r -= y[0];
            if (q == mm - 1) r -= y[T.n - 1];
        }
        v[at(i)] = r;
    }
    if (tid == 0) {
        double cp = 0.25;
        for (int q = 0; q < MOM_WARM; ++q) {
            cps[q] = cp;
            cp = 1.0 / (4.0 - cp);
        }
    }
    __syncthreads();
    auto cp = [&](int q) { return cps[q < MOM_WARM ? (q < 0 ? 0 : q) : MOM_WARM - 1]; };
    const int q0 = Q0 + tid * MOM_CHUNK;
    const double cpw = cps[MOM_WARM - 1];
    const bool head = q0 < 2 * MOM_WARM;  // within reach of the first cp_q
    double d[MOM_CHUNK], dp = 0.0;
#pragma unroll 16
    for (int i = 0; i < MOM_WARM; ++i) {  // before unknown 0 the r are zero and so stays d
        const int q = q0 - MOM_WARM + i;
        dp = (v[at(tid * MOM_CHUNK + i)] - dp) * (head ? cp(q) : cpw);
    }
#pragma unroll
    for (int i = 0; i < MOM_CHUNK; ++i)
        d[i] = dp = (v[at(tid * MOM_CHUNK + MOM_WARM + i)] - dp) * (head ? cp(q0 + i) : cpw);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MOM_CHUNK; ++i) v[at(tid * MOM_CHUNK + i)] = d[i] = q0 + i < mm ? d[i] : 0.0;
    __syncthreads();
    double x = 0.0;  // past the last unknown d is zero and so stays c
    if (tid < MOM_LANES - MOM_HALO) {
#pragma unroll 16
        for (int i = MOM_WARM - 1; i >= 0; --i) {
            const int q = q0 + MOM_CHUNK + i;
            x = v[at((tid + 1) * MOM_CHUNK + i)] - (head ? cp(q) : cpw) * x;
        }
#pragma unroll
        for (int i = MOM_CHUNK - 1; i >= 0; --i) d[i] = x = d[i] - (head ? cp(q0 + i) : cpw) * x;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MOM_CHUNK; ++i) v[at(tid * MOM_CHUNK + i)] = d[i];
    __syncthreads();
    const int nq = mm - Q0 < MOM_TILE ? mm - Q0 : MOM_TILE;
    for (int i = tid; i < nq; i += MOM_LANES) c[Q0 + i + 2] = v[at(i)];
    if (tid == 0 && Q0 == 0) {
        c[1] = y[0];
        c[0] = 2.0 * y[0] - v[at(0)];
    }
    if (tid == 0 && Q0 + nq == mm) {
        c[T.n] = y[T.n - 1];
        c[T.n + 1] = 2.0 * y[T.n - 1] - v[at(nq - 1)];
    }
}

// MomentTable(x) (interpolator.jl:60-68)
__device__ inline void mom_eval(const MomTab& T, double x, double* out) {
    if (T.xmin <= x && x <= T.xmax) {
        const double tt = (x - T.xmin) / T.dx;
        int i = (int)floor(tt);
        i = i < 0 ? 0 : (i > T.n - 2 ? T.n - 2 : i);
        const double s = tt - i, r = 1.0 - s;
        const double w0 = r * r * r / 6.0, w1 = 2.0 / 3.0 - s * s + 0.5 * s * s * s,
                     w2 = 2.0 / 3.0 - r * r + 0.5 * r * r * r, w3 = s * s * s / 6.0;
        for (int m = 0; m < T.order; ++m) {
            const double* c = T.coef + (size_t)m * (T.n + 2) + i;
            out[m] = w0 * c[0] + w1 * c[1] + w2 * c[2] + w3 * c[3];
        }
    } else if (x > T.xmax) {
        for (int m = 0; m < T.order; ++m) out[m] = mom_asymp(x, T.nu, m, T.pref[m]);
    } else {
        for (int m = 0; m < T.order; ++m) out[m] = mom_maclaurin64(x, T.nu, m);
    }
}

__global__ void __launch_bounds__(256) k_moment_eval(MomTab T, const double* x, int nx, double* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nx) return;
    double v[4];
    mom_eval(T, x[i], v);
    for (int m = 0; m < T.order; ++m) out[(size_t)i * T.order + m] = v[m];
}

// integrate_sph_bessel_filon (integrator.jl:5-18): the quadratic through f, f′,
// f″ at a against j_ν(kt) over (a, b); Ia = the moments at ka
__device__ inline double mom_filon(double f, double fp, double fpp, double k, double a, const double* Ia,
                                   const double* Ib) {
    const double c2 = fpp / 2.0, afpp = a * fpp, c1 = fp - afpp, c0 = f - a * (fp - afpp / 2.0);
    const double ki = 1.0 / k, ki2 = ki * ki, ki3 = ki2 * ki;
    return (c0 * ki) * (Ib[0] - Ia[0]) + (c1 * ki2) * (Ib[1] - Ia[1]) + (c2 * ki3) * (Ib[2] - Ia[2]);
}

__global__ void __launch_bounds__(256) k_filon(MomTab T, const double* f, const double* fp, const double* fpp,
                                              const double* k, const double* a, const double* b, int n, double* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double Ia[4], Ib[4];
    mom_eval(T, k[i] * b[i], Ib);
    mom_eval(T, k[i] * a[i], Ia);
    out[i] = mom_filon(f[i], fp[i], fpp[i], k[i], a[i], Ia, Ib);
}

// Σ_i Filon over (t_i, t_{i+1}) for each k (the loop form, integrator.jl:20-38):
// one block per k, lane l takes intervals l, l + blockDim.x, …, each reusing
// nothing across lanes (I(k t_i) is evaluated at both ends); the lanes' sums
// are added in a fixed order.  Latency of the table reads: with one wavefront, 16
// steps of two reads in turn, 1001 t x 700 k were 68 us; with four they are 40.  Up to
// 256 intervals take only the wavefronts that have one (20 t x 5000 k: a call with four
// is 83 us, with one 73).
constexpr int FILON_THREADS = 256;
__global__ void __launch_bounds__(FILON_THREADS) k_filon_sum(MomTab T, const double* t, const double* f,
                                                             const double* fp, const double* fpp, int nt,
                                                             const double* ks, double* out) {
    __shared__ double part[FILON_THREADS / WAVE];
    const double k = ks[blockIdx.x];
    double s = 0.0;
    for (int i = threadIdx.x; i + 1 < nt; i += blockDim.x) {
        double Ia[4], Ib[4];
        mom_eval(T, k * t[i + 1], Ib);
        mom_eval(T, k * t[i], Ia);
        s += mom_filon(f[i], fp[i], fpp[i], k, t[i], Ia, Ib);
    }
    s = wave_sum(s);
    if (threadIdx.x % WAVE == 0) part[threadIdx.x / WAVE] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)blockDim.x / WAVE; ++w) s += part[w];
        out[blockIdx.x] = s;
    }
}

// the moment functions themselves, per point: method 0 asymptotic, 1 FP64
// series, 2 a table node's method (x < 40: double-double series, identities)
__global__ void __launch_bounds__(256) k_sph_moments(int method, const double* x, const int* nu, const double* m, int n,
                                                    double* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double xi = x[i], mi = m[i];
    const int v = nu[i];
    out[i] = method == 0 ? mom_asymp(xi, v, mi, mom_asymp_prefactor(v, mi))
                         : (method == 1 ? mom_maclaurin64(xi, v, mi)
                                        : (xi < 20.0 ? mom_series_dd(xi, v, mi) : mom_closed(xi, v, (int)mi)));
}

struct bolt_moment_table {
    int device = 0;
    hipStream_t stream = nullptr;
    MomTab T{};
};

namespace {
// a host array of count doubles (or ints) on the device for one call
template <class V>
struct Scratch {
    V* p = nullptr;
    ~Scratch() { if (p) (void)hipFree(p); }
    hipError_t up(const V* h, size_t count, hipStream_t st) {
        hipError_t e = hipMalloc((void**)&p, sizeof(V) * (count ? count : 1));
        if (e != hipSuccess) return e;
        return count ? hipMemcpyAsync(p, h, sizeof(V) * count, hipMemcpyHostToDevice, st) : hipSuccess;
    }
    hipError_t alloc(size_t count) { return hipMalloc((void**)&p, sizeof(V) * (count ? count : 1)); }
};
}  // namespace

extern "C" {

int bolt_moment_table_create(bolt_ctx* ctx, int nu, int order, double x_min, double x_max, int n,
                             bolt_moment_table** out) {
    if (!ctx || !out) return set_error(BOLT_E_ARG, "bolt_moment_table_create: NULL argument");
    if (nu < 1 || nu > 3) return set_error(BOLT_E_ARG, "bolt_moment_table_create: tables hold ν = 1, 2 or 3");
    if (order < 3 || order > 4) return set_error(BOLT_E_ARG, "bolt_moment_table_create: order is 3 or 4");
    if (n < 4 || n > (1 << 28)) return set_error(BOLT_E_ARG, "bolt_moment_table_create: need 4 <= n <= 2^28 nodes");
    if (!(x_min >= 0.0) || !(x_max > x_min) || !std::isfinite(x_max))
        return set_error(BOLT_E_ARG, "bolt_moment_table_create: need 0 <= x_min < x_max");
    HIPCHK(hipSetDevice(ctx->device));
    auto tab = std::make_unique<bolt_moment_table>();
    tab->device = ctx->device;
    MomTab& T = tab->T;
    T.nu = nu; T.order = order; T.n = n; T.xmin = x_min; T.xmax = x_max;
    T.dx = (x_max - x_min) / (n - 1);
    for (int m = 0; m < 4; ++m) T.pref[m] = mom_asymp_prefactor(nu, m);
    HIPCHK(hipStreamCreateWithFlags(&tab->stream, hipStreamNonBlocking));
    if (hipMalloc((void**)&T.coef, sizeof(double) * (size_t)order * (n + 2)) != hipSuccess) {
        (void)hipStreamDestroy(tab->stream);
        return set_error(BOLT_E_NOMEM, "bolt_moment_table_create: coefficients");
    }
    Scratch<double> work;
    if (work.alloc((size_t)order * n) != hipSuccess) {
        (void)hipFree(T.coef);
        (void)hipStreamDestroy(tab->stream);
        return set_error(BOLT_E_NOMEM, "bolt_moment_table_create: work space");
    }
    hipStream_t st = tab->stream;
    const int nb = std::min((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_moment_nodes, dim3(nb, order), dim3(256), 0, st, T, work.p);
    hipLaunchKernelGGL(k_moment_prefilter, dim3((n - 2 + MOM_TILE - 1) / MOM_TILE, order), dim3(MOM_LANES), 0, st, T,
                       (const double*)work.p);
    const hipError_t e1 = hipGetLastError(), e2 = hipStreamSynchronize(st);
    if (e1 != hipSuccess || e2 != hipSuccess) {
        (void)hipFree(T.coef);
        (void)hipStreamDestroy(tab->stream);
        return set_error(BOLT_E_DEVICE, "bolt_moment_table_create: kernel failed");
    }
    *out = tab.release();
    return BOLT_OK;
}

int bolt_moment_table_destroy(bolt_moment_table* tab) {
    if (!tab) return BOLT_OK;
    (void)hipSetDevice(tab->device);
    if (tab->stream) (void)hipStreamSynchronize(tab->stream);
    if (tab->T.coef) (void)hipFree(tab->T.coef);
    if (tab->stream) (void)hipStreamDestroy(tab->stream);
    delete tab;
    return BOLT_OK;
}

int bolt_moment_table_coefficients(bolt_moment_table* tab, double* out) {
    if (!tab || !out) return set_error(BOLT_E_ARG, "bolt_moment_table_coefficients: NULL argument");
    HIPCHK(hipSetDevice(tab->device));
    HIPCHK(hipMemcpyAsync(out, tab->T.coef, sizeof(double) * (size_t)tab->T.order * (tab->T.n + 2),
                          hipMemcpyDeviceToHost, tab->stream));
    HIPCHK(hipStreamSynchronize(tab->stream));
    return BOLT_OK;
}

int bolt_moment_table_eval(bolt_moment_table* tab, const double* x, int nx, double* out) {
    if (!tab || (nx > 0 && (!x || !out)) || nx < 0) return set_error(BOLT_E_ARG, "bolt_moment_table_eval: bad argument");
    if (nx == 0) return BOLT_OK;
    HIPCHK(hipSetDevice(tab->device));
    hipStream_t st = tab->stream;
    Scratch<double> dx, dout;
    HIPCHK(dx.up(x, nx, st));
    HIPCHK(dout.alloc((size_t)nx * tab->T.order));
    hipLaunchKernelGGL(k_moment_eval, dim3((nx + 255) / 256), dim3(256), 0, st, tab->T, (const double*)dx.p, nx, dout.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, dout.p, sizeof(double) * (size_t)nx * tab->T.order, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return BOLT_OK;
}

int bolt_filon(bolt_moment_table* tab, const double* f, const double* fp, const double* fpp, const double* k,
               const double* a, const double* b, int n, double* out) {
    if (!tab || n < 0 || (n > 0 && (!f || !fp || !fpp || !k || !a || !b || !out)))
        return set_error(BOLT_E_ARG, "bolt_filon: bad argument");
    if (n == 0) return BOLT_OK;
    for (int i = 0; i < n; ++i)
        if (!(k[i] > 0.0)) return set_error(BOLT_E_ARG, "bolt_filon: k must be positive");
    HIPCHK(hipSetDevice(tab->device));
    hipStream_t st = tab->stream;
    Scratch<double> df, dfp, dfpp, dk, da, db, dout;
    HIPCHK(df.up(f, n, st)); HIPCHK(dfp.up(fp, n, st)); HIPCHK(dfpp.up(fpp, n, st));
    HIPCHK(dk.up(k, n, st)); HIPCHK(da.up(a, n, st)); HIPCHK(db.up(b, n, st));
    HIPCHK(dout.alloc(n));
    hipLaunchKernelGGL(k_filon, dim3((n + 255) / 256), dim3(256), 0, st, tab->T, (const double*)df.p,
                       (const double*)dfp.p, (const double*)dfpp.p, (const double*)dk.p, (const double*)da.p,
                       (const double*)db.p, n, dout.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, dout.p, sizeof(double) * n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return BOLT_OK;
}

int bolt_filon_sum(bolt_moment_table* tab, const double* t, const double* f, const double* fp, const double* fpp,
                   int nt, const double* k, int nk, double* out) {
    if (!tab || nt < 2 || nk < 0 || !t || !f || !fp || !fpp || (nk > 0 && (!k || !out)))
        return set_error(BOLT_E_ARG, "bolt_filon_sum: bad argument");
    if (nk == 0) return BOLT_OK;
    for (int i = 0; i < nk; ++i)
        if (!(k[i] > 0.0)) return set_error(BOLT_E_ARG, "bolt_filon_sum: k must be positive");
    HIPCHK(hipSetDevice(tab->device));
    hipStream_t st = tab->stream;
    Scratch<double> dt, df, dfp, dfpp, dk, dout;
    HIPCHK(dt.up(t, nt, st)); HIPCHK(df.up(f, nt, st)); HIPCHK(dfp.up(fp, nt, st)); HIPCHK(dfpp.up(fpp, nt, st));
    HIPCHK(dk.up(k, nk, st));
    HIPCHK(dout.alloc(nk));
    const int nthr = nt > FILON_THREADS ? FILON_THREADS : (nt + WAVE - 2) / WAVE * WAVE;
    hipLaunchKernelGGL(k_filon_sum, dim3(nk), dim3(nthr), 0, st, tab->T, (const double*)dt.p, (const double*)df.p,
                       (const double*)dfp.p, (const double*)dfpp.p, nt, (const double*)dk.p, dout.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, dout.p, sizeof(double) * nk, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return BOLT_OK;
}

int bolt_sph_moments(bolt_ctx* ctx, int method, const double* x, const int* nu, const double* m, int n, double* out) {
    if (!ctx || n < 0 || (n > 0 && (!x || !nu || !m || !out)) || method < 0 || method > 2)
        return set_error(BOLT_E_ARG, "bolt_sph_moments: bad argument");
    for (int i = 0; i < n; ++i) {
        if (nu[i] < 1 || nu[i] > 64) return set_error(BOLT_E_ARG, "bolt_sph_moments: need 1 <= ν <= 64");
        if (method == 2 && !(x[i] < 20.0) &&
            (x[i] >= MOM_CUT || nu[i] > 3 || m[i] != std::floor(m[i]) || m[i] < 0.0 || m[i] > 3.0))
            return set_error(BOLT_E_ARG,
                             "bolt_sph_moments: method 2 from x = 20 to 40 takes integer 0 <= m <= 3, ν <= 3");
        if (!(x[i] >= 0.0) || !(m[i] > -nu[i] - 1.0)) return set_error(BOLT_E_ARG, "bolt_sph_moments: need x >= 0, m > -ν-1");
        if (method == 0 && !(x[i] > nu[i])) return set_error(BOLT_E_ARG, "bolt_sph_moments: the asymptotic needs x > ν");
    }
    if (n == 0) return BOLT_OK;
    HIPCHK(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    Scratch<double> dx, dm, dout;
    Scratch<int> dnu;
    HIPCHK(dx.up(x, n, st)); HIPCHK(dm.up(m, n, st)); HIPCHK(dnu.up(nu, n, st));
    HIPCHK(dout.alloc(n));
    hipLaunchKernelGGL(k_sph_moments, dim3((n + 255) / 256), dim3(256), 0, st, method, (const double*)dx.p,
                       (const int*)dnu.p, (const double*)dm.p, n, dout.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, dout.p, sizeof(double) * n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return BOLT_OK;
}

}  // extern "C"

// ============================================================================
// Background, RECFAST and ionization tables on the device: bolt_host_tables'
// algorithm (src/background.jl:32-128, src/ionization/recfast.jl:22-536,
// 674-726, ionization.jl:95-137) with one wavefront per cosmology, so a batch
// of cosmologies builds its tables side by side.  The node-wise work (ρ₀ℳ, ℋ,
// η quadratures, τ′, g̃, c_s²) and the spline derivatives run across the
// wavefront's lanes; the spline prefilters run one table per lane; the
// RECFAST solve (two root finds, the He stage, the H + He stage, then the
// reionized matter temperature from z = 50) is one Dormand–Prince 5(4)
// integration by the wavefront, which evaluates each rate function's
// transcendental terms on separate lanes; the same steps and tolerances as
// the host's.  The
// arithmetic is the host's, uncontracted; only the transcendental functions
// differ (the device's math library), which moves the adaptive steps and
// leaves differences at the level of the ODE tolerance (1e-11).
// ============================================================================
namespace gbg {

// RECFAST's constants of one cosmology (the host RECFAST's constructor)
struct RfC {
    double Yp, OmegaB, HO, Tnow, mu_H, mu_T, fHe, Nnow;
};
struct Par {  // one cosmology: its parameters and Background's and RECFAST's constants (from the host)
    double h, Omega_r, Omega_b, Omega_c, N_nu, Sum_m_nu, Y_p;
    double H0, rho_crit, Omega_L, rad_fac, Tnu, logqmin, logqmax;
    RfC rc;
};
struct Args {
    const Par* par;
    int nx, nq;
    double x0, x1, dx;
    const double* xq;  // [nq] Gauss–Legendre nodes and weights
    const double* wq;
    double H0_conv, K_conv, m_H, sigma_T;
    double* coef;   // [ncosmo][BOLT_NTAB][nx + 2]
    double* scal;   // [ncosmo][BOLT_NSCAL]
    double* work;   // [ncosmo][WK][nx]
    int* status;    // [ncosmo]: 0, or 1 if the RECFAST integration ran out of steps
};
constexpr int WK = 12;

__device__ inline double node(const Args& A, int j) { return (A.x0 * (A.nx - 1 - j) + A.x1 * j) / (A.nx - 1); }

// CosmoT (host_tables.cpp; background.jl:21-77)
__device__ inline double f0(const Par& P, double q) {
#pragma clang fp contract(off)
    return 2.0 / pow(2.0 * M_PI, 3) / (exp(q / P.Tnu) + 1.0);
}
__device__ inline double from_ui(double x, double lo, double hi) {
#pragma clang fp contract(off)
    return lo + (hi - lo) / 2.0 * (x + 1.0);
}
__device__ inline double to_ui(double lq, double lo, double hi) {
#pragma clang fp contract(off)
    return -1.0 + 2.0 / (hi - lo) * (lq - lo);
}
__device__ inline double dxdq(double q, double lo, double hi) {
#pragma clang fp contract(off)
    return (1.0 + to_ui(1.0 + lo, lo, hi)) / (q * log(10.0));
}
__device__ inline double xq2q(double x, double lo, double hi) { return pow(10.0, from_ui(x, lo, hi)); }
__device__ double rho0_massive(const Args& A, const Par& P, double a) {
#pragma clang fp contract(off)
    const double m = P.Sum_m_nu;
    double s = 0.0;
    for (int i = 0; i < A.nq; ++i) {
        const double q = xq2q(A.xq[i], P.logqmin, P.logqmax);
        const double eps = sqrt(q * q + (a * m) * (a * m));
        const double I = q * q * eps * f0(P, q) / dxdq(q, P.logqmin, P.logqmax);
        s += I * A.wq[i];
    }
    return 4.0 * M_PI * pow(a, -4) * s;
}
__device__ double H_a(const Args& A, const Par& P, double a) {
#pragma clang fp contract(off)
    const double rho_nu = rho0_massive(A, P, a);
    return P.H0 * sqrt((P.Omega_c + P.Omega_b) * pow(a, -3) + rho_nu / P.rho_crit +
                       P.Omega_r * pow(a, -4) * P.rad_fac + P.Omega_L);
}
__device__ inline double Hc_a(const Args& A, const Par& P, double a) { return a * H_a(A, P, a); }
__device__ double eta(const Args& A, const Par& P, double x) {
#pragma clang fp contract(off)
    const double lo = -13.75, hi = log10(exp(x));
    double s = 0.0;
    for (int i = 0; i < A.nq; ++i) {
        const double ay = xq2q(A.xq[i], lo, hi);
        s += 1.0 / (ay * Hc_a(A, P, ay)) / dxdq(ay, lo, hi) * A.wq[i];
    }
    return s;
}

// uniform cubic B-spline with Line(OnGrid()) ends (util.jl:11-13): the host's
// prefilter_t, eval_t and node_derivatives
__device__ void prefilter(const double* y, int n, double* c) {
#pragma clang fp contract(off)
    c[1] = y[0];
    c[n] = y[n - 1];
    const int m = n - 2;
    // forward elimination into c[2 .. n-1]; cp_i = 1/(4 − cp_{i−1}) is bitwise
    // constant from i ≈ 20 on, so the backward pass recomputes only its first terms
    double cp = 0.25, dprev = 0.0;
    for (int i = 0; i < m; ++i) {
        double d = 6.0 * y[i + 1];
        if (i == 0) d -= c[1];
        if (i == m - 1) d -= c[n];
        if (i == 0) {
            d = d / 4.0;
        } else {
            const double den = 4.0 - cp;
            cp = 1.0 / den;
            d = (d - dprev) / den;
        }
        c[i + 2] = d;
        dprev = d;
    }
    double cpc = 0.25;
    for (int i = 1; i <= 64; ++i) cpc = 1.0 / (4.0 - cpc);  // the converged multiplier
    for (int i = m - 2; i >= 0; --i) {
        double cpi = cpc;
        if (i < 64) {
            cpi = 0.25;
            for (int k = 1; k <= i; ++k) cpi = 1.0 / (4.0 - cpi);
        }
        c[i + 2] -= cpi * c[i + 3];
    }
    c[0] = 2.0 * c[1] - c[2];
    c[n + 1] = 2.0 * c[n] - c[n - 1];
}
__device__ double spl(const double* c, int n, double x0, double dx, double x, int deriv) {
#pragma clang fp contract(off)
    const double t = (x - x0) / dx;
    int i = (int)floor(t);
    if (i < 0) i = 0;
    if (i > n - 2) i = n - 2;
    const double s = t - i, r = 1.0 - s;
    const double* p = c + i;
    if (deriv == 0) {
        const double w0 = r * r * r / 6.0, w1 = 2.0 / 3.0 - s * s + 0.5 * s * s * s,
                     w2 = 2.0 / 3.0 - r * r + 0.5 * r * r * r, w3 = s * s * s / 6.0;
        return w0 * p[0] + w1 * p[1] + w2 * p[2] + w3 * p[3];
    } else if (deriv == 1) {
        const double w0 = -0.5 * r * r, w1 = -2.0 * s + 1.5 * s * s, w2 = 2.0 * r - 1.5 * r * r, w3 = 0.5 * s * s;
        return (w0 * p[0] + w1 * p[1] + w2 * p[2] + w3 * p[3]) / dx;
    }
    const double w0 = r, w1 = -2.0 + 3.0 * s, w2 = -2.0 + 3.0 * r, w3 = s;
    return (w0 * p[0] + w1 * p[1] + w2 * p[2] + w3 * p[3]) / (dx * dx);
}
__device__ inline double node_deriv(const double* c, int j, double dx, int deriv) {
#pragma clang fp contract(off)
    const double* p = c + j;
    return deriv == 1 ? (p[2] - p[0]) / (2.0 * dx) : (p[0] - 2.0 * p[1] + p[2]) / (dx * dx);
}

// RECFAST (recfast.jl:22-121 constants, 156-310 rates, 363-427): the literal
// constants at compile time, the derived ones in constant memory (computed on
// the host with the host RECFAST's formulas), the cosmology's own in RfC
namespace rfc {
constexpr double C = 2.99792458e8, k_B = 1.380658e-23, h_P = 6.6260755e-34, m_e = 9.1093897e-31,
                 m_H = 1.673575e-27, not4 = 3.9715e0, sigma = 6.6524616e-29, a = 7.565914e-16, G = 6.6742e-11;
constexpr double Lambda = 8.2245809e0, Lambda_He = 51.3e0, L_H_ion = 1.096787737e7, L_H_alpha = 8.225916453e6,
                 L_He1_ion = 1.98310772e7, L_He2_ion = 4.389088863e7, L_He_2s = 1.66277434e7, L_He_2p = 1.71134891e7;
constexpr double A2P_s = 1.798287e9, A2P_t = 177.58e0, L_He_2Pt = 1.690871466e7, L_He_2St = 1.5985597526e7,
                 L_He2St_ion = 3.8454693845e6, sigma_He_2Ps = 1.436289e-22, sigma_He_2Pt = 1.484872e-22;
constexpr double AGauss1 = -0.14e0, AGauss2 = 0.079e0, zGauss1 = 7.28e0, zGauss2 = 6.73e0, wGauss1 = 0.18e0,
                 wGauss2 = 0.33e0;
constexpr double a_PPB = 4.309, b_PPB = -0.6166, c_PPB = 0.6703, d_PPB = 0.5300;
constexpr double b_VF = 0.711, b_trip = 0.761, H_frac = 1e-3, fu = 1.125, b_He = 0.86;
constexpr int Heswitch = 6;
}  // namespace rfc
struct RfK {
    double a_VF, T_0, T_1, a_trip, Lalpha, Lalpha_He, CDB, CDB_He, CB1, CB1_He1, CB1_He2, CR, CK, CK_He, CL, CL_He,
        CT, Bfact;
    // folded products for the rates: 1/T_0, 1/T_1, 2k_B/(m_H·not4·C²) (the Doppler width's),
    // 1/(8π L_He_2Pt³), and γ_2P's constant factors 3A2P·C²/(√π σ 8π (C L)²)
    double iT_0, iT_1, dop, itau_t, g2Ps, g2Pt;
};
__constant__ RfK c_rfk;

// one spline table's view for the rates: ℋ and ℋ′ coefficients
struct HcTab {
    const double* hc;
    const double* hcp;
    int nx;
    double x0, dx, iH0_conv;
};

struct R3 {
    double f1, f2, f3;
};

// ion_recfast (recfast.jl:156-310), evaluated by a whole wavefront (every
// lane calls it with the same arguments and receives the same result): its
// independent transcendental terms are one log, one sqrt, one pow and one
// exp across the lanes, lane i holding the i-th term's argument, then one
// exp and one pow more for the four terms that need ℋ and n_He; every lane
// combines them.  The formulas are the host's; divisions by T_mat, ℋ, 1+z and
// x are multiplications by their reciprocals, and products of constants are
// folded (constant memory, computed on the host), which moves results by
// ulps.  One out-of-line copy serves every stage of the integration.
__device__ __attribute__((noinline)) R3 rf_rates(double x_H, double x_He, double Tmat, double z, RfC P, HcTab H) {
    using namespace rfc;
    const RfK& K0 = c_rfk;
    const double fHe = P.fHe, Nnow = P.Nnow, Tnow = P.Tnow;
    const int L = threadIdx.x & (WAVE - 1);
    double f1 = 0.0, f2 = 0.0, f3 = 0.0;
    const double x = x_H + fHe * x_He;
    const double zp1 = 1.0 + z, i1z = 1.0 / zp1, iT = 1.0 / Tmat;
    const double Trad = Tnow * zp1;
    // lane 0: x_a = log a; lane 1: log(1 + z)
    const double lg = log(L == 0 ? i1z : zp1);
    const double x_a = readlane64(lg, 0), lz = readlane64(lg, 1);
    const double sq = sqrt(Tmat * (L == 0 ? K0.iT_0 : (L == 1 ? K0.iT_1 : K0.dop)));
    const double sq_0 = readlane64(sq, 0), sq_1 = readlane64(sq, 1), dsq = readlane64(sq, 2);
    double pb = 1.0, pe = 1.0;
    switch (L) {
        case 0: pb = zp1; pe = 3; break;
        case 1: pb = Tmat * 1e-4; pe = b_PPB; break;
        case 2: pb = Tmat * 1e-4; pe = d_PPB; break;
        case 3: pb = K0.CR * Tmat; pe = 1.5; break;
        case 4: pb = 1.0 + sq_0; pe = 1 - b_VF; break;
        case 5: pb = 1.0 + sq_1; pe = 1 + b_VF; break;
        case 6: pb = 1.0 + sq_0; pe = 1 - b_trip; break;
        case 7: pb = 1.0 + sq_1; pe = 1 + b_trip; break;
        case 8: pb = Trad; pe = 4; break;
        case 9: pb = zp1; pe = 1.5; break;
        case 10: pb = Trad; pe = 3; break;
        case 11: pb = (lz - zGauss1) * (1.0 / wGauss1); pe = 2; break;
        case 12: pb = (lz - zGauss2) * (1.0 / wGauss2); pe = 2; break;
        default: break;
    }
    const double pw = pow(pb, pe);
    const double p13 = readlane64(pw, 0), pT_b = readlane64(pw, 1), pT_d = readlane64(pw, 2);
    const double pCR = readlane64(pw, 3), pVF0 = readlane64(pw, 4), pVF1 = readlane64(pw, 5);
    const double pTr0 = readlane64(pw, 6), pTr1 = readlane64(pw, 7), pTrad4 = readlane64(pw, 8);
    const double pz15 = readlane64(pw, 9), pTrad3 = readlane64(pw, 10);
    const double pG1 = readlane64(pw, 11), pG2 = readlane64(pw, 12);
    // exp arguments: −E/T for the Boltzmann factors (E/k_B folded), the two Gaussians
    constexpr double kTrip = h_P * C * L_He2St_ion / k_B, kPSt = h_P * C * (L_He_2Pt - L_He_2St) / k_B,
                     k2St = h_P * C * L_He_2St / k_B;
    double ea = 0.0;
    switch (L) {
        case 0: ea = -K0.CDB * iT; break;
        case 1: ea = -K0.CDB_He * iT; break;
        case 2: ea = fmin(K0.Bfact * iT, 680.); break;
        case 3: ea = -pG1; break;
        case 4: ea = -pG2; break;
        case 5: ea = -kTrip * iT; break;
        case 6: ea = -kPSt * iT; break;
        case 7: ea = -K0.CL * iT; break;
        case 8: ea = -K0.CL_He * iT; break;
        case 9: ea = -k2St * iT; break;
        default: break;
    }
    const double ex = exp(ea);
    const double eCDB = readlane64(ex, 0), eCDBHe = readlane64(ex, 1), He_Boltz = readlane64(ex, 2);
    const double eG1 = readlane64(ex, 3), eG2 = readlane64(ex, 4), eTrip = readlane64(ex, 5);
    const double ePSt = readlane64(ex, 6), eCL = readlane64(ex, 7), eCLHe = readlane64(ex, 8);
    const double e2St = readlane64(ex, 9);
    const double hc = spl(H.hc, H.nx, H.x0, H.dx, x_a, 0), hcp = spl(H.hcp, H.nx, H.x0, H.dx, x_a, 0);
    const double n = Nnow * p13;
    const double n_He = fHe * Nnow * p13;
    const double Hz = hc * zp1 * H.iH0_conv, iHz = 1.0 / Hz;
    const double dHdz = (-hcp + hc) * H.iH0_conv;
    const double Rdown = 1e-19 * a_PPB * pT_b / (1. + c_PPB * pT_d);
    const double Rup = Rdown * pCR * eCDB;
    const double Rdown_He = K0.a_VF / (sq_0 * pVF0 * pVF1);
    const double Rup_He = 4. * (Rdown_He * pCR * eCDBHe);
    const double K = K0.CK * iHz * (1.0 + AGauss1 * eG1 + AGauss2 * eG2);
    const double Rdown_trip = K0.a_trip / (sq_0 * pTr0 * pTr1);
    const double Rup_trip = Rdown_trip * eTrip * pCR * (4.0 / 3.0);
    const int Heflag = ((x_He < 5.e-9) || (x_He > 0.980)) ? 0 : Heswitch;
    // second round: the terms that need n_He and ℋ
    const double tauHe_s = A2P_s * K0.CK_He * 3 * n_He * (1.0 - x_He) * iHz;
    const double tauHe_t = A2P_t * n_He * (1. - x_He) * 3 * iHz * K0.itau_t;
    const double gamma_2Ps = K0.g2Ps * fHe * (1.0 - x_He) / (dsq * (1.0 - x_H));
    const double gamma_2Pt = K0.g2Pt * fHe * (1.0 - x_He) / (dsq * (1.0 - x_H));
    // lanes 0, 1: exp(−τ_s), exp(−τ_t); lanes 2, 3: γ_2Ps^b_He, γ_2Pt^0.9
    const double e2 = exp(L == 0 ? -tauHe_s : -tauHe_t);
    const double p2 = pow(L == 2 ? gamma_2Ps : gamma_2Pt, L == 2 ? b_He : 0.9);
    const double etHs = readlane64(e2, 0), etHt = readlane64(e2, 1), pgPs = readlane64(p2, 2), pgPt = readlane64(p2, 3);
    double K_He, CfHe_t = 0.0;
    const double omHe = 1.0 - x_He, omH = 1.0 - x_H;
    if (Heflag == 0) {
        K_He = K0.CK_He * iHz;
    } else {
        const double pHe_s = (1.0 - etHs) / tauHe_s;
        K_He = 1.0 / (A2P_s * pHe_s * 3 * n_He * omHe);
        if (((Heflag == 2) || (Heflag >= 5)) && (x_H < 0.9999999)) {
            const double AHcon = A2P_s / (1.0 + 0.36 * pgPs);
            K_He = 1.0 / ((A2P_s * pHe_s + AHcon) * 3 * n_He * omHe);
        }
        if (Heflag >= 3) {
            const double pHe_t = (1.0 - etHt) / tauHe_t;
            if ((Heflag == 3) || (Heflag == 5) || (x_H > 0.99999)) {
                CfHe_t = A2P_t * pHe_t * ePSt;
            } else {
                const double AHcon = A2P_t / (1.0 + 0.66 * pgPt) * (1.0 / 3);
                CfHe_t = (A2P_t * pHe_t + AHcon) * ePSt;
            }
            CfHe_t = CfHe_t / (Rup_trip + CfHe_t);
        }
    }
    const double ix = 1.0 / x;
    const double timeTh = (1.0 + x + fHe) * ix / (K0.CT * pTrad4);
    const double timeH = 2.0 / (3 * P.HO * pz15);
    const double iHz1z = iHz * i1z;  // 1 / (ℋ(1 + z)), in the rates' units
    if (x_H > 0.99) {
        f1 = 0.;
    } else if (x_H > 0.985) {
        f1 = (x * x_H * n * Rdown - Rup * omH * eCL) * iHz1z;
    } else {
        const double KLn = K * Lambda * n * omH;
        f1 = ((x * x_H * n * Rdown - Rup * omH * eCL) * (1.0 + KLn)) * iHz1z /
             ((1.0 / fu) * (1.0 + KLn) + K * Rup * n * omH);
    }
    if (x_He < 1e-15) {
        f2 = 0.;
    } else {
        const double KB = K_He * n_He * omHe * He_Boltz;
        f2 = ((x * x_He * n * Rdown_He - Rup_He * omHe * eCLHe) * (1.0 + KB * Lambda_He)) * iHz1z /
             (1.0 + KB * (Lambda_He + Rup_He));
        if (Heflag >= 3) f2 = f2 + (x * x_He * n * Rdown_trip - omHe * 3 * Rup_trip * e2St) * CfHe_t * iHz1z;
    }
    if (timeTh < H_frac * timeH) {
        const double epsilon = Hz * (1.0 + x + fHe) * ix / (K0.CT * pTrad3);
        f3 = Tnow + epsilon * ((1.0 + fHe) / (1.0 + fHe + x)) * ((f1 + fHe * f2) * ix) - epsilon * dHdz * iHz +
             3 * epsilon * i1z;
    } else {
        f3 = K0.CT * pTrad4 * x / (1.0 + x + fHe) * (Tmat - Trad) * iHz1z + 2 * Tmat * i1z;
    }
    return {f1, f2, f3};
}
__device__ inline double saha_rhs(double z, double cb, const RfC& P) {
#pragma clang fp contract(off)
    return exp(1.5 * log(c_rfk.CR * P.Tnow / (1.0 + z)) - cb / (P.Tnow * (1.0 + z))) / P.Nnow;
}
__device__ inline double he_saha_x0(double z, const RfC& P) {
#pragma clang fp contract(off)
    const double rhs = saha_rhs(z, c_rfk.CB1_He1, P) * 4;
    return 0.5 * (sqrt((rhs - 1.0) * (rhs - 1.0) + 4 * (1.0 + P.fHe) * rhs) - (rhs - 1.0));
}
__device__ inline double x_H0_saha(double z, const RfC& P) {
#pragma clang fp contract(off)
    const double rhs = saha_rhs(z, c_rfk.CB1, P);
    return 0.5 * (sqrt(rhs * rhs + 4 * rhs) - rhs);
}
template <class F>
__device__ double rf_bisect(F&& g, double lo, double hi) {
    double flo = g(lo);
    for (int it = 0; it < 200; ++it) {
        const double mid = 0.5 * (lo + hi);
        const double fm = g(mid);
        if ((fm > 0) == (flo > 0)) { lo = mid; flo = fm; } else { hi = mid; }
        if (fabs(hi - lo) <= 1e-13 * fmax(1.0, fabs(mid))) break;
    }
    return 0.5 * (lo + hi);
}
__device__ inline double xe_saha_early(double z, const RfC& P) {
#pragma clang fp contract(off)
    const double fHe = P.fHe;
    if (z > 8000.) return 1.0 + 2 * fHe;
    if (z > 5000.) {
        const double rhs = saha_rhs(z, c_rfk.CB1_He2, P);
        return 0.5 * (sqrt((rhs - 1.0 - fHe) * (rhs - 1.0 - fHe) + 4 * (1.0 + 2 * fHe) * rhs) - (rhs - 1.0 - fHe));
    }
    if (z > 3500.) return 1.0 + fHe;
    return he_saha_x0(z, P);
}

// dopri_outputs (host_tables.cpp): explicit Dormand–Prince 5(4) with step
// clipping onto the requested outputs zout(0..nout-1); out(i, y) receives them.
// Returns false if 500,000 steps ran out (a cosmology attempts some 3e4) or the
// step size fell below 1e-12 of z.
template <int N, class F, class Z, class O>
__device__ bool dopri(F&& f, double z0, double* y, int nout, Z&& zout, O&& out, double rtol, double atol) {
#pragma clang fp contract(off)
    const double c2 = 1.0 / 5, c3 = 3.0 / 10, c4 = 4.0 / 5, c5 = 8.0 / 9;
    const double a21 = 1.0 / 5;
    const double a31 = 3.0 / 40, a32 = 9.0 / 40;
    const double a41 = 44.0 / 45, a42 = -56.0 / 15, a43 = 32.0 / 9;
    const double a51 = 19372.0 / 6561, a52 = -25360.0 / 2187, a53 = 64448.0 / 6561, a54 = -212.0 / 729;
    const double a61 = 9017.0 / 3168, a62 = -355.0 / 33, a63 = 46732.0 / 5247, a64 = 49.0 / 176, a65 = -5103.0 / 18656;
    const double b1 = 35.0 / 384, b3 = 500.0 / 1113, b4 = 125.0 / 192, b5 = -2187.0 / 6784, b6 = 11.0 / 84;
    const double e1 = 71.0 / 57600, e3 = -71.0 / 16695, e4 = 71.0 / 1920, e5 = -17253.0 / 339200, e6 = 22.0 / 525,
                 e7 = -1.0 / 40;
    double z = z0;
    double h = (nout == 0 ? 0.0 : (zout(nout - 1) < z0 ? -1e-3 : 1e-3)) * fmax(1.0, fabs(z0));
    double k1[N], k2[N], k3[N], k4[N], k5[N], k6[N], k7[N], yt[N], yn[N];
    f(z, y, k1);
    long long guard = 0;
    for (int io = 0; io < nout; ++io) {
        const double zt = zout(io);
        while (z != zt) {
            if (++guard > 500000 || !(fabs(h) > 1e-12 * fmax(1.0, fabs(z)))) return false;
            const double dir = (zt < z) ? -1.0 : 1.0;
            if (h * dir <= 0) h = -h;
            bool last = false;
            if (fabs(h) >= fabs(zt - z)) { h = zt - z; last = true; }
            for (int i = 0; i < N; ++i) yt[i] = y[i] + h * a21 * k1[i];
            f(z + c2 * h, yt, k2);
            for (int i = 0; i < N; ++i) yt[i] = y[i] + h * (a31 * k1[i] + a32 * k2[i]);
            f(z + c3 * h, yt, k3);
            for (int i = 0; i < N; ++i) yt[i] = y[i] + h * (a41 * k1[i] + a42 * k2[i] + a43 * k3[i]);
            f(z + c4 * h, yt, k4);
            for (int i = 0; i < N; ++i) yt[i] = y[i] + h * (a51 * k1[i] + a52 * k2[i] + a53 * k3[i] + a54 * k4[i]);
            f(z + c5 * h, yt, k5);
            for (int i = 0; i < N; ++i)
                yt[i] = y[i] + h * (a61 * k1[i] + a62 * k2[i] + a63 * k3[i] + a64 * k4[i] + a65 * k5[i]);
            f(z + h, yt, k6);
            for (int i = 0; i < N; ++i) yn[i] = y[i] + h * (b1 * k1[i] + b3 * k3[i] + b4 * k4[i] + b5 * k5[i] + b6 * k6[i]);
            f(z + h, yn, k7);
            double err = 0.0;
            for (int i = 0; i < N; ++i) {
                const double e = h * (e1 * k1[i] + e3 * k3[i] + e4 * k4[i] + e5 * k5[i] + e6 * k6[i] + e7 * k7[i]);
                const double sc = atol + rtol * fmax(fabs(y[i]), fabs(yn[i]));
                err += (e / sc) * (e / sc);
            }
            err = sqrt(err / N);
            if (!(err == err)) err = 1e10;
            if (err <= 1.0) {
                z = last ? zt : z + h;
                for (int i = 0; i < N; ++i) { y[i] = yn[i]; k1[i] = k7[i]; }
                const double fac = (err == 0.0) ? 5.0 : fmin(5.0, fmax(0.2, 0.9 * pow(err, -0.2)));
                if (!last) h *= fac;
            } else {
                h *= fmax(0.1, 0.9 * pow(err, -0.2));
            }
        }
        out(io, y);
    }
    return true;
}

// IonizationHistory(RECFAST) on the grid (recfast.jl:446-536, 674-726): X_e and
// T_mat at every node into xe[], tm[], by one whole wavefront (the rates are
// evaluated across its lanes; every lane carries the same integration)
__device__ bool recfast_grid(const Args& A, const Par& Pc, const double* coef, double* xe, double* tm) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & (WAVE - 1);
    const RfC P = Pc.rc;
    HcTab H;
    H.hc = coef + (size_t)BOLT_T_HC * (A.nx + 2);
    H.hcp = coef + (size_t)BOLT_T_HC_P * (A.nx + 2);
    H.nx = A.nx; H.x0 = A.x0; H.dx = A.dx; H.iH0_conv = 1.0 / A.H0_conv;
    const double fHe = P.fHe, Tnow = P.Tnow;
    const int nx = A.nx;
    const double zinitial = 10000.0;
    const double x_init = log(1.0 / (zinitial + 1.0));
    const double zre_ini = 50.0;
    int j_init = nx;
    for (int j = 0; j < nx; ++j)
        if (!(node(A, j) < x_init)) { j_init = j; break; }
    auto zj = [&](int j) { return 1.0 / exp(node(A, j)) - 1.0; };
    // the stage switches (recfast.jl:373-380, 408, 451-459)
    const double zHeS = rf_bisect([&](double z) { return (he_saha_x0(z, P) - 1.0) / fHe - 0.99; }, 3500.0, 0.0);
    const double zHHS = rf_bisect([&](double z) { return x_H0_saha(z, P) - 0.985; }, zHeS, 0.0);
    // node ranges by stage, in descending z (ascending j)
    int jHe = j_init;  // first node with z <= zHeS
    while (jHe < nx && zj(jHe) > zHeS) ++jHe;
    int jHH = jHe;     // first node with z <= zHHS
    while (jHH < nx && zj(jHH) > zHHS) ++jHH;
    int jre = jHH;     // first node with z <= 50
    while (jre < nx && zj(jre) > zre_ini) ++jre;
    for (int j = lane; j < jHe; j += WAVE) {
        const double Trad = Tnow * (1 + (1.0 / exp(node(A, j)) - 1.0));
        if (j < j_init) { xe[j] = 1.0 + 2 * fHe; tm[j] = Trad; }
        else { const double z = zj(j); xe[j] = xe_saha_early(z, P); tm[j] = Tnow * (1.0 + z); }
    }
    // stage 2: He + Tmat with H in Saha (recfast.jl:461-465, 383-399), outputs
    // at the nodes, then at zHHS
    double y2[2];
    {
        const double x0 = he_saha_x0(zHeS, P);
        y2[0] = (x0 - 1.0) / fHe;
        y2[1] = Tnow * (1.0 + zHeS);
    }
    auto fHe_stage = [&](double z, const double* y, double* dy) {
        const R3 f = rf_rates(x_H0_saha(z, P), y[0], y[1], z, P, H);
        dy[0] = f.f2;
        dy[1] = f.f3;
    };
    const int n2 = jHH - jHe;
    bool ok = dopri<2>(fHe_stage, zHeS, y2, n2 + 1, [&](int i) { return i < n2 ? zj(jHe + i) : zHHS; },
                       [&](int i, const double* y) {
                           if (i < n2 && lane == 0) {
                               const double z = zj(jHe + i);
                               xe[jHe + i] = x_H0_saha(z, P) + fHe * y[0];
                               tm[jHe + i] = y[1];
                           }
                       }, 1e-11, 1e-14);
    // stage 3: H + He + Tmat down to z = 50 (recfast.jl:467-471)
    double y3[3] = {x_H0_saha(zHHS, P), y2[0], y2[1]};
    auto fHH = [&](double z, const double* y, double* dy) {
        const R3 f = rf_rates(y[0], y[1], y[2], z, P, H);
        dy[0] = f.f1; dy[1] = f.f2; dy[2] = f.f3;
    };
    const int n3 = jre - jHH;
    ok = ok && dopri<3>(fHH, zHHS, y3, n3 + 1, [&](int i) { return i < n3 ? zj(jHH + i) : zre_ini; },
                        [&](int i, const double* y) {
                            if (i < n3 && lane == 0) {
                                xe[jHH + i] = y[0] + fHe * y[1];
                                tm[jHH + i] = y[2];
                            }
                        }, 1e-11, 1e-14);
    // stage 4: with the reionized matter temperature from z = 50 (recfast.jl:478-536)
    const double X_fin = 1.0 + P.Yp / (rfc::not4 * (1.0 - P.Yp));
    const double zre = 7.6711, alpha = 1.5, dH = 0.5, zHe = 3.5, dHe = 0.5;
    const double fHe_r = X_fin - 1.0;
    auto reio_xe = [&](double z, double x_orig) {
        const double xH = (X_fin - x_orig) / 2 *
                              (1.0 + tanh((pow(1 + zre, alpha) - pow(1.0 + z, alpha)) / (alpha * pow(1 + zre, alpha - 1)) / dH)) +
                          x_orig;
        const double xHe = fHe_r / 2 * (1.0 + tanh((zHe - z) / dHe));
        return xH + xHe;
    };
    double y4[4] = {y3[0], y3[1], y3[2], y3[2]};
    auto f4 = [&](double z, const double* y, double* dy) {
        const R3 f = rf_rates(y[0], y[1], y[2], z, P, H);
        dy[0] = f.f1; dy[1] = f.f2; dy[2] = f.f3;
        const double xr = reio_xe(z, y[0] + fHe * y[1]);
        const double aa = 1.0 / (1.0 + z);
        const double Hz = spl(H.hc, H.nx, H.x0, H.dx, log(aa), 0) / aa / A.H0_conv;
        const double Trad = Tnow * (1.0 + z);
        dy[3] = c_rfk.CT * pow(Trad, 4) * xr / (1.0 + xr + fHe) * (y[3] - Trad) / (Hz * (1.0 + z)) + 2 * y[3] / (1.0 + z);
    };
    const int n4 = nx - jre;
    ok = ok && dopri<4>(f4, zre_ini, y4, n4, [&](int i) { return zj(jre + i); },
                        [&](int i, const double* y) {
                            if (lane != 0) return;
                            const double z = zj(jre + i);
                            xe[jre + i] = reio_xe(z, y[0] + fHe * y[1]);
                            tm[jre + i] = y[3];
                        }, 1e-11, 1e-14);
    return ok;
}

// one wavefront per cosmology: the RECFAST integration needs exactly one, and
// the node-wise phases are short, so more cosmologies fit on a CU at once
__global__ void __launch_bounds__(WAVE) k_tables(Args A) {
#pragma clang fp contract(off)
    const int c = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
    const Par P = A.par[c];
    const int nx = A.nx;
    double* coef = A.coef + (size_t)c * BOLT_NTAB * (nx + 2);
    double* W = A.work + (size_t)c * WK * nx;
    auto tab = [&](int k) { return coef + (size_t)k * (nx + 2); };
    auto w = [&](int k) { return W + (size_t)k * nx; };
    // ρ₀ℳ, ℋ, η at the nodes (background.jl:106-108)
    for (int j = t; j < nx; j += nt) {
        const double x = node(A, j);
        w(0)[j] = rho0_massive(A, P, exp(x));
        w(1)[j] = Hc_a(A, P, exp(x));
        w(2)[j] = eta(A, P, x);
    }
    __syncthreads();
    if (t == 0) prefilter(w(0), nx, tab(BOLT_T_RHO0M));
    if (t == 1) prefilter(w(1), nx, tab(BOLT_T_HC));
    if (t == 2) prefilter(w(2), nx, tab(BOLT_T_ETA));
    __syncthreads();
    // ℋ′, ℋ″, η′, η″: splines of the node derivatives (util.jl:12-13)
    for (int j = t; j < nx; j += nt) {
        w(3)[j] = node_deriv(tab(BOLT_T_HC), j, A.dx, 1);
        w(4)[j] = node_deriv(tab(BOLT_T_HC), j, A.dx, 2);
        w(5)[j] = node_deriv(tab(BOLT_T_ETA), j, A.dx, 1);
        w(6)[j] = node_deriv(tab(BOLT_T_ETA), j, A.dx, 2);
    }
    __syncthreads();
    if (t == 0) prefilter(w(3), nx, tab(BOLT_T_HC_P));
    if (t == 1) prefilter(w(4), nx, tab(BOLT_T_HC_PP));
    if (t == 2) prefilter(w(5), nx, tab(BOLT_T_ETA_P));
    if (t == 3) prefilter(w(6), nx, tab(BOLT_T_ETA_PP));
    if (t == 4) A.scal[(size_t)c * BOLT_NSCAL + BOLT_S_ETA0] = eta(A, P, 0.0);  // background.jl:112
    __syncthreads();
    // RECFAST on the first wavefront: X_e into w(7), T_mat into w(8)
    if (t < WAVE) {
        const bool ok = recfast_grid(A, P, coef, w(7), w(8));
        if (t == 0) A.status[c] = ok ? 0 : 1;
    }
    __syncthreads();
    // τ′ at the nodes, its reverse cumulative trapezoid, g̃ (ionization.jl:107-129)
    const double rho_crit = P.rho_crit;
    for (int j = t; j < nx; j += nt) {
        const double x = node(A, j), a = exp(x);
        const double nH = P.Omega_b * rho_crit / (A.m_H * a * a * a) * (1.0 - P.Y_p);
        w(9)[j] = -w(7)[j] * nH * a * A.sigma_T / spl(tab(BOLT_T_HC), nx, A.x0, A.dx, x, 0);
    }
    __syncthreads();
    if (t == 0) {
        double* tau = w(10);
        const double* tp = w(9);
        tau[nx - 1] = 0.0;
        for (int j = nx - 2; j >= 0; --j) tau[j] = tau[j + 1] + (node(A, j) - node(A, j + 1)) * (tp[j] + tp[j + 1]) * 0.5;
        A.scal[(size_t)c * BOLT_NSCAL + BOLT_S_TAU0] = tau[nx - 1];
    }
    __syncthreads();
    for (int j = t; j < nx; j += nt) w(11)[j] = -w(9)[j] * exp(-w(10)[j]);  // g̃_function
    __syncthreads();
    if (t == 0) prefilter(w(7), nx, tab(BOLT_T_XE));
    if (t == 1) prefilter(w(10), nx, tab(BOLT_T_TAU));
    if (t == 2) prefilter(w(11), nx, tab(BOLT_T_G));
    if (t == 3) prefilter(w(8), nx, tab(BOLT_T_TMAT));
    __syncthreads();
    for (int j = t; j < nx; j += nt) {
        w(0)[j] = node_deriv(tab(BOLT_T_TAU), j, A.dx, 1);
        w(1)[j] = node_deriv(tab(BOLT_T_TAU), j, A.dx, 2);
        w(2)[j] = node_deriv(tab(BOLT_T_G), j, A.dx, 1);
        w(3)[j] = node_deriv(tab(BOLT_T_G), j, A.dx, 2);
        w(4)[j] = node_deriv(tab(BOLT_T_TMAT), j, A.dx, 1);
    }
    __syncthreads();
    if (t == 0) prefilter(w(0), nx, tab(BOLT_T_TAU_P));
    if (t == 1) prefilter(w(1), nx, tab(BOLT_T_TAU_PP));
    if (t == 2) prefilter(w(2), nx, tab(BOLT_T_G_P));
    if (t == 3) prefilter(w(3), nx, tab(BOLT_T_G_PP));
    // sound speed (recfast.jl:710-712), with RECFAST's SI constants
    {
        const double C = 2.99792458e8, k_B = 1.380658e-23, m_H = 1.673575e-27, not4 = 3.9715e0;
        const double Yp = P.Y_p, mu_T = not4 / (not4 - (not4 - 1) * Yp);
        for (int j = t; j < nx; j += nt) {
            const double x = node(A, j);
            const double pre = pow(C, -2) * k_B / m_H * (1.0 / mu_T + (1.0 - Yp) * spl(tab(BOLT_T_XE), nx, A.x0, A.dx, x, 0));
            w(5)[j] = pre * (spl(tab(BOLT_T_TMAT), nx, A.x0, A.dx, x, 0) - 1.0 / 3.0 * w(4)[j]);
        }
    }
    __syncthreads();
    if (t == 0) prefilter(w(5), nx, tab(BOLT_T_CSB2));
    if (t == 1) {
        double* s = A.scal + (size_t)c * BOLT_NSCAL;
        s[BOLT_S_H0] = P.H0;
        s[BOLT_S_RHO_CRIT] = P.rho_crit;
        s[BOLT_S_OMEGA_L] = P.Omega_L;
    }
}

}  // namespace gbg

namespace gbg {
// RECFAST's derived constants and one cosmology's, as the host RECFAST's
// constructor computes them (host_tables.cpp, RecfastT; recfast.jl:22-121)
static RfK rf_constants() {
#pragma clang fp contract(off)
    using namespace rfc;
    RfK k;
    k.a_VF = std::pow(10.0, -16.744);
    k.T_0 = std::pow(10.0, 0.477121);
    k.T_1 = std::pow(10.0, 5.114);
    k.a_trip = std::pow(10.0, -16.306);
    k.Lalpha = 1 / L_H_alpha;
    k.Lalpha_He = 1 / L_He_2p;
    const double DeltaB = h_P * C * (L_H_ion - L_H_alpha);
    k.CDB = DeltaB / k_B;
    const double DeltaB_He = h_P * C * (L_He1_ion - L_He_2s);
    k.CDB_He = DeltaB_He / k_B;
    k.CB1 = h_P * C * L_H_ion / k_B;
    k.CB1_He1 = h_P * C * L_He1_ion / k_B;
    k.CB1_He2 = h_P * C * L_He2_ion / k_B;
    k.CR = 2 * M_PI * (m_e / h_P) * (k_B / h_P);
    k.CK = std::pow(k.Lalpha, 3) / (8 * M_PI);
    k.CK_He = std::pow(k.Lalpha_He, 3) / (8 * M_PI);
    k.CL = C * h_P / (k_B * k.Lalpha);
    k.CL_He = C * h_P / (k_B / L_He_2s);
    k.CT = (8.0 / 3.0) * (sigma / (m_e * C)) * a;
    k.Bfact = h_P * C * (L_He_2p - L_He_2s) / k_B;
    k.iT_0 = 1.0 / k.T_0;
    k.iT_1 = 1.0 / k.T_1;
    k.dop = 2 * k_B / (m_H * not4 * C * C);
    k.itau_t = 1.0 / (8 * M_PI * std::pow(L_He_2Pt, 3));
    k.g2Ps = 3 * A2P_s * C * C / (std::sqrt(M_PI) * sigma_He_2Ps * 8 * M_PI * C * L_He_2p) / std::pow(C * L_He_2p, 2);
    k.g2Pt = 3 * A2P_t * C * C / (std::sqrt(M_PI) * sigma_He_2Pt * 8 * M_PI * C * L_He_2Pt) / std::pow(C * L_He_2Pt, 2);
    return k;
}
static RfC rf_cosmology(const bolt_cosmo_params& p, double H0, double rho_crit) {
#pragma clang fp contract(off)
    using namespace rfc;
    const bolt::NaturalUnits& u = bolt::natural_units();
    RfC r;
    r.Yp = p.Y_p;
    r.OmegaB = p.Omega_b;
    r.HO = H0 / u.H0_conv;
    const double OmegaG = p.Omega_r;
    r.Tnow = std::pow(15.0 / (M_PI * M_PI) * rho_crit * OmegaG, 0.25) * u.K_conv;
    r.mu_H = 1.0 / (1.0 - r.Yp);
    r.mu_T = not4 / (not4 - (not4 - 1) * r.Yp);
    r.fHe = r.Yp / (not4 * (1.0 - r.Yp));
    r.Nnow = 3.0 * r.HO * r.HO * r.OmegaB / (8 * M_PI * G * r.mu_H * m_H);
    return r;
}
}  // namespace gbg

extern "C" {

int bolt_device_tables_batch(bolt_ctx* ctx, const bolt_cosmo_params* pars, int ncosmo, double x0, double x1, int nx,
                             int nq, double* coef_out, double* scal_out, double* xq_out, double* wq_out, int* status) {
    if (!ctx || !pars || ncosmo < 0 || !coef_out || !scal_out || !xq_out || !wq_out || !status)
        return set_error(BOLT_E_ARG, "bolt_device_tables_batch: NULL argument or negative count");
    if (nx < 4 || nx > (1 << 20) || nq < 1 || nq > SV_MAX_NQ || !(x1 > x0))
        return set_error(BOLT_E_ARG, "bolt_device_tables_batch: bad grid");
    for (int c = 0; c < ncosmo; ++c)
        if (!(pars[c].Omega_r > 0) || !(pars[c].N_nu > 0) || !(pars[c].h > 0))
            return set_error(BOLT_E_ARG, "bolt_device_tables_batch: Omega_r, N_nu and h must be positive");
    if (ncosmo == 0) return BOLT_OK;
    // Background's constants per cosmology, from the host's own CosmoT
    std::vector<gbg::Par> hp(ncosmo);
    std::vector<double> xq, wq;
    for (int c = 0; c < ncosmo; ++c) {
        const bolt::CosmoT<double> cm(bolt::ParamsT<double>(pars[c]), nq);
        gbg::Par& P = hp[c];
        P.h = pars[c].h; P.Omega_r = pars[c].Omega_r; P.Omega_b = pars[c].Omega_b; P.Omega_c = pars[c].Omega_c;
        P.N_nu = pars[c].N_nu; P.Sum_m_nu = pars[c].Sum_m_nu; P.Y_p = pars[c].Y_p;
        P.H0 = cm.H0; P.rho_crit = cm.rho_crit; P.Omega_L = cm.Omega_L; P.rad_fac = cm.rad_fac; P.Tnu = cm.Tnu;
        P.logqmin = cm.logqmin; P.logqmax = cm.logqmax;
        P.rc = gbg::rf_cosmology(pars[c], cm.H0, cm.rho_crit);
        if (c == 0) { xq = cm.xq; wq = cm.wq; }
    }
    HIPCHK(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    // RECFAST's constants do not depend on the cosmology: calls from several
    // contexts at once write the same bytes into the device's constant block
    const gbg::RfK rk = gbg::rf_constants();
    HIPCHK(hipMemcpyToSymbolAsync(HIP_SYMBOL(gbg::c_rfk), &rk, sizeof(rk), 0, hipMemcpyHostToDevice, st));
    const size_t ntab = (size_t)BOLT_NTAB * (nx + 2);
    Scratch<gbg::Par> dpar;
    Scratch<double> dxq, dwq, dcoef, dscal, dwork;
    Scratch<int> dst;
    HIPCHK(dpar.up(hp.data(), ncosmo, st));
    HIPCHK(dxq.up(xq.data(), nq, st));
    HIPCHK(dwq.up(wq.data(), nq, st));
    if (dcoef.alloc(ntab * ncosmo) != hipSuccess || dscal.alloc((size_t)BOLT_NSCAL * ncosmo) != hipSuccess ||
        dwork.alloc((size_t)gbg::WK * nx * ncosmo) != hipSuccess || dst.alloc(ncosmo) != hipSuccess)
        return set_error(BOLT_E_NOMEM, "bolt_device_tables_batch: device memory");
    const bolt::NaturalUnits& u = bolt::natural_units();
    gbg::Args A;
    A.par = dpar.p; A.nx = nx; A.nq = nq; A.x0 = x0; A.x1 = x1; A.dx = (x1 - x0) / (nx - 1);
    A.xq = dxq.p; A.wq = dwq.p;
    A.H0_conv = u.H0_conv; A.K_conv = u.K_conv; A.m_H = u.m_H; A.sigma_T = u.sigma_T;
    A.coef = dcoef.p; A.scal = dscal.p; A.work = dwork.p; A.status = dst.p;
    hipLaunchKernelGGL(gbg::k_tables, dim3(ncosmo), dim3(WAVE), 0, st, A);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(coef_out, dcoef.p, sizeof(double) * ntab * ncosmo, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(scal_out, dscal.p, sizeof(double) * BOLT_NSCAL * ncosmo, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(status, dst.p, sizeof(int) * ncosmo, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    for (int i = 0; i < nq; ++i) { xq_out[i] = xq[i]; wq_out[i] = wq[i]; }
    int bad = 0;
    for (int c = 0; c < ncosmo; ++c) {
        if (!status[c]) {
            const double* cf = coef_out + ntab * c;
            for (size_t i = 0; i < ntab; ++i)
                if (!std::isfinite(cf[i])) { status[c] = BOLT_E_NUMERIC; break; }
        } else {
            status[c] = BOLT_E_NUMERIC;
        }
        bad += status[c] != 0;
    }
    if (bad) return set_error(BOLT_E_NUMERIC, "bolt_device_tables_batch: a cosmology's tables failed (status)");
    return BOLT_OK;
}

}  // extern "C"
